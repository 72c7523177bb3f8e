"""Waits of hand-pipelined kernels, read from the assembly that the extension's flags give."""
import os
import re
import subprocess

import pytest

from rag_tl_domainllm_optimizer_amd import _build

HIPCC = os.path.join(_build.ROCM, "bin", "hipcc")


def _assembly(kernel, tmp_path):
    out = tmp_path / "k.s"
    subprocess.run([HIPCC, *_build.kernel_flags(), "-S", "--offload-device-only", os.path.join(_build.CSRC, "kernels", kernel), "-o", str(out)],
                   check=True, capture_output=True)
    return out.read_text()


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_product_and_norm_fills_no_place_that_is_being_read(tmp_path):
    """Behind each barrier of the product's loop the places of the granule of w that was read before it are filled again: none of its reads may be
    under way there, in whatever order the compiler asked for them. LDS reads of a wave come back in their order; those of w lie behind the
    places of x, which is how the two are told apart."""
    text = _assembly("gemm_norm.hip", tmp_path)
    kernels = re.findall(r"^(_ZN2rt2gn16gemm_norm_kernelILi(\d+)ELi(\d+)ELi(\d+)E\S*):(.*?)^\.Lfunc_end", text, re.M | re.S)
    assert len(kernels) == 4
    for _, wc, fm, np_, body in kernels:
        wc, fm, np_ = int(wc), int(fm), int(np_)
        first_w = 3 * (8 // wc * 16 * fm) * 128
        under_way, reads, counted = [], 0, 0
        for line in body.split("\n"):
            op = line.split(";")[0].split()
            if not op:
                continue
            if op[0] == "ds_write_b64":  # the epilogue: the loop is over
                break
            if op[0].startswith("ds_read"):
                at = re.search(r"offset:(\d+)", line)
                under_way.append("w" if at and int(at.group(1)) >= first_w else "x")
                reads += under_way[-1] == "w"
            elif op[0] == "s_waitcnt":
                left = re.search(r"lgkmcnt\((\d+)\)", line)
                if left:
                    n = int(left.group(1))
                    under_way = under_way[len(under_way) - n:] if n else []
            elif op[0] == "s_barrier":
                assert "w" not in under_way, (wc, fm, np_, under_way)
                counted += bool(under_way)
        # two steps and the last one, each of np_ phases that read a granule but the very last; x under way at the first phases' barriers
        assert reads == 2 * (8 // wc) * 3 * np_ and counted >= 2, (reads, counted)
