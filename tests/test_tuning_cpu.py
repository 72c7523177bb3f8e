"""Launch paths carry no hidden state: no environment lookups and no mutable process globals in the
native launchers (per-call operands are arguments; kernel-selection knobs live in ONE struct,
rt::Tuning, set from Python). Static source checks plus the set/get round trip of the binding."""
import glob
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NATIVE = sorted(glob.glob(os.path.join(ROOT, "csrc", "kernels", "*.hip"))) + [os.path.join(ROOT, "csrc", "bindings.cpp")]


def _code(path):
    """Source without // and /* */ comments."""
    s = open(path).read()
    s = re.sub(r"/\*.*?\*/", "", s, flags=re.S)
    return re.sub(r"//[^\n]*", "", s)


def test_no_getenv_in_launchers():
    hits = [(os.path.basename(p), m.group(0)) for p in NATIVE for m in re.finditer(r"\bgetenv\s*\(", _code(p))]
    assert not hits, hits


def test_no_mutable_globals_in_launchers():
    """File-scope (or function-scope static) non-const variables would be state shared by every
    launching thread. Allowed: constexpr / const tables, and the decode-workspace registry of the
    bindings (a mutex-guarded per-stream cache, not a launch parameter)."""
    decl = re.compile(r"^\s*static\s+(?!const\b|constexpr\b|inline\b|__device__|__global__|__forceinline__)"
                      r"([\w:<>,\s\*]+?)\s+\**(\w+)\s*(=|;|\[)", re.M)
    # mutex-guarded caches of the bindings: the decode / stream-K workspace registries and the zero page
    allowed = {"g_ws_map", "g_ws_mu", "g_skws_map", "g_skws_mu", "mu", "map"}
    bad = []
    for p in NATIVE:
        for m in decl.finditer(_code(p)):
            name = m.group(2)
            if "(" in m.group(0) or name in allowed:
                continue
            bad.append((os.path.basename(p), name))
    assert not bad, bad


def test_no_side_channel_setters():
    for p in NATIVE:
        code = _code(p)
        for sym in ("rt_attn_decode_set_qkv_slabs", "rt_attn_decode_set_fp8kv", "rt_attn_o_set_stamps",
                    "rt_attn_decode_set_nk", "rt_gemm_set_"):
            assert sym not in code, (os.path.basename(p), sym)


def test_tuning_roundtrip():
    from rag_tl_domainllm_optimizer_amd import ops

    if not ops.native_available():
        pytest.skip("native extension not built")
    t0 = ops.get_tuning()
    assert t0["decode_mw_kpp"] == 512 and t0["gemm_variant"] == 0 and abs(t0["gemm_bn128_cost"] - 0.55) < 1e-6
    # round-5 defaults: short-sequence attention tiles on up to 1024 positions, the small-batch
    # decode attention unpartitioned up to 1024 cache slots
    assert t0["attn_fwd_hp_maxs"] == 1024 and t0["attn_dq_hp_maxs"] == 1024 and t0["decode_mw_smax"] == 1024
    # only knobs with a live alternative remain (measured-slower paths left the product kernels)
    for gone in ("gemm_streamk", "gemm_ring", "attn_fwd_w8", "attn_bwd_atomic_dq", "gemm_fp8_256", "gemm_tr_builtin",
                 "decode_mw", "decode_mfma"):
        assert gone not in t0, gone
    with ops.tuning(decode_split=2, gemm_bn128_cost=0.7):
        t = ops.get_tuning()
        assert t["decode_split"] == 2 and abs(t["gemm_bn128_cost"] - 0.7) < 1e-6
        assert {k: v for k, v in t.items() if k not in ("decode_split", "gemm_bn128_cost")} == \
            {k: v for k, v in t0.items() if k not in ("decode_split", "gemm_bn128_cost")}
    assert ops.get_tuning() == t0
    with pytest.raises(KeyError):
        ops.set_tuning(no_such_knob=1)


def test_gemm_plan_saves_a_round():
    """GELU products beyond the two-workgroup form's K: rows leave the 256 x 256 tiles only where those then take a round of
    workgroups fewer; a product that fills whole rounds stays one launch."""
    from rag_tl_domainllm_optimizer_amd import ops

    def rounds(rows, N):
        return ((rows + 255) // 256 * ((N + 255) // 256) + 255) // 256

    for K in (2112, 2560, 3072, 4096, 10240):
        for N in (768, 1024, 2560, 4096, 6144, 10240, 16384):
            for M in (513, 700, 1000, 1500, 2100, 3000, 4096, 8192, 10000, 16384, 23500):
                rows, form = ops.native().gemm_plan(M, N, K, ops.ACT_IDS["gelu"])
                assert 0 <= rows <= M and (rows == M or (form in (1, 2, 3) and rounds(rows, N) < rounds(M, N))), (M, N, K, rows, form)
    assert ops.native().gemm_plan(4096, 4096, 4096, ops.ACT_IDS["gelu"])[0] == 4096


@pytest.mark.parametrize("K", [384, 768, 1024])
def test_gemm_plan_of_one_round(K):
    """Without an activation a product that 256 x 256 tiles take in one round of workgroups is not cut to the two-workgroup form,
    which is behind there; beyond a round it is."""
    from rag_tl_domainllm_optimizer_amd import ops

    for M, N in ((10000, 1024), (16384, 1024), (16384, 768), (4096, 4096), (3000, 4096), (4500, 3072), (10000, 1152)):
        rows, form = ops.native().gemm_plan(M, N, K, 0)
        assert rows == M or (rows == 0 and form), (M, N, rows, form)
    for M, N in ((23500, 1152), (8192, 3072), (8192, 4096), (23500, 1024)):
        assert ops.native().gemm_plan(M, N, K, 0)[0] == -1, (M, N)


@pytest.mark.parametrize("nq,nprobe,nlist,d,maxlen,total,probe,by_list", [
    (1, 1, 1, 384, 400000, 400000, 63, 105), (1, 3, 3, 384, 133333, 400000, 62, 76), (2, 8, 64, 384, 8735, 400000, 20, 27),
    (8, 16, 256, 384, 1091, 200000, 20, 29), (256, 16, 4096, 384, 136, 400000, 53, 57), (4, 16, 512, 384, 3539, 200000, 25, 28),
    (4, 1, 1, 128, 400000, 400000, 61, 69), (512, 16, 4096, 128, 136, 400000, 36, 65), (4096, 32, 4096, 72, 136, 400000, 319, 506),
    (8, 1, 1, 384, 400000, 400000, 300, 130), (256, 16, 512, 384, 273, 100000, 84, 27), (12, 16, 256, 384, 7909, 200000, 101, 36),
    (4096, 32, 4096, 384, 136, 400000, 1335, 555), (10000, 8, 1024, 384, 136, 100000, 787, 152), (16, 1, 1, 128, 400000, 400000, 243, 85)])
def test_ivf_scan_form(nq, nprobe, nlist, d, maxlen, total, probe, by_list):
    """Scans take the form that was the faster one when both were timed (us)."""
    from rag_tl_domainllm_optimizer_amd import ops

    assert ops.native().ivf_by_list(nq, nprobe, nlist, d, maxlen, total) == (by_list < probe)


def test_token_plans():
    """The plans that ops.gemm and the encoder's native forward share: whole products beyond 512 rows, parts that fill the chip up to
    there, and the 64 x 64 tiles where their time by the planner's model is below a split product's and its reduction's."""
    from rag_tl_domainllm_optimizer_amd.ops.linear import small_tiles, splitk_plan

    assert splitk_plan(513, 4096, 4096) == (1, 0) and splitk_plan(256, 6144, 4096) == (5, 128) and splitk_plan(256, 4096, 14336) == (8, 128)
    assert splitk_plan(256, 28672, 4096, 5) == (1, 128) and splitk_plan(256, 32000, 4096) == (1, 128)
    assert splitk_plan(300, 1536, 384, 2) == (1, 0) and splitk_plan(400, 16384, 2048, 2) == (1, 0) and splitk_plan(300, 768, 3072, 3) == (6, 256)
    for act in (0, 2):
        assert small_tiles(65, 768, 768, act) and small_tiles(512, 768, 3072, act) and small_tiles(512, 2304, 1408, act)
        assert not small_tiles(64, 768, 768, act) and not small_tiles(513, 768, 768, act) and not small_tiles(300, 768, 776, act)
        assert not small_tiles(512, 10240, 2560, act) and not small_tiles(300, 768, 3136, act)
    assert not small_tiles(300, 768, 768, 1)


def test_nn_split():
    """Products of a gradient with few tiles: K in parts that do not take more than a round, the ones that were the fastest when timed;
    whole where the tiles fill half the chip, where K is short and where the sums of the parts cost more than they save."""
    from rag_tl_domainllm_optimizer_amd import ops

    split = ops.native().nn_split
    for M, N, K, want in ((115, 4096, 28672, (8, 128)), (500, 4096, 28672, (8, 256)), (1000, 4096, 28672, (4, 256)),
                          (1656, 4096, 28672, (2, 256)), (2048, 4096, 28672, (2, 256)), (1000, 4096, 4096, (2, 128))):
        assert split(M, N, K // 64) == want, (M, N, K)
    for M, N, K in ((2049, 4096, 28672), (4016, 4096, 28672), (1656, 4096, 4096), (1656, 4096, 6144), (256, 256, 960), (115, 4092, 28672)):
        assert split(M, N, K // 64)[0] == 1, (M, N, K)


def test_nn_plan_follows_its_knob():
    """The planner's ratio of half tiles reaches the products of a gradient too, whose half tiles cost more (0.62 where the others' cost
    0.55): rows on 256 x 256 tiles at the default and under overrides, with the SwiGLU backward in the epilogue or not."""
    from rag_tl_domainllm_optimizer_amd import ops

    plan = ops.native().gemm_plan
    for act in (0, ops.ACT_DSWIGLU):
        nn = lambda M, N: plan(M, N, 4096, act, ops.KMAJ)[0]  # noqa: E731
        assert nn(4016, 14336) == 4016 and nn(8000, 7168) == 8000
        with ops.tuning(gemm_bn128_cost=0.48):
            assert nn(4016, 14336) == 0 and nn(8000, 7168) == 0
        with ops.tuning(gemm_bn128_cost=1.0):
            assert nn(2048, 4096) == 2048
        assert nn(2048, 4096) == 0
