"""The encoders' native batch preparation against encode_batch and pad."""
import random

import pytest
import torch

from rag_tl_domainllm_optimizer_amd.tokenizer import Tokenizer


@pytest.mark.parametrize("arch", ["bert", "mpnet", "llama"])
@pytest.mark.parametrize("n,batch,max_length", [(1, 8, 16), (7, 3, 4), (130, 64, 9), (64, 64, 1), (5, 2, 2)])
def test_encode_sorted(arch, n, batch, max_length):
    tok = Tokenizer.synthetic(400, arch)
    words, r = tok.words(), random.Random(n)
    texts = ["", *(" ".join(r.choices(words, k=r.randint(0, 12))) for _ in range(n - 1))]
    enc = tok.encode_batch(texts, True, max_length)
    order = sorted(range(n), key=lambda i: len(enc[i]))
    got, groups = tok.encode_sorted(texts, max_length, batch, "cpu")
    assert got.tolist() == order and len(groups) == (n + batch - 1) // batch
    for g, (ids, lengths) in enumerate(groups):
        want = tok.pad([enc[i] for i in order[g * batch:(g + 1) * batch]], side="right")
        assert torch.equal(ids, want["input_ids"]) and torch.equal(lengths, want["lengths"])


def test_encode_sorted_refuses():
    tok = Tokenizer.synthetic(400, "bert")
    for batch, max_length in ((0, 4), (4, 0)):
        with pytest.raises(RuntimeError):
            tok.encode_sorted(["a"], max_length, batch, "cpu")
