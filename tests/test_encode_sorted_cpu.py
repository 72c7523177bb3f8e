"""The encoders' native batch preparation against encode_batch, and encoding without padding."""
import random

import pytest
import torch

from rag_tl_domainllm_optimizer_amd import models
from rag_tl_domainllm_optimizer_amd.models import PRESETS
from rag_tl_domainllm_optimizer_amd.tokenizer import Tokenizer


@pytest.mark.parametrize("arch", ["bert", "mpnet", "llama"])
@pytest.mark.parametrize("n,batch,max_length", [(1, 8, 16), (7, 3, 4), (130, 64, 9), (64, 64, 1), (5, 2, 2)])
def test_encode_sorted(arch, n, batch, max_length):
    tok = Tokenizer.synthetic(400, arch)
    words, r = tok.words(), random.Random(n)
    texts = ["", *(" ".join(r.choices(words, k=r.randint(0, 12))) for _ in range(n - 1))]
    enc = tok.encode_batch(texts, True, max_length)
    order = sorted(range(n), key=lambda i: len(enc[i]))
    got, groups = tok.encode_sorted(texts, max_length, batch, "cpu", 2)
    assert got.tolist() == order and len(groups) == (n + batch - 1) // batch
    for g, (ids, pos, off, longest) in enumerate(groups):
        want = [enc[i] for i in order[g * batch:(g + 1) * batch]]
        assert ids.tolist() == sum(want, []) and pos.tolist() == [2 + k for w in want for k in range(len(w))]
        assert off.tolist() == [sum(map(len, want[:k])) for k in range(len(want) + 1)]
        assert longest == len(want[-1])


@pytest.mark.parametrize("preset", ["tiny-bert", "tiny-mpnet"])
def test_encode_packed_equals_padded(preset):
    """Texts without padding give what the padded batch gives, a text of no tokens among them."""
    cfg = PRESETS[preset]
    m = models.SentenceEncoder(cfg, dtype=torch.float32, seed=1)
    lens = torch.tensor([0, 1, 3, 9, 17])
    g = torch.Generator().manual_seed(0)
    ids = torch.randint(5, cfg.vocab_size, (5, 17), generator=g)
    off = torch.nn.functional.pad(lens.cumsum(0), (1, 0))
    flat = torch.cat([ids[b, :n] for b, n in enumerate(lens)])
    pos = torch.cat([torch.arange(n) for n in lens]) + m.first_position
    torch.testing.assert_close(m.encode_packed(flat, pos, off, 17), m.encode_ids(ids, lens), rtol=1e-5, atol=1e-6)
    none = torch.zeros(0, dtype=torch.long)
    assert torch.equal(m.encode_packed(none, none, torch.zeros(3, dtype=torch.long), 0), torch.zeros(2, cfg.hidden_size))


def test_encode_sorted_refuses():
    tok = Tokenizer.synthetic(400, "bert")
    for batch, max_length in ((0, 4), (4, 0)):
        with pytest.raises(RuntimeError):
            tok.encode_sorted(["a"], max_length, batch, "cpu")


def test_encoder_calls_parts_of_ones_own():
    """A model that pools in its own way, another tokenizer and patched objects are called as for padded batches."""
    from rag_tl_domainllm_optimizer_amd.retrieval import Encoder

    class FirstToken(models.SentenceEncoder):
        def encode_ids(self, input_ids, lengths, normalize=True):
            B, S = input_ids.shape
            return self.forward(input_ids, lengths).view(B, S, -1)[:, 0]

    class Letters:
        def encode_batch(self, texts, special=True, max_length=None):
            return [[5 + ord(c) % 300 for c in t][:max_length] for t in texts]

        def pad(self, seqs, side=None, max_length=None, device=None):
            return tok.pad(seqs, side, max_length, device)

    cfg = PRESETS["tiny-bert"]
    tok = Tokenizer.synthetic(cfg.vocab_size, "bert")
    words = tok.words()
    texts = [" ".join(words[i:i + 1 + i % 5]) for i in range(9)]
    plain, first = (c(cfg, dtype=torch.float32, seed=1) for c in (models.SentenceEncoder, FirstToken))

    def padded(model, t):
        batch = t.pad(t.encode_batch(texts, True, 16), side="right")
        return model.encode_ids(batch["input_ids"], batch["lengths"])

    for model, t in ((first, tok), (plain, Letters()), (plain, tok)):
        torch.testing.assert_close(Encoder(model, t, 16, batch_size=4).encode(texts), padded(model, t), rtol=1e-5, atol=1e-6)
    plain.encode_ids = lambda ids, lengths, normalize=True: torch.full((len(ids), cfg.hidden_size), 0.5)
    assert bool((Encoder(plain, tok, 16).encode(texts) == 0.5).all())


@pytest.mark.parametrize("most", [1, 40, 100, 10 ** 6])
def test_encode_sorted_merges_batches(most):
    """Batches go together while their rows fit, a single one whatever it has; the texts and their order are the same."""
    tok = Tokenizer.synthetic(400, "bert")
    words, r = tok.words(), random.Random(3)
    texts = [" ".join(r.choices(words, k=r.randint(0, 12))) for _ in range(50)]
    order, single = tok.encode_sorted(texts, 16, 8, "cpu", 2)
    got, groups = tok.encode_sorted(texts, 16, 8, "cpu", 2, most)
    assert torch.equal(got, order)
    at = 0
    for ids, pos, off, longest in groups:
        parts = []
        while sum(len(p[2]) - 1 for p in parts) < len(off) - 1:
            parts.append(single[at + len(parts)])
        at += len(parts)
        assert torch.equal(ids, torch.cat([p[0] for p in parts])) and torch.equal(pos, torch.cat([p[1] for p in parts]))
        assert longest == parts[-1][3] and off.diff().tolist() == sum((p[2].diff().tolist() for p in parts), [])
        rows = len(ids)
        assert len(parts) == 1 or rows <= most
        assert at == len(single) or rows + len(single[at][0]) > most
    assert at == len(single)
