"""Batched sentence encoder (mean pooling + L2 normalisation), one forward for many strings.

Replaces the reference's per-string ``SentenceTransformer.encode`` calls (1 + k + 2 (+2) separate
forwards per reward, reinforcement_learning_optimization_after_rag.py:66-67,75-76,102-103): texts
are tokenised natively in parallel and sorted by length into batches without padding, which go up in one copy and
are encoded on the GPU.
"""
from __future__ import annotations

from typing import List, Optional, Sequence

import torch

from ..models import build_model
from ..models.encoder import SentenceEncoder
from ..tokenizer import Tokenizer, load_tokenizer


BATCH_SIZE = 256        # the default
MERGED_BYTES = 1 << 30  # of activations of default batches that are encoded in one forward: what one of 256 long texts takes alone


class Encoder:
    """``batch_size``: the most texts of a forward, where it is not the default. ``max_rows``: on a GPU batches go together up to so
    many tokens (0: none do); None: those of the default size do, up to ``MERGED_BYTES`` of activations, others don't. A text's
    last bits depend on the rows beside it in its forward, whose number chooses the order in which products are summed."""

    def __init__(self, model: SentenceEncoder, tokenizer: Tokenizer, max_length: int = 256, batch_size: int = BATCH_SIZE,
                 max_rows: Optional[int] = None):
        self.model = model
        self.tokenizer = tokenizer
        self.max_length = min(max_length, model.cfg.max_position - model.cfg.position_offset)
        self.batch_size = batch_size
        self.max_rows = max_rows

    @classmethod
    def from_name(cls, name_or_path: str = "all-MiniLM-L6-v2:random", device="cpu", max_length: int = 256,
                  batch_size: int = BATCH_SIZE, seed: int = 0, max_rows: Optional[int] = None) -> "Encoder":
        model = build_model(name_or_path, device=device, seed=seed)
        tok = load_tokenizer(name_or_path, model.cfg.vocab_size, model.cfg.arch)
        return cls(model.eval(), tok, max_length, batch_size, max_rows)

    @property
    def device(self):
        return self.model.word_embed.device

    @property
    def dim(self) -> int:
        return self.model.cfg.hidden_size

    def _as_made(self) -> bool:
        """Whether model and tokenizer do their parts of a padded batch as this package has them do: others (a pooling of
        one's own, another tokenizer) are called for each."""
        return all(getattr(type(o), n, None) is getattr(c, n) and n not in vars(o) for o, c, names in (
            (self.model, SentenceEncoder, ("forward", "encode_ids")), (self.tokenizer, Tokenizer, ("encode_batch", "pad", "_wrap")))
            for n in names)

    def _rows_together(self) -> int:
        """Tokens up to which further batches go into a forward on a GPU."""
        if self.max_rows is not None:
            return self.max_rows
        c = self.model.cfg
        return MERGED_BYTES // (2 * (7 * c.hidden_size + c.intermediate_size)) if self.batch_size == BATCH_SIZE else 0

    @torch.no_grad()
    def encode(self, texts: Sequence[str], normalize: bool = True) -> torch.Tensor:
        """-> fp32 [N, dim] on the model's device (unit vectors when normalize)."""
        texts = list(texts)
        N = len(texts)
        out = torch.empty(N, self.dim, dtype=torch.float32, device=self.device)
        if N == 0:
            return out
        if not self._as_made():
            enc = self.tokenizer.encode_batch(texts, True, self.max_length)
            order = sorted(range(N), key=lambda i: len(enc[i]))
            for s in range(0, N, self.batch_size):
                idx = order[s:s + self.batch_size]
                batch = self.tokenizer.pad([enc[i] for i in idx], side="right", device=self.device)
                emb = self.model.encode_ids(batch["input_ids"], batch["lengths"], normalize)
                out[torch.tensor(idx, device=self.device)] = emb.float()
            return out
        # every batch is tokenised and uploaded ahead of the first forward: between them the host only launches
        r, m, tok = 0, self.model, self.tokenizer
        placed = type(m).encode_packed is SentenceEncoder.encode_packed and "encode_packed" not in vars(m)
        # On a GPU batches go together: each product's last round of tiles leaves CUs idle once, not once a batch (1024 texts of
        # 20 to 120 words, MiniLM, four batches 3231 -> 2869 us)
        most = {}
        if placed and self.device.type == "cuda" and type(tok).encode_sorted is Tokenizer.encode_sorted and "encode_sorted" not in vars(tok):
            most = dict(most_rows=self._rows_together())
        order, batches = tok.encode_sorted(texts, self.max_length, self.batch_size, self.device, m.first_position, **most)
        for ids, pos, off, longest in batches:
            n = len(off) - 1
            if placed:
                m.encode_packed(ids, pos, off, longest, normalize, out, order[r:r + n])
            else:
                out[order[r:r + n]] = m.encode_packed(ids, pos, off, longest, normalize).float()
            r += n
        return out

    def encode_unique(self, texts: Sequence[str], normalize: bool = True):
        """Encode each distinct string once; returns (embeddings [U, d], index map list -> row)."""
        uniq, where = {}, []
        for t in texts:
            if t not in uniq:
                uniq[t] = len(uniq)
            where.append(uniq[t])
        emb = self.encode(list(uniq.keys()), normalize)
        return emb, torch.tensor(where, dtype=torch.long, device=emb.device)
