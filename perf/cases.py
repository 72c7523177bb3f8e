"""What a user of this framework has it do, as cases that can be timed and checked.

Each case is one pass through the public entry points of a part of the pipeline: retrieval, sentence embedding,
prompt processing, one decoded token per row, and a PPO update, over the models, batch sizes and lengths of this
repository's benchmark, presets and tests. Decoders run with a few of their layers (like ``bench.py --mode
layered``): every layer does the same work, and weights are drawn anew for each state.

``listed()`` names cases, ``draw(rng)`` gives more of the same ranges, ``prepare`` makes what a program holds before
the call, ``run`` is the pass, ``work`` the bytes and operations it cannot do without, ``tolerance`` what another
correct implementation at the same precision may differ by, ``exact`` the same result in plain torch at 64 bits."""
from __future__ import annotations

import dataclasses
import math
import random

import torch
import torch.nn.functional as F

from rag_tl_domainllm_optimizer_amd import models, ops
from rag_tl_domainllm_optimizer_amd.generation import PAGE, KVCache, StepEngine
from rag_tl_domainllm_optimizer_amd.retrieval import Encoder, IVFIndex
from rag_tl_domainllm_optimizer_amd.runtime import GraphRunner
from rag_tl_domainllm_optimizer_amd.tokenizer import Tokenizer
from rag_tl_domainllm_optimizer_amd.train.common import score_sequences

DEV = "cuda"
BF16 = torch.bfloat16
INV_TEMP = 1 / 0.7  # sampling temperature of the rollouts and answers


# ---------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # one user's question: embed the query, search the corpus (RagPipeline.retrieve)
        dict(name="retrieve_1", kind="retrieve", queries=1, words=12, docs=100_000, k=3),
        # sentences of a reward batch or of a corpus being indexed (reward encoder)
        dict(name="embed_256", kind="embed", encoder="mpnet-base", texts=256, lo=16, hi=160),
        # the same with the retrieval encoder, a large indexing batch
        dict(name="embed_1024", kind="embed", encoder="minilm-l6", texts=1024, lo=20, hi=120),
        # one answer being written: every token is one such step
        dict(name="decode_1", kind="decode", model="mistral-7b", rows=1, lo=300, hi=300, fp8=False),
        # continuous batching: the rows of a serving batch are at different lengths
        dict(name="decode_48", kind="decode", model="mistral-7b", rows=48, lo=150, hi=1200, fp8=False),
        # PPO rollouts
        dict(name="decode_256", kind="decode", model="mistral-7b", rows=256, lo=173, hi=301, fp8=False),
        # retrieval-augmented prompts of a rollout batch, lengths as documents give them
        dict(name="prompt_32", kind="prompt", model="mistral-7b", rows=32, lo=90, hi=320),
        # one PPO minibatch: forward, loss, backward of the adapters
        dict(name="update_16", kind="update", model="mistral-7b", rows=16, prompt_lo=120, prompt_hi=173, new=128),
        # layered decoders: prompts (a batch of documents; one long one) and serving batches
        dict(name="vezatar_prompt", kind="prompt", model="vezatar-7b", rows=8, lo=700, hi=1024),
        dict(name="vezatar_decode", kind="decode", model="vezatar-7b", rows=16, lo=500, hi=1500, fp8=False),
        dict(name="pafolorn_prompt", kind="prompt", model="pafolorn-7b", rows=2, lo=3000, hi=4096),
        dict(name="pafolorn_decode", kind="decode", model="pafolorn-7b", rows=64, lo=300, hi=1100, fp8=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["retrieve", "embed", "decode", "decode", "prompt", "prompt", "update"])
    if kind == "retrieve":
        return dict(kind=kind, queries=_log(rng, 1, 256), words=rng.randint(4, 40), docs=_log(rng, 10_000, 200_000),
                    k=rng.randint(1, 10))
    if kind == "embed":
        lo = rng.randint(4, 60)
        name = rng.choice(["mpnet-base", "minilm-l6"])
        return dict(kind=kind, encoder=name, texts=_log(rng, 1, 256 if name == "mpnet-base" else 1024), lo=lo,
                    hi=lo + rng.randint(0, 100))
    if kind == "update":
        lo = rng.randint(30, 170)
        return dict(kind=kind, model=rng.choice(["mistral-7b", "mistral-2k"]), rows=rng.randint(4, 16), prompt_lo=lo,
                    prompt_hi=lo + rng.randint(0, 40), new=rng.randint(32, 128))
    if kind == "prompt":
        model = rng.choice(["mistral-7b", "mistral-2k", "vezatar-7b", "vezatar-2k", "pafolorn-7b", "pafolorn-2k"])
        mean = _log(rng, 60, 3500)
        rows = max(1, min(64, _log(rng, 500, 7000) // mean))
        return dict(kind=kind, model=model, rows=rows, lo=max(1, mean - rng.randint(0, mean // 2)),
                    hi=mean + rng.randint(0, mean // 8))
    model, fp8 = rng.choice([("mistral-7b", False), ("mistral-2k", False), ("llama2-13b", False), ("llama2-13b", True),
                             ("vezatar-7b", False), ("vezatar-2k", False), ("pafolorn-7b", False), ("pafolorn-2k", False)])
    rows = _log(rng, 1, 256)
    lo = _log(rng, 20, 1200 if rows < 64 else 300)
    return dict(kind=kind, model=model, rows=rows, lo=lo, hi=lo + rng.randint(0, lo), fp8=fp8)


# ---------------------------------------------------------------------------------------------- models
def _config(name, kind="decode"):
    cfg = models.resolve_preset(name)
    n = 2 if kind == "update" else 4
    return dataclasses.replace(cfg, num_layers=n, layers=cfg.layers[:n] if cfg.is_layered else None)


@torch.no_grad()
def _weights(model, g):
    """Random weights of a trained model's scales: norms around 1, decays from slow to fast, a router that prefers
    some experts."""
    for name, p in model.named_parameters():
        leaf = name.rsplit(".", 1)[-1]
        if "lora" in name:
            continue
        if leaf.endswith("_b"):
            p.normal_(0, 0.02, generator=g)
        elif "norm" in leaf or "ln" in leaf:
            p.normal_(1, 0.1, generator=g)
        elif leaf in ("ls1", "ls2"):
            p.normal_(0.7, 0.1, generator=g)
        elif leaf in ("A_log", "dt_bias"):
            p.normal_(-1, 1, generator=g)
        elif leaf == "conv_w":
            p.normal_(0.3, 0.5, generator=g)
        elif leaf == "sink":
            p.normal_(0, 1, generator=g)
        elif leaf == "correction":
            p.normal_(0, 0.001, generator=g)
        elif leaf == "router_w":
            p.normal_(0, 0.08, generator=g)
        else:
            p.normal_(0, 0.02, generator=g)


def _decoder(case, seed, g):
    cfg = _config(case["model"], case["kind"])
    m = models.model_class(cfg)(cfg, device=DEV, dtype=BF16, init=False).eval()
    _weights(m, g)
    if not cfg.tie_embeddings:
        m.embed.normal_(0, 1, generator=g)
    if not cfg.tie_embeddings and case["kind"] != "update":
        # one next token stands out, as from a trained model
        perm = torch.randperm(cfg.vocab_size, generator=g, device=DEV)
        m.lm_head[perm] += 0.02 * m.embed
    return m


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _lengths(case, seed, lo="lo", hi="hi"):
    r = random.Random(seed * 7 + 1)
    n = [r.randint(case[lo], case[hi]) for _ in range(case["rows"])]
    n[0] = case[hi]
    return n


_TOKENIZERS = {}


def _encoder(name, g):
    cfg = models.resolve_preset(name)
    m = models.SentenceEncoder(cfg, device=DEV, dtype=BF16, init=False).eval()
    _weights(m, g)
    if name not in _TOKENIZERS:
        t = Tokenizer.synthetic(cfg.vocab_size, cfg.arch)
        _TOKENIZERS[name] = t, t.words()
    t, words = _TOKENIZERS[name]
    return Encoder(m, t, max_length=128 if name == "minilm-l6" else 256), words


def _texts(words, n, lo, hi, r):
    return [" ".join(r.choices(words, k=r.randint(lo, hi))) for _ in range(n)]


# ---------------------------------------------------------------------------------------------- states
def prepare(case, seed):
    with torch.no_grad():
        return {"retrieve": _prepare_retrieve, "embed": _prepare_embed, "decode": _prepare_decode, "prompt": _prepare_prompt,
                "update": _prepare_update}[case["kind"]](case, seed)


def run(state):
    return {"retrieve": _run_retrieve, "embed": _run_embed, "decode": _run_decode, "prompt": _run_prompt,
            "update": _run_update}[state["case"]["kind"]](state)


# -- retrieval
def _prepare_retrieve(case, seed):
    """A trained index over documents that lie around the embeddings of texts; every query has its own few documents
    nearby, at different distances."""
    g, r = _generator(seed), random.Random(seed)
    enc, words = _encoder("minilm-l6", g)
    queries = _texts(words, case["queries"], case["words"], case["words"], r)
    around = enc.encode(_texts(words, 1024, 8, 40, r))
    near = enc.encode(queries)
    n, k, nlist = case["docs"], case["k"], 512

    def noise(rows, size):
        z = torch.randn(rows, enc.dim, generator=g, device=DEV)
        return z * (size / math.sqrt(enc.dim))
    docs = around[torch.randint(0, len(around), (n - k * len(queries),), generator=g, device=DEV)]
    docs = docs + noise(len(docs), 1.0)
    step = torch.linspace(0.1, 0.6, k, device=DEV).repeat_interleave(len(queries))[:, None]
    docs = F.normalize(torch.cat([docs, near.repeat(k, 1) + noise(k * len(queries), 1.0) * step]), dim=-1)
    docs = docs[torch.randperm(n, generator=g, device=DEV)].to(BF16).float()
    cen = docs[torch.randperm(n, generator=g, device=DEV)[:nlist]]
    for _ in range(3):
        a = (docs @ cen.t()).argmax(-1)
        cen = F.normalize(torch.zeros_like(cen).index_add_(0, a, docs) + 1e-6 * cen, dim=-1)
    a, order = torch.sort((docs @ cen.t()).argmax(-1), stable=True)
    index = IVFIndex(enc.dim, nlist, "ip", DEV, nprobe=16)
    index.load_state({"vecs": docs[order], "ids": order, "centroids": cen,
                      "offsets": torch.searchsorted(a, torch.arange(nlist + 1, device=DEV)).cpu()})
    return dict(case=case, enc=enc, index=index, queries=queries)


def _run_retrieve(s):
    q = s["enc"].encode(s["queries"])
    scores, ids = s["index"].search(q, s["case"]["k"])
    return {"query": q, "scores": scores, "ids": ids}


# -- sentence embedding
def _prepare_embed(case, seed):
    g, r = _generator(seed), random.Random(seed)
    enc, words = _encoder(case["encoder"], g)
    return dict(case=case, enc=enc, texts=_texts(words, case["texts"], case["lo"], case["hi"], r))


def _run_embed(s):
    return s["enc"].encode(s["texts"])


# -- one decoded token per row
def _fill_fp8(cache, cfg, rows, slots, g):
    for li in range(cfg.num_layers):
        qkv = torch.randn(rows * slots, cfg.qkv_dim, generator=g, device=DEV, dtype=BF16)
        ks, vs = cache.scales(li)
        ops.kv_store_fp8(qkv, cache.k[li], cache.v[li], ks, vs, rows, slots, cfg.num_heads)


def _prepare_decode(case, seed):
    """A model in the middle of generation: caches hold every row's context, the decode step is captured (as the
    generators do) with the sampler behind it."""
    g = _generator(seed)
    m = _decoder(case, seed, g)
    cfg, rows = m.cfg, case["rows"]
    if case["fp8"]:
        m.set_fp8(True)
    n = _lengths(case, seed)  # tokens in the cache; the next one goes behind them
    tok = torch.randint(3, cfg.vocab_size, (rows,), generator=g, device=DEV)
    active = torch.ones(rows, dtype=torch.uint8, device=DEV)
    offset = torch.zeros(1, dtype=torch.long, device=DEV)
    sampled = torch.zeros(rows, dtype=torch.long, device=DEV)
    sampled_lp = torch.zeros(rows, dtype=torch.float32, device=DEV)
    s = dict(case=case, model=m, tok=tok, n=n, sampled=sampled)
    if cfg.is_layered:
        cache = m.make_cache(rows, max(n) + 1)
        for b in range(rows):
            cache.reserve(b, n[b] + 1)
        cache.sync()
        held = [t for t in (cache.pool(i) for i in range(cfg.num_layers)) if t is not None]
        for t in held:
            t.normal_(0, 1, generator=g)
        states = [t for i in range(cfg.num_layers) for t in cache.state(i)]
        for t in states:
            t.normal_(0, 0.1 if t.dtype == torch.float32 else 1.3, generator=g)
        pos = torch.tensor(n, dtype=torch.int32, device=DEV)
        args = (tok, pos, None, None, None, cache.rows_view(0, rows))
        s.update(cache=cache, pos=pos, held=held + states)
    else:
        slots = (max(n) + 64) // 64 * 64
        cache = KVCache(cfg.num_layers, rows, cfg.num_kv_heads, slots, cfg.head_dim, torch.device(DEV), BF16, fp8=case["fp8"])
        if case["fp8"]:
            _fill_fp8(cache, cfg, rows, slots, g)
        else:
            cache.k.normal_(0, 1, generator=g)
            cache.v.normal_(0, 1, generator=g)
        slot = torch.tensor(n, dtype=torch.int32, device=DEV)
        start = torch.zeros_like(slot)
        ws = ops.decode_workspace(rows, cfg.num_heads, cfg.num_kv_heads, cfg.head_dim, slots, DEV)
        args = (tok, slot, slot, slot + 1, start, cache, ws)
        s.update(cache=cache, held=[cache.k, cache.v])
    out = {}

    def step():
        with torch.no_grad():
            out["logits"] = m.logits(m.decode(*args))
            ops.sample(out["logits"], INV_TEMP, 50, 1.0, False, 0, offset, active, sampled, sampled_lp)
    if hasattr(m, "refresh_decode_weights"):
        m.refresh_decode_weights(rows)
    # the graph goes by these tensors' addresses: they live as long as it does
    runner, keep = GraphRunner(), (tok, active, offset, sampled, sampled_lp, args)
    if cfg.is_layered:
        with cache.parked():
            runner.capture(step, keep=keep)
    else:
        runner.capture(step, keep=keep)
    s.update(runner=runner, out=out)
    return s


def _run_decode(s):
    s["runner"].replay()
    return {"logits": s["out"]["logits"], "tokens": s["sampled"], "held": s["held"]}


# -- prompts
def _prepare_prompt(case, seed):
    g, r = _generator(seed), random.Random(seed)
    m = _decoder(case, seed, g)
    cfg, n = m.cfg, _lengths(case, seed)
    prompts = [[r.randrange(3, cfg.vocab_size) for _ in range(k)] for k in n]
    s = dict(case=case, model=m, prompts=prompts, n=n)
    if cfg.is_layered:
        pages = len(n) * ((case["hi"] + PAGE - 1) // PAGE)
        s["engine"] = StepEngine(m, len(n), pages * PAGE, case["hi"])
    else:
        S = max(n)
        ids = torch.zeros(len(n), S, dtype=torch.long)
        for b, p in enumerate(prompts):
            ids[b, S - n[b]:] = torch.tensor(p)
        start = torch.tensor([S - k for k in n], dtype=torch.int32)
        cache = KVCache(cfg.num_layers, len(n), cfg.num_kv_heads, S, cfg.head_dim, torch.device(DEV), BF16)
        cache.k.zero_()
        cache.v.zero_()
        s.update(ids=ids.to(DEV), start=start.to(DEV), host_start=start.numpy(), cache=cache, packed=sum(n) < 0.97 * len(n) * S)
    return s


def _run_prompt(s):
    m = s["model"]
    if m.cfg.is_layered:
        eng = s["engine"]
        rows = [eng.admit() for _ in s["prompts"]]
        logits = eng.step([(row, p, [len(p) - 1]) for row, p in zip(rows, s["prompts"])])
        for row in reversed(rows):
            eng.release(row)
        held = [t for i in range(m.cfg.num_layers) for t in [eng.cache.pool(i), *eng.cache.state(i)] if t is not None]
        return {"logits": logits, "held": held}
    with torch.no_grad():
        B, S = s["ids"].shape
        packed = models.packed_index(s["host_start"], [S] * B, S, s["ids"].device) if s["packed"] else None
        h = m.prefill(s["ids"], s["start"], s["cache"], packed=packed)
        return {"logits": m.logits(h), "held": [s["cache"].k, s["cache"].v]}


# -- PPO update
def _prepare_update(case, seed):
    """A minibatch of rollouts: responses behind left-padded prompts, the log-probs they were drawn with (the policy's
    own, up to the decode engine's numerics), advantages and returns; adapters in the middle of training."""
    g = _generator(seed)
    m = _decoder(case, seed, g)
    cfg, rows, T = m.cfg, case["rows"], case["new"]
    m.add_lora(16, 32.0, "all")
    for p in m.lora_parameters():
        p.normal_(0, 0.01, generator=g)
    m.freeze_base()
    vh = models.ValueHead(cfg.hidden_size, device=DEV)
    flat = ops.flat_params(list(m.lora_parameters()) + list(vh.parameters()))
    opt = ops.FusedAdamW(flat, lr=5e-5, max_grad_norm=0.5)
    m.refresh_lora()
    n = _lengths(case, seed, "prompt_lo", "prompt_hi")
    S = max(n)
    r = random.Random(seed)
    new = [T] + [T if r.random() < 0.7 else r.randint(max(1, T // 4), T) for _ in range(rows - 1)]
    prompt = torch.randint(3, cfg.vocab_size, (rows, S), generator=g, device=DEV)
    resp = torch.randint(3, cfg.vocab_size, (rows, T), generator=g, device=DEV)
    start, lens = torch.tensor([S - k for k in n]), torch.tensor(new)
    s = dict(case=case, model=m, vh=vh, flat=flat, opt=opt, prompt=prompt, resp=resp, start=start.to(DEV), lens=lens.to(DEV),
             host=(start.numpy(), lens.numpy()))

    def randn():
        return torch.randn(rows, T, generator=g, device=DEV)
    lp, _, _, _ = score_sequences(m, prompt, s["start"], resp, s["lens"], INV_TEMP, None, lengths=s["host"])
    # most ratios near 1, some beyond the clip's edges, none so close to them that rounding takes it across
    u = 2 * torch.rand(rows, T, generator=g, device=DEV) - 1
    far = torch.rand(rows, T, generator=g, device=DEV) < 0.07
    old = lp + torch.where(far, 0.4 * u.sign() + 0.1 * u, 0.12 * u)
    s.update(old=old, ref=lp + 0.2 * randn(), adv=randn(), ret=randn())
    return s


def _run_update(s):
    s["opt"].zero_grad()
    lp, ent, val, mask = score_sequences(s["model"], s["prompt"], s["start"], s["resp"], s["lens"], INV_TEMP, s["vh"],
                                         lengths=s["host"])
    loss, _ = ops.ppo_loss(lp, val, ent, s["old"], s["adv"], s["ret"], mask, 0.2, 0.5, 0.01, None, None, s["ref"], 0.05)
    loss.backward()
    return {"logp": lp, "entropy": ent, "values": val, "grad": s["flat"].grad}


# ---------------------------------------------------------------------------------------------- work
def _encoder_work(name, tokens, square):
    c = models.resolve_preset(name)
    H, F_ = c.hidden_size, c.intermediate_size
    per = 4 * H * H + 2 * H * F_
    return 2 * c.num_layers * (per * tokens + 2 * H * square), 2 * (c.num_layers * per + H * tokens) + 4 * H * tokens


def _layer_sizes(layer, width):
    """(weights read by a token, weights of the layer, cached bytes of a token, state bytes of a row, flops of a
    (query, key) pair, window) of one layered decoder layer"""
    mx, ml = layer.mixer, layer.mlp
    kv = state = pair = w = window = 0
    branches = [mx.left, mx.right] if hasattr(mx, "left") else [mx]
    for x in branches:
        if hasattr(x, "kv_rank"):
            own = x.kv_from is None
            w += width * (x.heads * (x.dim + x.rot_dim + 2 * x.vdim) + (x.kv_rank + x.rot_dim if own else 0))
            w += x.heads * (x.dim + x.vdim) * x.kv_rank
            kv += 2 * (x.kv_rank + x.rot_dim)
            pair += 2 * x.heads * (x.dim + x.rot_dim + x.vdim)
        elif hasattr(x, "conv"):
            c = 2 * x.kv_heads * x.dim + x.heads * x.vdim
            w += width * (c + x.heads) + x.heads * x.vdim * width
            if x.channel:
                w += width * (x.a_rank + x.g_rank) + x.heads * (x.a_rank * x.dim + x.g_rank * x.vdim)
            else:
                w += width * (x.heads * x.vdim + x.heads)
            state += 8 * x.heads * x.dim * x.vdim + 2 * x.conv * c
        else:
            w += width * (x.heads * (x.dim + x.vdim) + x.kv_heads * (x.dim + x.vdim))
            kv += 2 * x.kv_heads * (x.dim + x.vdim)
            pair += 2 * x.heads * (x.dim + x.vdim)
            window = x.window
    if ml is None:
        return w, w, kv, state, pair, window
    if ml.kind == "moe":
        e = 3 * width * ml.ff
        per = ml.top * e + 3 * width * ml.shared_ff + width * ml.experts
        return w + per, w + ml.experts * e + 3 * width * ml.shared_ff, kv, state, pair, window
    f = (2 if ml.kind == "relu2" else 3) * width * ml.ff
    return w + f, w + f, kv, state, pair, window


def _decoder_work(cfg, new, ctx, outs, elem=2.0, kv_elem=2):
    """``new`` tokens per row behind ``ctx`` cached ones, logits of ``outs`` tokens; ``elem`` bytes a weight"""
    H, tokens = cfg.hidden_size, sum(new)
    pairs = sum(n * c + n * (n + 1) // 2 for n, c in zip(new, ctx))
    head = cfg.vocab_size * H
    flops = 2.0 * head * outs
    nbytes = 2.0 * head + 4 * cfg.vocab_size * outs + 2 * H * tokens
    if not cfg.is_layered:
        w = H * cfg.qkv_dim + H * cfg.num_heads * cfg.head_dim + 3 * H * cfg.intermediate_size
        kv = 2 * kv_elem * cfg.num_kv_heads * cfg.head_dim
        flops += cfg.num_layers * (2.0 * w * tokens + 4.0 * cfg.num_heads * cfg.head_dim * pairs)
        return nbytes + cfg.num_layers * (elem * w + kv * (sum(ctx) + tokens)), flops
    for layer in cfg.layers:
        act, w, kv, state, pair, window = _layer_sizes(layer, H)
        if layer.mlp is not None and layer.mlp.kind == "moe":
            # distinct experts that the tokens are expected to read
            e = 3 * H * layer.mlp.ff
            miss = (1 - layer.mlp.top / layer.mlp.experts) ** tokens
            w -= layer.mlp.experts * e * miss
        flops += 2.0 * act * tokens + pair * pairs + state / 8 * 2 * tokens * 4
        nbytes += 2.0 * w + kv * (sum(ctx) + tokens) + state * (2 if ctx[0] else 1) / 2 * len(new)
    return nbytes, flops


def work(case):
    kind = case["kind"]
    if kind == "retrieve":
        t = (case["words"] + 2) * case["queries"]
        fl, by = _encoder_work("minilm-l6", t, t * (case["words"] + 2))
        # the probed lists, 16 of 512, read once by each query (all of them at most once in all)
        scan = min(1.0, case["queries"] * 16 / 512) * case["docs"] * 384 * 2
        return {"bytes": by + scan + 512 * 384 * 2, "flops": fl + 2 * case["queries"] * 384 * (512 + case["docs"] / 32)}
    if kind == "embed":
        mean = min((case["lo"] + case["hi"]) / 2 + 2, 256)
        fl, by = _encoder_work(case["encoder"], case["texts"] * mean, case["texts"] * mean * mean)
        return {"bytes": by, "flops": fl}
    cfg = _config(case["model"], kind)
    if kind == "update":
        mean, T = (case["prompt_lo"] + case["prompt_hi"]) / 2, case["new"] * 0.9
        tokens = case["rows"] * (mean + T)
        H = cfg.hidden_size
        w = H * cfg.qkv_dim + H * cfg.num_heads * cfg.head_dim + 3 * H * cfg.intermediate_size
        pairs = case["rows"] * (mean + T) ** 2 / 2
        # forward and the inputs' gradients (the base weights have none)
        fl = cfg.num_layers * (4 * w * tokens + 3.5 * 4 * cfg.num_heads * cfg.head_dim * pairs)
        fl += 4 * H * cfg.vocab_size * case["rows"] * T
        return {"bytes": 4.0 * (cfg.num_layers * w + H * cfg.vocab_size), "flops": fl}
    n = [(case["lo"] + case["hi"]) // 2] * case["rows"]
    if kind == "prompt":
        by, fl = _decoder_work(cfg, n, [0] * len(n), len(n))
    else:
        by, fl = _decoder_work(cfg, [1] * len(n), n, len(n), 1.0 if case["fp8"] else 2.0, 1 if case["fp8"] else 2)
    return {"bytes": by, "flops": fl}


def tolerance(case):
    """bf16 operands with 32-bit sums, 0.004 to 0.02 off the exact result; the ids of a search, the sampled tokens and
    the bytes of an 8-bit cache may differ in a tie. The widest for gradients, which sum terms of both signs, and for
    experts, where a close routing call may fall the other way."""
    if case["kind"] in ("retrieve", "embed"):
        return {"rel": 0.02, "max": 0.3, "differ": 0.01}
    wide = case["kind"] == "update" or case["model"].startswith("vezatar")
    return {"rel": 0.03 if wide else 0.02, "max": 0.5, "differ": 0.01}


# ---------------------------------------------------------------------------------------------- 64 bits
def exact(case, seed):
    if case.get("fp8"):
        return None  # scaled 8-bit weights and caches have no plain form
    s = prepare(case, seed)
    if case["kind"] == "update":
        return _exact_update(s)
    with torch.no_grad():
        if case["kind"] in ("retrieve", "embed"):
            return _exact_encode(s)
        m = s["model"]
        fn = {"vezatar": _exact_vezatar, "pafolorn": _exact_pafolorn}.get(m.cfg.arch, _exact_causal)
        return fn(s)


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _mm(x, w):
    return x @ w.double().t()


def _exact_encode(s):
    enc = s["enc"]
    m, c = enc.model, enc.model.cfg
    texts = s.get("queries") or s["texts"]
    tokens = enc.tokenizer.encode_batch(texts, True, enc.max_length)
    H, nh, D = c.hidden_size, c.num_heads, c.head_dim

    def ln(x, w, b):
        return F.layer_norm(x, (H,), w.double(), b.double(), c.norm_eps)
    S = max(len(t) for t in tokens)
    ids = torch.zeros(len(tokens), S, dtype=torch.long)
    for b, t in enumerate(tokens):
        ids[b, :len(t)] = torch.tensor(t)
    out = []
    for b0 in range(0, len(tokens), 64):
        i = ids[b0:b0 + 64].to(DEV)
        B = i.shape[0]
        n = torch.tensor([len(t) for t in tokens[b0:b0 + 64]], device=DEV)
        ar = torch.arange(S, device=DEV)
        valid = ar[None] < n[:, None]
        pos = ar + c.pad_token_id + 1 if c.arch == "mpnet" else ar
        x = m.word_embed.double()[i] + m.pos_embed.double()[pos.clamp(max=c.max_position - 1)]
        if c.type_vocab_size:
            x = x + m.type_embed.double()[0]
        x = ln(x, m.emb_ln_w, m.emb_ln_b)
        bias = 0
        if c.arch == "mpnet":
            rel = ar[None] - ar[:, None]
            half = c.relative_buckets // 2
            d = rel.abs()
            far = half // 2 + (torch.log(d.float().clamp(min=1) / (half // 2)) / math.log(c.relative_max_distance / (half // 2))
                               * (half - half // 2)).long()
            bias = m.rel_bias.double()[(rel > 0).long() * half + torch.where(d < half // 2, d, far.clamp(max=half - 1))]
            bias = bias.permute(2, 0, 1)
        for L in m.layers:
            q, k, v = (_mm(x, L.qkv_w) + L.qkv_b.double()).view(B, S, 3, nh, D).permute(2, 0, 3, 1, 4)
            sc = q @ k.transpose(-1, -2) / math.sqrt(D) + bias
            a = torch.softmax(sc.masked_fill(~valid[:, None, None], -math.inf), -1) @ v
            a = _mm(a.transpose(1, 2).reshape(B, S, H), L.o_w) + L.o_b.double()
            x = ln(x + a, L.ln1_w, L.ln1_b)
            f = _mm(F.gelu(_mm(x, L.fc1_w) + L.fc1_b.double()), L.fc2_w) + L.fc2_b.double()
            x = ln(x + f, L.ln2_w, L.ln2_b)
        out.append(F.normalize((x * valid[..., None]).sum(1) / n[:, None], dim=-1))
    e = torch.cat(out)
    if "index" not in s:
        return e
    # the best of the lists whose centroids are nearest
    index = s["index"]
    near = (e @ index.centroids.double().t()).topk(index.nprobe, -1).indices
    probed = torch.zeros(len(e), index.nlist, dtype=torch.bool, device=DEV).scatter(1, near, True)
    of = torch.repeat_interleave(torch.arange(index.nlist, device=DEV), index.lsize.long())
    sc = (e @ index.vecs.double().t()).masked_fill(~probed[:, of], -math.inf)
    return {"query": e, "scores": sc.topk(s["case"]["k"], -1).values, "ids": None}


def _halves(x, pos, base, dims):
    """x [T, heads, D]: column i < dims / 2 turned together with column i + dims / 2"""
    f = base ** (-torch.arange(0, dims, 2, dtype=torch.float64, device=x.device) / dims)
    a = pos.double()[:, None] * f
    c, s = a.cos()[:, None], a.sin()[:, None]
    h = dims // 2
    u, v = x[..., :h], x[..., h:dims]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., dims:]], -1)


def _attend(q, k, v, i, scale, see=None, softcap=0.0, sink=None):
    """q [T, H, D] at positions i over keys k [N, G, D], values v [N, G, V] at positions 0.. -> [T, H * V]"""
    T, H = q.shape[:2]
    k, v = (t.repeat_interleave(H // t.shape[1], 1).transpose(0, 1) for t in (k, v))
    sc = q.transpose(0, 1) @ k.transpose(-1, -2) * scale
    if softcap:
        sc = softcap * torch.tanh(sc / softcap)
    j = torch.arange(k.shape[1], device=q.device)[None]
    ok = j <= i[:, None]
    if see is not None:
        ok = ok & see(i[:, None], j)
    sc = sc.masked_fill(~ok, -math.inf)
    if sink is not None:
        sc = torch.cat([sc, sink.double().view(H, 1, 1).expand(-1, T, 1)], -1)
    p = torch.softmax(sc, -1)[..., :k.shape[1]]
    return (p @ v).transpose(0, 1).reshape(T, -1)


def _causal_layers(m, x, attend, lora=None):
    c = m.cfg

    def proj(layer, h, w, names):
        y = _mm(h, w)
        if lora is None:
            return y
        parts, at = [], 0
        for nm, rows in names:
            A, B = lora[layer][nm]
            parts.append(y[:, at:at + rows] + 2.0 * ((h @ A.t()) @ B.t()))
            at += rows
        return torch.cat(parts, 1)
    D, Hq, Hk, Fi, H = c.head_dim, c.num_heads, c.num_kv_heads, c.intermediate_size, c.hidden_size
    for li, L in enumerate(m.layers):
        h = _rms(x, L.ln1_w, c.norm_eps)
        qkv = proj(li, h, L.qkv_w, [("q_proj", Hq * D), ("k_proj", Hk * D), ("v_proj", Hk * D)])
        q, k, v = qkv.split([Hq * D, Hk * D, Hk * D], 1)
        a = attend(li, q.view(-1, Hq, D), k.view(-1, Hk, D), v.view(-1, Hk, D))
        x = x + proj(li, a, L.o_w, [("o_proj", H)])
        h = _rms(x, L.ln2_w, c.norm_eps)
        gt, u = proj(li, h, L.gate_up_w, [("gate_proj", Fi), ("up_proj", Fi)]).chunk(2, 1)
        x = x + proj(li, F.silu(gt) * u, L.down_w, [("down_proj", H)])
    return _rms(x, m.norm_w, c.norm_eps)


def _exact_causal(s):
    m, c = s["model"], s["model"].cfg
    decode, n = s["case"]["kind"] == "decode", s["n"]
    kc, vc = s["cache"].k, s["cache"].v
    scale = c.head_dim ** -0.5

    def see(i, j):
        return i - j < c.sliding_window
    see = see if c.sliding_window else None
    if decode:
        x = m.embed.double()[s["tok"]]
        pos = torch.tensor(n, device=DEV)
        kc, vc = kc.double(), vc.double()

        def attend(li, q, k, v):
            q, k = _halves(q, pos, c.rope_theta, c.head_dim), _halves(k, pos, c.rope_theta, c.head_dim)
            out = []
            for b in range(len(n)):
                kc[li, b, :, n[b]], vc[li, b, :, n[b]] = k[b], v[b]
                e = n[b] + 1
                out.append(_attend(q[b:b + 1], kc[li, b, :, :e].transpose(0, 1), vc[li, b, :, :e].transpose(0, 1),
                                   pos[b:b + 1], scale, see))
            return torch.cat(out)
        h = _causal_layers(m, x, attend)
        return {"logits": _mm(h, m.lm_head), "tokens": None, "held": [kc, vc]}
    S = max(n)
    kc, vc = torch.zeros_like(kc, dtype=torch.float64), torch.zeros_like(vc, dtype=torch.float64)
    x = m.embed.double()[torch.cat([torch.tensor(p) for p in s["prompts"]]).to(DEV)]

    def attend(li, q, k, v):
        out, at = [], 0
        for b, L in enumerate(n):
            pos = torch.arange(L, device=DEV)
            r = slice(at, at + L)
            qb, kb = _halves(q[r], pos, c.rope_theta, c.head_dim), _halves(k[r], pos, c.rope_theta, c.head_dim)
            kc[li, b, :, S - L:], vc[li, b, :, S - L:] = kb.transpose(0, 1), v[r].transpose(0, 1)
            out.append(_attend(qb, kb, v[r], pos, scale, see))
            at += L
        return torch.cat(out)
    h = _causal_layers(m, x, attend)
    last = torch.cumsum(torch.tensor(n), 0).to(DEV) - 1
    # without packing the pads' rows are computed too, to no end
    return {"logits": _mm(h[last], m.lm_head), "held": [kc, vc] if s["packed"] or min(n) == S else [None, None]}


def _exact_update(s):
    m, c, case = s["model"], s["model"].cfg, s["case"]
    B, S = s["prompt"].shape
    T = case["new"]
    start, lens = s["host"]
    leaf, lora = {}, []
    for layer in m.layers:
        d = {}
        for key, p in layer.lora_params.items():
            leaf[id(p)] = p.detach().double().requires_grad_(True)
            d.setdefault(key[:-2], {})[key[-1]] = leaf[id(p)]
        lora.append({k: (v["A"], v["B"]) for k, v in d.items()})
    vw, vb = s["vh"].linear.weight, s["vh"].linear.bias
    for p in (vw, vb):
        leaf[id(p)] = p.detach().double().requires_grad_(True)
    seq = torch.cat([s["prompt"], s["resp"]], 1)
    rows = [seq[b, int(start[b]):S + int(lens[b]) - 1] for b in range(B)]
    scale = c.head_dim ** -0.5

    def attend(li, q, k, v):
        out, at = [], 0
        for t in rows:
            L = len(t)
            pos = torch.arange(L, device=DEV)
            r = slice(at, at + L)
            out.append(_attend(_halves(q[r], pos, c.rope_theta, c.head_dim), _halves(k[r], pos, c.rope_theta, c.head_dim),
                               v[r], pos, scale))
            at += L
        return torch.cat(out)
    h = _causal_layers(m, m.embed.detach().double()[torch.cat(rows)], attend, lora)
    sel, at = [], 0
    for b, t in enumerate(rows):
        first = S - 1 - int(start[b])
        sel.append(torch.arange(at + first, at + first + int(lens[b]), device=DEV))
        at += len(t)
    mask = torch.arange(T, device=DEV)[None] < s["lens"][:, None]
    h = h[torch.cat(sel)]
    lsm = torch.log_softmax(h @ m.lm_head.detach().double().t() * INV_TEMP, -1)
    lp = lsm.gather(1, s["resp"][mask][:, None])[:, 0]
    ent = -(lsm.exp() * lsm).sum(-1)
    val = h @ leaf[id(vw)][0] + leaf[id(vb)]
    old, ref, adv, ret = (s[k][mask].double() for k in ("old", "ref", "adv", "ret"))
    ratio = torch.exp(lp - old)
    loss = -torch.min(ratio * adv, ratio.clamp(0.8, 1.2) * adv).mean() + 0.25 * ((val - ret) ** 2).mean()
    d = ref - lp
    loss = loss - 0.01 * ent.mean() + 0.05 * (torch.exp(d) - d - 1).mean()
    loss.backward()
    flat = s["flat"]
    grad = torch.zeros(flat.numel, dtype=torch.float64, device=DEV)
    for p, o in zip(flat.params, flat.offsets):
        grad[o:o + p.numel()] = leaf[id(p)].grad.reshape(-1)

    def grid(x):
        return torch.zeros(B, T, dtype=torch.float64, device=DEV).masked_scatter(mask, x.detach())
    # a forward that is not packed gives entropies and values at masked places too, which nothing reads
    whole = len(torch.cat(rows)) < 0.97 * B * (S + T) or bool(mask.all())
    return {"logp": grid(lp), "entropy": grid(ent) if whole else None, "values": grid(val) if whole else None, "grad": grad}


def _rows_of(s):
    """per request: its tokens, their positions and its cache row"""
    if s["case"]["kind"] == "decode":
        return [(s["tok"][b:b + 1], torch.tensor([n], device=DEV), b) for b, n in enumerate(s["n"])]
    return [(torch.tensor(p, device=DEV), torch.arange(len(p), device=DEV), b) for b, p in enumerate(s["prompts"])]


def _spread(f, reqs, *xs):
    """f(request, its rows of xs) for every request, results one behind the other"""
    out, at = [], 0
    for r in reqs:
        n = len(r[0])
        out.append(f(r, *(x[at:at + n] for x in xs)))
        at += n
    return torch.cat(out)


def _outputs(s, reqs, logits, held):
    if s["case"]["kind"] == "decode":
        return {"logits": logits, "tokens": None, "held": held}
    last = torch.cumsum(torch.tensor([len(r[0]) for r in reqs]), 0).to(DEV) - 1
    return {"logits": logits(last), "held": held}


def _held_none(s):
    if s["case"]["kind"] == "decode":
        return [None] * len(s["held"])
    c = s["engine"].cache
    return [None for i in range(s["model"].cfg.num_layers) for t in [c.pool(i), *c.state(i)] if t is not None]


def _exact_vezatar(s):
    m, c = s["model"], s["model"].cfg
    reqs = _rows_of(s)
    x = m.embed.double()[torch.cat([r[0] for r in reqs])]
    pos = torch.cat([r[1] for r in reqs])
    cache = s.get("cache")

    def rotate(y, rot):
        sc, i = rot.scaling, torch.arange(rot.dims // 2, dtype=torch.float64, device=DEV)

        def at(turns):
            return rot.dims * math.log(sc.original / (2 * math.pi * turns)) / (2 * math.log(rot.base))
        lo, hi = max(math.floor(at(sc.fast)), 0), min(math.ceil(at(sc.slow)), rot.dims - 1)
        ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        f = rot.base ** (-2 * i / rot.dims)
        a = pos.double()[:, None] * (f / sc.factor * ramp + f * (1 - ramp))
        mult = 0.1 * math.log(sc.factor) + 1
        cs, sn = ((t * mult).view(len(pos), *[1] * (y.dim() - 2), -1) for t in (a.cos(), a.sin()))
        u, v = y[..., 0::2], y[..., 1::2]
        return torch.stack([u * cs - v * sn, v * cs + u * sn], -1).flatten(-2)
    eps, latents = c.norm_eps, {}
    for li, L in enumerate(m.layers):
        mx, sp = L.mix, c.layers[li].mixer
        H, D, R, V, C = sp.heads, sp.dim, sp.rot_dim, sp.vdim, sp.kv_rank
        h = _rms(x, L.norm1_w, eps)
        y = _mm(h, mx.in_w)
        own = sp.kv_from is None
        q, y = y[:, :H * (D + R)].view(-1, H, D + R), y[:, H * (D + R):]
        if own:
            lat = torch.cat([_rms(y[:, :C], mx.latent_norm_w, eps), rotate(y[:, C:C + R], sp.rot)], 1)
            latents[li] = {r[2]: t for r, t in zip(reqs, lat.split([len(r[0]) for r in reqs]))}
            if cache is not None:
                for tk, p, b in reqs:
                    n = int(p[0])
                    pages = cache.pool(li)[cache.table[b].long()[:n // PAGE + 1]].flatten(0, 1)[:n].double()
                    latents[li][b] = torch.cat([pages, latents[li][b]])
            y = y[:, C + R:]
        src = latents[li if own else sp.kv_from]
        uk, uv = mx.kv_up_w[:H * D], mx.kv_up_w[H * D:]
        q = torch.cat([q[..., :D], rotate(q[..., D:], sp.rot)], -1)

        def attend(r, qb):
            t = src[r[2]]
            k = torch.cat([_mm(t[:, :C], uk).view(-1, H, D), t[:, None, C:].expand(-1, H, -1)], -1)
            return _attend(qb, k, _mm(t[:, :C], uv).view(-1, H, V), r[1], sp.scale, sink=mx.sink)
        a = _spread(attend, reqs, q) * torch.sigmoid(y[:, :H * V])
        x = x + _rms(_mm(a, mx.o_w), L.norm1b_w, eps)
        h, f = _rms(x, L.norm2_w, eps), L.mlp
        if c.layers[li].mlp.kind == "dense":
            gt, u = _mm(h, f.gate_up_w).chunk(2, 1)
            gt, u = gt.clamp(max=f.glu.limit), u.clamp(-f.glu.limit, f.glu.limit)
            y = _mm(gt * torch.sigmoid(1.702 * gt) * (u + 1), f.down_w)
        else:
            ml = f.spec
            z = _mm(h, f.router_w)
            p = torch.softmax(z[:, :ml.experts], -1)
            idx = (p + f.correction.double()).topk(ml.top, -1).indices
            wt = torch.zeros_like(p).scatter(1, idx, p.gather(1, idx))
            wt = torch.cat([wt, torch.sigmoid(z[:, ml.experts:ml.experts + 1]).expand(-1, f.nshared)], 1)
            y = torch.zeros_like(h)
            for e in range(wt.shape[1]):
                t = torch.nonzero(wt[:, e]).flatten()
                gt, u = _mm(h[t], f.gate_up_w[e * 2 * ml.ff:(e + 1) * 2 * ml.ff]).chunk(2, 1)
                y[t] += wt[t, e:e + 1] * _mm(F.silu(gt) * u, f.down_w[e * c.hidden_size:(e + 1) * c.hidden_size])
        x = x + _rms(y, L.norm2b_w, eps)
    h = _rms(x, m.norm_w, eps)
    held = _held_none(s)
    if cache is not None:
        return _outputs(s, reqs, _mm(h, m.lm_head), held)
    return _outputs(s, reqs, lambda last: _mm(h[last], m.lm_head), held)


def _exact_pafolorn(s):
    m, c = s["model"], s["model"].cfg
    reqs, eps, cache = _rows_of(s), c.norm_eps, s.get("cache")
    pos = torch.cat([r[1] for r in reqs])
    sizes = [len(r[0]) for r in reqs]
    x = _rms(m.embed.double()[torch.cat([r[0] for r in reqs])], m.embed_norm_w, eps)
    held, pools = [], []

    def window(mix, sp, b, y, rows, li):
        H, G, D, V = sp.heads, sp.kv_heads, sp.dim, sp.vdim
        q, k, v = (y[:, rows[t][0]:rows[t][0] + rows[t][1]] for t in "qkv")
        q = _halves(_rms(q, b.q_norm_w, eps).view(-1, H, D), pos, sp.rot.base, sp.rot.dims)
        k = _halves(_rms(k, b.k_norm_w, eps).view(-1, G, D), pos, sp.rot.base, sp.rot.dims)

        def see(i, j):
            return (i - j < sp.window) | (j < sp.keep_first)

        def one(r, qb, kb, vb):
            if cache is not None:
                n = int(r[1][0])
                old = cache.pool(li).view(-1, G, PAGE, D + V)[cache.table[r[2]].long()[:n // PAGE + 1]]
                old = old.transpose(1, 2).flatten(0, 1)[:n].double()
                kb, vb = torch.cat([old[..., :D], kb]), torch.cat([old[..., D:], vb])
            return _attend(qb, kb, vb, r[1], sp.scale, see, sp.softcap)
        return _spread(one, reqs, q, k, v.view(-1, G, V))

    def delta(sp, b, y, rows, li):
        H, K, D, V, taps = sp.heads, sp.kv_heads, sp.dim, sp.vdim, sp.conv
        c0 = rows["q"][0]
        u = y[:, c0:c0 + b.channels]

        def col(name, n):
            return y[:, rows[name][0]:rows[name][0] + n]
        if sp.channel:
            a, z = _mm(col("a1", b.a2_w.shape[1]), b.a2_w), torch.sigmoid(_mm(col("g1", b.g2_w.shape[1]), b.g2_w))
        else:
            a, z = col("a", H), F.silu(col("g", H * V))
        decay = torch.exp(-torch.exp(b.A_log.double())[:, None] * F.softplus(a + b.dt_bias.double()).view(len(a), H, -1))
        beta = torch.sigmoid(col("b", H))

        def conv(r, ub):
            hist = torch.zeros(taps - 1, b.channels, dtype=torch.float64, device=DEV)
            if cache is not None:
                p, ring = int(r[1][0]), cache.state(li)[1][r[2]].double()
                for j in range(1, min(taps, p + 1)):
                    hist[taps - 1 - j] = ring[(p - j) % taps]
            t = torch.cat([hist, ub])
            return F.silu(sum(t[j:j + len(ub)] * b.conv_w[:, j].double() for j in range(taps)))
        u = _spread(conv, reqs, u)
        q, k, v = u[:, :K * D].view(-1, K, D), u[:, K * D:2 * K * D].view(-1, K, D), u[:, 2 * K * D:].view(-1, H, V)
        q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
        q, k = (t.repeat_interleave(H // K, 1) for t in (q * D ** -0.5, k))
        # all requests side by side, one token at a time
        S = torch.zeros(len(reqs), H, D, V, dtype=torch.float64, device=DEV)
        if cache is not None:
            S = cache.state(li)[0].double()
        at = torch.cumsum(torch.tensor([0] + sizes[:-1]), 0).to(DEV)
        n = torch.tensor(sizes, device=DEV)
        o = torch.zeros(len(u), H, V, dtype=torch.float64, device=DEV)
        for t in range(max(sizes)):
            live = torch.arange(len(reqs), device=DEV) if min(sizes) > t else torch.nonzero(n > t).flatten()
            i = at[live] + t
            St = S[live] * decay[i][..., None]
            w = beta[i][..., None] * (v[i] - (k[i][:, :, None] @ St)[:, :, 0])
            St = St + k[i][..., None] * w[:, :, None]
            S[live] = St
            o[i] = (q[i][:, :, None] @ St)[:, :, 0]
        held.append(S)
        o = _rms(o, b.out_norm_w, eps).reshape(len(u), -1)
        return o * z
    for li, L in enumerate(m.layers):
        mix = L.mix
        y = _mm(x, mix.in_w)
        parts = torch.zeros(len(x), mix.o_w.shape[1], dtype=torch.float64, device=DEV)
        for side, sp, mul in mix.sides:
            b, rows = getattr(mix, side), mix.rows[side]
            c0, n = mix.cols[side]
            f = delta(sp, b, y, rows, li) if hasattr(sp, "conv") else window(mix, sp, b, y, rows, li)
            parts[:, c0:c0 + n] = f * mul
        x = x + _rms(_mm(parts, mix.o_w), L.norm1_w, eps) * L.ls1.double()
        if L.mlp is not None:
            u = _mm(x, L.mlp.up_w).clamp(min=0)
            x = x + _rms(_mm(u * u, L.mlp.down_w), L.norm2_w, eps) * L.ls2.double()
    h = _rms(x, m.norm_w, eps) * c.logit_scale
    cc = cache if cache is not None else s["engine"].cache
    # of the caches, the recurrent states have one place per request; pages and rings are laid out by the framework
    states, order = iter(held), []
    for i in range(c.num_layers):
        st = cc.state(i)
        order.append(([None] if cc.pool(i) is not None else [], [next(states), None] if st else []))
    if cache is not None:
        held = [t for p, _ in order for t in p] + [t for _, q in order for t in q]
        return _outputs(s, reqs, _mm(h, m.embed), held)
    return _outputs(s, reqs, lambda last: _mm(h[last], m.embed), [t for p, q in order for t in p + q])
