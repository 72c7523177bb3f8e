"""Data parallelism on CPU with gloo (world 2): bucketed/overlapped all-reduce == one process on the
whole batch; seed-synchronised init; rank-sharded loader is disjoint and covering."""
import os
import socket

import pytest
import torch
import torch.multiprocessing as mp


def _free_port():
    s = socket.socket()
    s.bind(("127.0.0.1", 0))
    p = s.getsockname()[1]
    s.close()
    return p


def _examples(tok, n=8):
    words = tok.words()
    return [{"prompt": " ".join(words[i:i + 6]), "answer": " ".join(words[50 + i:50 + i + 4])} for i in range(n)]


def _worker(rank, world, port, out_dir, bucket_bytes):
    os.environ.update(RANK=str(rank), WORLD_SIZE=str(world), LOCAL_RANK=str(rank), MASTER_ADDR="127.0.0.1",
                      MASTER_PORT=str(port))
    from rag_tl_domainllm_optimizer_amd import models, parallel
    from rag_tl_domainllm_optimizer_amd.models.config import PRESETS
    from rag_tl_domainllm_optimizer_amd.tokenizer import Tokenizer
    from rag_tl_domainllm_optimizer_amd.train.sft import SFTConfig, SFTTrainer

    parallel.init(device="cpu")
    torch.manual_seed(0)
    cfg = PRESETS["tiny-llama"]
    tok = Tokenizer.synthetic(cfg.vocab_size, "llama")
    m = models.CausalLM(cfg, dtype=torch.float32, seed=1)
    tr = SFTTrainer(m, tok, SFTConfig(lr=1e-2, lora_r=4, lr_schedule="constant", warmup_steps=0, batch_size=4,
                                      bucket_mb=bucket_bytes / (1 << 20)))
    assert len(tr.sync.buckets) >= (2 if bucket_bytes < 4096 else 1)
    # make B non-zero so every LoRA parameter has a non-trivial gradient
    with torch.no_grad():
        for p in m.lora_parameters():
            p.normal_(0, 0.05)
    m.refresh_lora()
    ex = _examples(tok)
    mine = ex[rank::world]
    tr.opt.zero_grad()
    tr.sync.start()
    ids, start, tgt = tr.encode([e["prompt"] for e in mine], [e["answer"] for e in mine])
    loss, _ = tr.loss(ids, start, tgt)
    loss.backward()
    tr.sync.finish()
    if rank == 0:
        torch.save(tr.flat.grad.clone(), os.path.join(out_dir, "dp.pt"))
    parallel.barrier()
    parallel.shutdown()


@pytest.mark.parametrize("world,bucket_bytes", [(2, 1 << 10), (2, 64 << 20), (4, 1 << 12)])
def test_dp_allreduce_equals_single_process(tmp_path, world, bucket_bytes):
    from rag_tl_domainllm_optimizer_amd import models
    from rag_tl_domainllm_optimizer_amd.models.config import PRESETS
    from rag_tl_domainllm_optimizer_amd.tokenizer import Tokenizer
    from rag_tl_domainllm_optimizer_amd.train.sft import SFTConfig, SFTTrainer

    mp.start_processes(_worker, args=(world, _free_port(), str(tmp_path), bucket_bytes), nprocs=world,
                       start_method="spawn", join=True)
    dp = torch.load(tmp_path / "dp.pt")
    # single process on the full batch, accumulated over the same shards == mean of shard means
    torch.manual_seed(0)
    cfg = PRESETS["tiny-llama"]
    tok = Tokenizer.synthetic(cfg.vocab_size, "llama")
    m = models.CausalLM(cfg, dtype=torch.float32, seed=1)
    tr = SFTTrainer(m, tok, SFTConfig(lr=1e-2, lora_r=4, lr_schedule="constant", warmup_steps=0, batch_size=4))
    with torch.no_grad():
        for p in m.lora_parameters():
            p.normal_(0, 0.05)
    m.refresh_lora()
    ex = _examples(tok)
    tr.opt.zero_grad()
    for r in range(world):
        shard = ex[r::world]
        ids, start, tgt = tr.encode([e["prompt"] for e in shard], [e["answer"] for e in shard])
        loss, _ = tr.loss(ids, start, tgt)
        (loss / world).backward()
    tr.flat.relink_grads()
    torch.testing.assert_close(dp, tr.flat.grad, rtol=1e-4, atol=1e-7)
    assert dp.abs().sum() > 0


def test_record_loader_sharding():
    from rag_tl_domainllm_optimizer_amd.data import RecordLoader

    recs = [{"query": str(i), "retrieved_docs": [], "ground_truth": None} for i in range(10)]
    seen = []
    for r in range(3):
        L = RecordLoader(recs, 2, seed=1, rank=r, world=3)
        seen.append([q for b in L for q in b["query"]])
    flat = sum(seen, [])
    assert set(flat) == {str(i) for i in range(10)}
    assert len(seen[0]) == len(seen[1]) == len(seen[2])


def _mixed_worker(rank, world, port, out_dir, bucket_bytes):
    os.environ.update(RANK=str(rank), WORLD_SIZE=str(world), LOCAL_RANK=str(rank), MASTER_ADDR="127.0.0.1",
                      MASTER_PORT=str(port))
    from rag_tl_domainllm_optimizer_amd import ops, parallel
    from rag_tl_domainllm_optimizer_amd.parallel import GradSync

    parallel.init(device="cpu")
    ps = [torch.nn.Parameter(torch.zeros(40, dtype=torch.bfloat16)),
          torch.nn.Parameter(torch.zeros(24, dtype=torch.bfloat16)), torch.nn.Parameter(torch.zeros(7))]
    flat = ops.MixedFlatParams(ps)
    sync = GradSync(flat, bucket_bytes=bucket_bytes)
    flat.zero_grad()
    sync.start()
    c = float(rank + 1)
    sum(((p.float() * (i + 1) * c).sum() for i, p in enumerate(ps))).backward()
    sync.finish()
    torch.save({"g16": flat.grad16.clone(), "g32": flat.grad32.clone(), "buckets": len(sync.buckets)},
               os.path.join(out_dir, f"mixed{rank}.pt"))
    parallel.barrier()
    parallel.shutdown()


@pytest.mark.parametrize("bucket_bytes", [64, 64 << 20])
def test_dp_mixed_precision_grads(tmp_path, bucket_bytes):
    """Full-parameter training buffers (bf16 weights + fp32 value head): buckets per buffer, one
    bucket across the bf16 / fp32 seam, averaged over ranks."""
    world = 2
    mp.start_processes(_mixed_worker, args=(world, _free_port(), str(tmp_path), bucket_bytes), nprocs=world,
                       start_method="spawn", join=True)
    mean_c = sum(r + 1 for r in range(world)) / world
    for r in range(world):
        d = torch.load(tmp_path / f"mixed{r}.pt")
        g16, g32 = d["g16"].float(), d["g32"]
        assert torch.equal(g16[:40], torch.full((40,), mean_c))
        assert torch.equal(g16[48:72], torch.full((24,), 2 * mean_c))
        assert torch.equal(g32[:7], torch.full((7,), 3 * mean_c))
        assert d["buckets"] == (3 if bucket_bytes == 64 else 1)


def _bf16_worker(rank, world, port, out_dir, mode):
    os.environ.update(RANK=str(rank), WORLD_SIZE=str(world), LOCAL_RANK=str(rank), MASTER_ADDR="127.0.0.1",
                      MASTER_PORT=str(port))
    from rag_tl_domainllm_optimizer_amd import ops, parallel
    from rag_tl_domainllm_optimizer_amd.parallel import GradSync

    parallel.init(device="cpu")
    g = torch.Generator().manual_seed(100 + rank)
    n = 4099  # not a multiple of the world: the padded reduce-scatter tail
    ps = [torch.nn.Parameter(torch.zeros(n, dtype=torch.bfloat16)), torch.nn.Parameter(torch.zeros(5))]
    flat = ops.MixedFlatParams(ps)
    sync = GradSync(flat, bucket_bytes=1 << 12, bf16_reduce=mode)
    flat.zero_grad()
    sync.start()
    local = (torch.randn(n, generator=g) * torch.exp(torch.randn(n, generator=g))).to(torch.bfloat16)
    (ps[0].float() * local.float()).sum().backward()
    sync.finish()
    torch.save({"g": flat.grad16[:n].clone(), "local": local, "bytes": sync.comm_bytes},
               os.path.join(out_dir, f"bf{rank}.pt"))
    parallel.barrier()
    parallel.shutdown()


def test_dp_bf16_grads_reduced_in_fp32_world8(tmp_path):
    """Full fine-tuning at world 8: bf16 gradients are reduce-scattered in fp32 and rounded ONCE
    (rs32), so the averaged gradient is within one bf16 rounding of the exact mean on every rank —
    unlike a ring that sums in bf16 (simulated here), which loses ~3 bits at world 8."""
    world = 8
    mp.start_processes(_bf16_worker, args=(world, _free_port(), str(tmp_path), "rs32"), nprocs=world,
                       start_method="spawn", join=True)
    outs = [torch.load(tmp_path / f"bf{r}.pt") for r in range(world)]
    exact = sum(o["local"].double() for o in outs) / world
    got = outs[0]["g"].double()
    for o in outs[1:]:
        assert torch.equal(o["g"], outs[0]["g"])  # identical on every rank
    scale = exact.abs().clamp(min=1e-30)
    rel = ((got - exact).abs() / scale)
    assert float(rel.max()) <= 2.0 ** -8 + 1e-12
    # a bf16 ring: the running sum is rounded to bf16 at every hop
    ring = outs[0]["local"].clone()
    for o in outs[1:]:
        ring = (ring.float() + o["local"].float()).to(torch.bfloat16)
    ring_rel = ((ring.double() / world - exact).abs() / scale)
    assert float(rel.mean()) < 0.5 * float(ring_rel.mean())
    # link payload: fp32 reduce-scatter (4 B) + bf16 all-gather (2 B) per weight (+ fp32 value head)
    assert outs[0]["bytes"] >= 6 * 4099


def test_sft_fit_reports_each_steps_grad_norm():
    """fit() queues up to log_every steps before one D2H copy; every queued step must report ITS
    gradient norm (a snapshot), equal to a run that syncs after every step."""
    from rag_tl_domainllm_optimizer_amd import models
    from rag_tl_domainllm_optimizer_amd.models.config import PRESETS
    from rag_tl_domainllm_optimizer_amd.tokenizer import Tokenizer
    from rag_tl_domainllm_optimizer_amd.train.sft import SFTConfig, SFTTrainer

    cfg = PRESETS["tiny-llama"]
    tok = Tokenizer.synthetic(cfg.vocab_size, "llama")
    ex = _examples(tok, 16)

    def trainer():
        m = models.CausalLM(cfg, dtype=torch.float32, seed=1)
        return SFTTrainer(m, tok, SFTConfig(lr=3e-2, lora_r=4, lr_schedule="constant", warmup_steps=0, batch_size=2,
                                            seed=3))

    a = trainer()
    queued = a.fit(ex, epochs=1, shuffle=False, log_every=4)
    b = trainer()
    synced = [b.step(ex[k * 2:(k + 1) * 2]) for k in range(8)]
    na = [m["grad_norm"] for m in queued]
    nb = [m["grad_norm"] for m in synced]
    assert len(na) == 8
    assert len(set(round(x, 6) for x in na)) > 1  # not one repeated value
    torch.testing.assert_close(torch.tensor(na), torch.tensor(nb), rtol=1e-5, atol=1e-7)


def _broadcast_worker(rank, world, port):
    os.environ.update(RANK=str(rank), WORLD_SIZE=str(world), LOCAL_RANK=str(rank), MASTER_ADDR="127.0.0.1",
                      MASTER_PORT=str(port))
    from rag_tl_domainllm_optimizer_amd import parallel
    from rag_tl_domainllm_optimizer_amd.parallel.dist import broadcast_module_

    parallel.init(device="cpu")
    m = torch.nn.Linear(4, 3)
    with torch.no_grad():
        m.weight.fill_(rank + 1.0)
    before = [p._version for p in m.parameters()]
    broadcast_module_(m, 1)
    assert bool((m.weight == 2).all())
    assert all(p._version > v for p, v in zip(m.parameters(), before))
    parallel.shutdown()


def test_broadcast_counts_as_a_change():
    """Derived decode weights are kept by the parameters' version counters: a broadcast advances them."""
    mp.spawn(_broadcast_worker, args=(2, _free_port()), nprocs=2, join=True)
