"""Forms of kernels that a dispatch rule picks by size, at the edges of their ranges, against the oracle or the
general form of the same operation."""
import math

import numpy as np
import pytest
import torch

from rag_tl_domainllm_optimizer_amd import ops
from rag_tl_domainllm_optimizer_amd.generation.ragged import RaggedBatch
from rag_tl_domainllm_optimizer_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _close(a, b, rtol=2e-2, atol=2e-2):
    torch.testing.assert_close(a.float(), b.float(), rtol=rtol, atol=atol)


# ---------------------------------------------------------------------------------------------- sampler
@pytest.mark.parametrize("V,top_k,top_p", [(32000, 50, 1.0), (32000, 256, 0.9), (32000, 1, 1.0), (128, 50, 0.7),
                                           (4, 4, 0.5), (40004, 7, 0.95), (70000, 200, 1.0), (4096, 256, 1.0)])
def test_sampler_f32_topk_equals_general_form(V, top_k, top_p):
    """fp32 logits: the one-pass form (rows of 16-byte multiples) draws what the general one does from the same
    values at an odd row stride; rows with ties at the threshold, a plateau that overflows its candidate list, -inf
    entries, and inactive rows included."""
    B = 9
    g = torch.Generator(device=DEV).manual_seed(V + top_k)
    x = torch.randn(B, V, generator=g, device=DEV) * 3
    x[1] = 0.25                                            # one plateau: every token is a candidate
    x[2, ::2] = float("-inf")
    x[3, : min(V, 3 * top_k)] = x[3].max() + 1             # ties at the threshold
    x[4] *= 1e-3
    x[5] = torch.arange(V, device=DEV).float()             # the largest ones in a few threads' hands
    wide = torch.empty(B, V + 1, device=DEV)
    wide[:, :V] = x
    act = torch.ones(B, dtype=torch.uint8, device=DEV)
    act[6] = 0
    same = 0
    for o in range(4):
        off = torch.full((1,), o, dtype=torch.long, device=DEV)
        t1, l1 = ops.sample(x, 1 / 0.7, top_k=top_k, top_p=top_p, seed=3, offset=off, active=act)
        t0, l0 = ops.sample(wide[:, :V], 1 / 0.7, top_k=top_k, top_p=top_p, seed=3, offset=off, active=act)
        if top_p == 1.0:
            assert torch.equal(t1, t0)
        same += int((t1 == t0).sum())
        # the normaliser is a sum of V terms in another order: V * 2^-24 of it at most, in practice far less
        hit = t1 == t0
        torch.testing.assert_close(l1[hit], l0[hit], rtol=1e-5, atol=1e-4)
    # a nucleus cut within rounding of top_p may take one token more or less
    assert same >= 4 * B - 2


def test_sampler_f32_nan_logits_keep_general_draw():
    """A NaN among the logits leaves no nucleus mass to compare with: every top-k token stays in the draw, as in the
    general form. NaNs count as the largest logits on both sides; infinities of both signs beside them."""
    V, B = 4096, 8
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn(B, V, generator=g, device=DEV) * 3
    x[0, 17] = float("nan")
    x[1, ::5] = float("nan")
    x[2, 3], x[2, 9] = float("nan"), float("inf")
    x[3, 100:] = float("-inf")
    x[4] = float("-inf")
    x[5, 7] = float("inf")
    wide = torch.empty(B, V + 1, device=DEV)
    wide[:, :V] = x
    for top_p in (1.0, 0.9):
        drawn = set()
        for o in range(8):
            off = torch.full((1,), o, dtype=torch.long, device=DEV)
            t1, l1 = ops.sample(x, 1 / 0.7, top_k=40, top_p=top_p, seed=3, offset=off)
            t0, l0 = ops.sample(wide[:, :V], 1 / 0.7, top_k=40, top_p=top_p, seed=3, offset=off)
            assert torch.equal(t1, t0), (top_p, o, t1, t0)
            assert torch.equal(l1.isnan(), l0.isnan())
            drawn.add(int(t1[0]))
        assert len(drawn) > 1


@pytest.mark.parametrize("V,top_k,top_p", [(32000, 256, 1.0), (32000, 200, 0.9), (32000, 50, 1.0), (512, 64, 1.0), (8, 8, 1.0),
                                           (4096, 1024, 0.8), (40000, 500, 1.0)])
def test_sampler_bf16_bound_from_thread_maxima(V, top_k, top_p):
    """bf16 rows whose window fits badly (narrow, wide, plateaus, -inf) draw what the full-row search draws."""
    B = 8
    g = torch.Generator(device=DEV).manual_seed(V + top_k)
    x = torch.randn(B, V, generator=g, device=DEV) * torch.tensor([0.01, 0.3, 1, 4, 30, 1, 1, 1], device=DEV)[:, None]
    x[5] = 0.25
    x[6, ::2] = float("-inf")
    x[7] = torch.arange(V, device=DEV) / V
    x = x.bfloat16()
    for o in range(3):
        off = torch.full((1,), o, dtype=torch.long, device=DEV)
        got = []
        for window in (1, 0):
            with ops.tuning(sample_window=window):
                got.append(ops.sample(x, 1 / 0.7, top_k=top_k, top_p=top_p, seed=3, offset=off))
        assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


# ---------------------------------------------------------------------------------------------- decode attention
@pytest.mark.parametrize("B,Hq,Hkv,Smax,window", [(33, 32, 8, 300, 0), (64, 32, 8, 1100, 200), (65, 32, 8, 1023, 0),
                                                  (65, 32, 8, 1024, 0), (70, 64, 8, 1030, 0), (130, 4, 4, 70, 0),
                                                  (14, 40, 40, 1200, 0), (257, 8, 2, 33, 0)])
def test_decode_attention_waves_per_pair(B, Hq, Hkv, Smax, window):
    """One and four waves per (row, kv head) at the lines between them; rows from one key to the whole cache."""
    D = 128
    g = torch.Generator(device=DEV).manual_seed(B + Smax)
    kc = torch.randn(B, Hkv, Smax, D, generator=g, device=DEV).to(torch.bfloat16)
    vc = torch.randn(B, Hkv, Smax, D, generator=g, device=DEV).to(torch.bfloat16)
    slot = torch.randint(0, Smax, (B,), generator=g, device=DEV, dtype=torch.int32)
    slot[:5] = torch.tensor([0, Smax - 1, 15, 16, 17], device=DEV)
    start = torch.minimum(torch.randint(0, 20, (B,), generator=g, device=DEV, dtype=torch.int32), slot)
    tail = torch.arange(Smax, device=DEV)[None, None, :, None] >= slot.long()[:, None, None, None]
    kc.masked_fill_(tail, float("nan"))
    vc.masked_fill_(tail, float("nan"))
    cos, sin = ref.rope_tables(D, 4096, 10000.0, DEV)
    pos = slot - start
    qkv = torch.randn(B, (Hq + 2 * Hkv) * D, generator=g, device=DEV).to(torch.bfloat16)
    k2, v2 = kc.clone(), vc.clone()
    out = ops.decode_step_attention(qkv, kc, vc, slot, slot + 1, Hq, pos, cos, sin, start, window)
    q = ops.rope_qkv_(qkv.clone(), pos, cos, sin, Hq, Hkv, D, S=1, k_cache=k2, v_cache=v2, slot_base=slot)
    _close(out, ref.decode_attention(q, k2, v2, slot + 1, Hq, start, window, 1.0 / math.sqrt(D)))
    assert torch.equal(kc.nan_to_num(), k2.nan_to_num()) and torch.equal(vc.nan_to_num(), v2.nan_to_num())


@pytest.mark.parametrize("B,Hkv,G,W", [(70, 8, 4, 1), (70, 16, 16, 1), (34, 8, 4, 4), (34, 8, 8, 4), (34, 8, 1, 4), (32, 4, 4, 8), (32, 2, 2, 8)])
def test_decode_attention_of_one_to_seven_tiles_a_wave(B, Hkv, G, W):
    """Rows that end in each of a wave's first seven tiles of 16 keys and around their edges, waves of no tile, of one, of three and
    of a refilled fourth among them, with keys that begin anywhere; slots behind the new token hold NaN."""
    D, Smax, scale = 128, 16 * 7 * W + 8 * W, 128 ** -0.5
    g = torch.Generator(device=DEV).manual_seed(B * W + G)
    ends = [max(1, 16 * W * j + e) for j in range(8) for e in (-1, 0, 1, 8 * W)]
    n = torch.tensor((ends * 3)[:B], dtype=torch.int32, device=DEV)
    start = torch.minimum(torch.randint(0, 9, (B,), generator=g, device=DEV, dtype=torch.int32), n - 1)
    kc, vc = torch.randn(2, B, Hkv, Smax, D, generator=g, device=DEV).bfloat16()
    tail = torch.arange(Smax, device=DEV)[None, None, :, None] >= (n - 1).long()[:, None, None, None]
    kc.masked_fill_(tail, float("nan"))
    vc.masked_fill_(tail, float("nan"))
    qkv = torch.randn(B, (G + 2) * Hkv * D, generator=g, device=DEV).bfloat16()
    out = ops.decode_step_attention(qkv, kc, vc, n - 1, n, G * Hkv, kv_start=start).view(B, Hkv, G, D).double()
    for b in range(B):
        lo, hi = int(start[b]), int(n[b])
        k, v = kc[b, :, lo:hi].double(), vc[b, :, lo:hi].double()
        assert torch.equal(k[:, -1].flatten(), qkv[b, G * Hkv * D:(G + 1) * Hkv * D].double())
        p = torch.softmax((qkv[b, :G * Hkv * D].view(Hkv, G, 1, D).double() * k[:, None]).sum(-1) * scale, -1)[..., None]
        want, size = ((p * x[:, None]).sum(2) for x in (v, v.abs()))
        # p and the result round to bf16 (half an ulp: 2^-8 each)
        assert ((out[b] - want).abs() - (2.0 ** -7 + 2.0 ** -11) * size).max() < 1e-6, (b, lo, hi)


@pytest.mark.parametrize("B,Hkv,G", [(13, 40, 1), (33, 16, 2), (65, 8, 4), (65, 8, 8)])
def test_decode_attention_form_whatever_the_free_slots(B, Hkv, G):
    """Beyond 512 (row, kv head) pairs short rows cost no more in a cache of many slots: the same form, so the same bits."""
    D, n = 128, 70
    g = torch.Generator(device=DEV).manual_seed(B)
    kv = torch.randn(2, B, Hkv, n, D, generator=g, device=DEV).to(torch.bfloat16)
    qkv = torch.randn(B, (G + 2) * Hkv * D, generator=g, device=DEV).to(torch.bfloat16)
    slot = torch.randint(0, n, (B,), generator=g, device=DEV, dtype=torch.int32)
    outs = []
    for Smax in (n, 1023, 1024, 2048):
        kc, vc = torch.zeros(2, B, Hkv, Smax, D, dtype=torch.bfloat16, device=DEV)
        kc[:, :, :n], vc[:, :, :n] = kv[0], kv[1]
        outs.append(ops.decode_step_attention(qkv, kc, vc, slot, slot + 1, G * Hkv))
    assert all(torch.equal(o, outs[0]) for o in outs[1:])


# ---------------------------------------------------------------------------------------------- retrieval
@pytest.mark.parametrize("nq,N,k", [(1, 40, 40), (3, 512, 16), (2, 1024, 32), (2, 1025, 32), (2, 700, 33), (5, 4097, 128),
                                    (2, 4096, 128), (2, 300, 129), (4, 9600, 3), (1, 100003, 512), (2, 70, 100), (300, 64, 1)])
def test_topk_forms(nq, N, k):
    """Every thread count of the selection, rows that are strided, tied, flat, or short of finite scores, with ids mapped:
    the order of a stable sort."""
    g = torch.Generator(device=DEV).manual_seed(N + k)
    s = torch.randn(nq, N + 3, generator=g, device=DEV)[:, :N]
    if nq > 1:
        s[0] = torch.randint(0, 5, (N,), generator=g, device=DEV).float()  # ties
        s[1, N // 4:] = float("-inf")
    if nq > 3:
        s[2] = 0.5                                                         # a plateau
        s[3] = torch.arange(N, device=DEV).float() / N
    cid = torch.randint(0, 1 << 40, (nq, N), generator=g, device=DEV)
    v, i = ops.topk(s, k, cid, finite=True)
    vs, order = torch.sort(s, dim=-1, descending=True, stable=True)
    n = min(k, N)
    fits = torch.tensor([int((s[r] >= vs[r, n - 1]).sum()) <= 1024 for r in range(nq)])  # ties within the candidate list
    assert torch.equal(v[:, :n], vs[:, :n])
    want = torch.where(torch.isfinite(vs), cid.gather(1, order), torch.full_like(cid, -1))[:, :n]
    ok = fits.to(DEV)[:, None] | (v[:, :n] > vs[:, n - 1:n])
    assert torch.equal(torch.where(ok, i[:, :n], 0), torch.where(ok, want, 0))
    if k > N:
        assert bool((v[:, n:] == float("-inf")).all()) and bool((i[:, n:] == -1).all())


@pytest.mark.parametrize("N,k", [(8, 3), (512, 32), (513, 32), (2048, 33), (2049, 20), (8192, 31), (8193, 7)])
def test_topk_candidates_around_a_wave(N, k):
    """Rows of at most eight elements a thread and just longer ones, with a wave's worth of candidates and one more or less at
    the k-th score: the order of a stable sort."""
    g = torch.Generator(device=DEV).manual_seed(N + k)
    s = torch.rand(8, N, generator=g, device=DEV) - 2
    for r, ties in enumerate((1, 3, 62, 63, 64, 65, 66)):
        at = torch.randperm(N, generator=g, device=DEV)[:ties]
        s[r, at] = 0.0
        s[r, at[0]] = 1.0
    cid = torch.randint(0, 1 << 40, s.shape, generator=g, device=DEV)
    vs, order = torch.sort(s, dim=-1, descending=True, stable=True)
    v, i = ops.topk(s, k, cid)
    assert torch.equal(v, vs[:, :k]) and torch.equal(i, cid.gather(1, order)[:, :k])


@pytest.mark.parametrize("N,k", [(1500, 3), (5000, 3), (5000, 128), (9600, 40), (100003, 512)])
def test_topk_rows_with_more_ties_than_candidates(N, k):
    """Rows whose k-th score is shared by more entries than the candidate list holds: all larger scores come first, then the
    ties of the lowest indices; the same for fewer than k finite scores. The order of a stable sort, each time."""
    g = torch.Generator(device=DEV).manual_seed(N + k)
    s = torch.full((7, N), 0.5, device=DEV)
    s[0, -1] = 1.0
    s[1, torch.randperm(N, generator=g, device=DEV)[:k - 1]] = 0.75 + torch.rand(k - 1, generator=g, device=DEV)
    s[2] = float("-inf")
    s[2, N - k // 2 - 1:] = torch.randn(k // 2 + 1, generator=g, device=DEV)
    s[3] = torch.where(torch.rand(N, generator=g, device=DEV) < 0.5, 0.5, 0.25)
    s[3, N // 2] = 2.0
    s[4] = float("-inf")
    s[5] = torch.where(torch.rand(N, generator=g, device=DEV) < 0.9, 0.0, -1.0)
    s[5, -1] = 1e-30
    cid = torch.randint(0, 1 << 40, s.shape, generator=g, device=DEV)
    vs, order = torch.sort(s, dim=-1, descending=True, stable=True)
    want = torch.where(torch.isfinite(vs), cid.gather(1, order), torch.full_like(cid, -1))[:, :k]
    for _ in range(3):
        v, i = ops.topk(s, k, cid, finite=True)
        assert torch.equal(v, vs[:, :k])
        assert torch.equal(i, want)


def test_ivf_search_with_fewer_documents_than_asked():
    """Fewer than k documents in the probed lists, whose slots are more than the candidate list holds: all are found."""
    from rag_tl_domainllm_optimizer_amd.retrieval.index import IVFIndex

    g = torch.Generator().manual_seed(0)
    x = torch.randn(1500, 64, generator=g)
    x[:1400] = x[0] + 0.01 * torch.randn(1400, 64, generator=g)  # one list holds most documents
    x = torch.nn.functional.normalize(x, dim=-1)
    ix = IVFIndex(64, nlist=24, device=DEV)
    ix.train(x, niter=4)
    ix.add(x)
    q = x[1400:].to(DEV)
    for nprobe in (2, 4, 24):
        held = ix.lsize[ix._coarse(q, nprobe).long()].sum(1).clamp(max=500).tolist()
        _, ids = ix.search(q, 500, nprobe=nprobe)
        found = [len(row[row >= 0].unique()) for row in ids]
        assert found == held, nprobe


@pytest.mark.parametrize("d", [8, 72, 384, 1000])
@pytest.mark.parametrize("l2", [False, True])
def test_ivf_scan_lists(d, l2):
    """Lists of 0 to 200 vectors (pieces of 64), an unused probe, odd widths: against the products in float64."""
    g = torch.Generator(device=DEV).manual_seed(d)
    size = torch.tensor([0, 1, 63, 64, 65, 200], dtype=torch.int32, device=DEV)
    start = torch.tensor([0, 0, 5, 70, 140, 210], dtype=torch.int32, device=DEV)
    vecs = torch.randn(410, d, generator=g, device=DEV).to(torch.bfloat16)
    q = torch.randn(3, d, generator=g, device=DEV).to(torch.bfloat16)
    probes = torch.tensor([[0, 1, 2], [3, 4, 5], [-1, 5, 0]], dtype=torch.int32, device=DEV)
    sq, ids, maxlen = vecs.float().pow(2).sum(-1), torch.arange(410, device=DEV) + 7, 200
    cand, cid = ops.ivf_scan(q, probes, start, size, vecs, ids, maxlen, sq, l2)
    full = q.double() @ vecs.double().t()
    if l2:
        full = 2 * full - sq.double() - q.double().pow(2).sum(-1, keepdim=True)
    want = torch.full((3, 3, maxlen), float("-inf"), dtype=torch.float64, device=DEV)
    wid = torch.full((3, 3, maxlen), -1, device=DEV)
    for i in range(3):
        for p in range(3):
            L = int(probes[i, p])
            n = int(size[L]) if L >= 0 else 0
            if n:
                b = int(start[L])
                want[i, p, :n], wid[i, p, :n] = full[i, b:b + n], ids[b:b + n]
    assert torch.equal(cid, wid.view(3, -1))
    # d fp32 additions of terms of size 1: d * 2^-24 * sqrt(d) at the very most
    torch.testing.assert_close(cand.double(), want.view(3, -1), rtol=1e-5, atol=d ** 1.5 * 2 ** -24 + 1e-6)


@pytest.mark.parametrize("d", [8, 384, 392, 800])
@pytest.mark.parametrize("l2", [False, True])
@pytest.mark.parametrize("nq,nlist", [(1, 9), (3, 40), (17, 6), (700, 6)])
def test_ivf_scan_by_list_and_by_probe(d, l2, nq, nlist):
    """A workgroup per list or per probe, queries around the tiles of 16, more than 4096 probes, an unaligned first query."""
    g = torch.Generator(device=DEV).manual_seed(d + nq)
    size = torch.zeros(nlist, dtype=torch.int32, device=DEV)
    size[:6] = torch.tensor([0, 1, 15, 16, 17, 150], dtype=torch.int32, device=DEV)
    start = torch.cumsum(size, 0).int() - size
    vecs = torch.randn(int(size.sum()), d, generator=g, device=DEV).to(torch.bfloat16)
    q = torch.randn(nq * d + 1, generator=g, device=DEV).to(torch.bfloat16)[1:].view(nq, d)
    nprobe = 6
    probes = torch.stack([torch.randperm(6, generator=g, device=DEV) for _ in range(nq)]).int()
    probes[nq // 2, 2] = -1
    sq, ids, maxlen = vecs.float().pow(2).sum(-1), torch.arange(len(vecs), device=DEV) + 7, 151
    cand, cid = ops.ivf_scan(q, probes, start, size, vecs, ids, maxlen, sq, l2)
    full = q.double() @ vecs.double().t()
    if l2:
        full = 2 * full - sq.double() - q.double().pow(2).sum(-1, keepdim=True)
    j = torch.arange(maxlen, device=DEV)
    L = probes.long().clamp(min=0)
    ok = (j < size[L][..., None]) & (probes >= 0)[..., None]
    at = (start[L][..., None] + j).clamp(max=len(vecs) - 1)
    want = full.gather(1, at.view(nq, -1)).view(nq, nprobe, maxlen).masked_fill(~ok, float("-inf"))
    assert torch.equal(cid, ids[at].masked_fill(~ok, -1).view(nq, -1))
    torch.testing.assert_close(cand.double(), want.view(nq, -1), rtol=1e-5, atol=d ** 1.5 * 2 ** -24 + 1e-6)


@pytest.mark.parametrize("nq,d", [(3, 384), (2000, 384), (3, 72)])
def test_ivf_scan_of_vectors_off_16_bytes(nq, d):
    """Vectors that begin at any element: one list of them, for few queries and as many as would go by list."""
    g = torch.Generator(device=DEV).manual_seed(nq)
    n = 300
    vecs = torch.randn(n * d + 1, generator=g, device=DEV).to(torch.bfloat16)[1:].view(n, d)
    q = torch.randn(nq, d, generator=g, device=DEV).to(torch.bfloat16)
    size, start = torch.tensor([n], dtype=torch.int32, device=DEV), torch.tensor([0], dtype=torch.int32, device=DEV)
    ids = torch.arange(n, device=DEV)
    cand, cid = ops.ivf_scan(q, torch.zeros(nq, 1, dtype=torch.int32, device=DEV), start, size, vecs, ids, n)
    torch.testing.assert_close(cand.double(), q.double() @ vecs.double().t(), rtol=1e-5, atol=d ** 1.5 * 2 ** -24 + 1e-6)
    assert torch.equal(cid, ids.expand(nq, n))


@pytest.mark.parametrize("d", [264, 352])
def test_ivf_scan_width_between_fragments(d):
    """Widths of the form that multiplies by probe, with a last fragment that is not whole."""
    for l2 in (False, True):
        test_ivf_scan_lists(d, l2)
        test_ivf_scan_by_list_and_by_probe(d, l2, 3, 40)


@pytest.mark.parametrize("nq,nlist,nprobe,d,most", [(5000, 2, 2, 384, 70), (4500, 1, 1, 1000, 130), (900, 9, 4, 768, 65), (64, 3, 3, 72, 9000)])
@pytest.mark.parametrize("l2", [False, True])
def test_ivf_scan_by_list_rounds(nq, nlist, nprobe, d, most, l2):
    """By list: more queries of a list than a workgroup holds, vectors in one to three parts, lists of several workgroups that go round,
    probes of no list."""
    g = torch.Generator(device=DEV).manual_seed(nq)
    size = torch.randint(0, most + 1, (nlist,), generator=g, device=DEV, dtype=torch.int32)
    size[0] = most
    start = torch.cumsum(size, 0).int() - size
    vecs = torch.randn(int(size.sum()), d, generator=g, device=DEV).to(torch.bfloat16)
    q = torch.randn(nq, d, generator=g, device=DEV).to(torch.bfloat16)
    probes = torch.rand(nq, nlist, generator=g, device=DEV).topk(nprobe)[1].int()
    probes[nq // 2, 0], probes[nq // 3, 0] = -1, nlist
    sq, ids, maxlen = vecs.float().pow(2).sum(-1), torch.arange(len(vecs), device=DEV) + 7, most + 1
    assert ops.native().ivf_by_list(nq, nprobe, nlist, d, maxlen, len(vecs))
    cand, cid = ops.ivf_scan(q, probes, start, size, vecs, ids, maxlen, sq, l2)
    full = q.double() @ vecs.double().t()
    if l2:
        full = 2 * full - sq.double() - q.double().pow(2).sum(-1, keepdim=True)
    j = torch.arange(maxlen, device=DEV)
    L = probes.long().clamp(0, nlist - 1)
    ok = (j < size[L][..., None]) & ((probes >= 0) & (probes < nlist))[..., None]
    at = (start[L][..., None] + j).clamp(max=len(vecs) - 1)
    want = full.gather(1, at.view(nq, -1)).view(nq, nprobe, maxlen).masked_fill(~ok, float("-inf"))
    assert torch.equal(cid, ids[at].masked_fill(~ok, -1).view(nq, -1))
    torch.testing.assert_close(cand.double(), want.view(nq, -1), rtol=1e-5, atol=d ** 1.5 * 2 ** -24 + 1e-6)


def test_ivf_scan_of_a_list_longer_than_a_grid():
    """A list of more 64-vector pieces than a grid's third dimension holds, and a short one beside it."""
    d, n = 8, 65535 * 64 + 1000
    g = torch.Generator(device=DEV).manual_seed(0)
    vecs = torch.randn(n + 70, d, generator=g, device=DEV).to(torch.bfloat16)
    size = torch.tensor([n, 70], dtype=torch.int32, device=DEV)
    start = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    q = torch.randn(1, d, generator=g, device=DEV).to(torch.bfloat16)
    ids = torch.arange(n + 70, device=DEV) + 7
    maxlen = n + 30
    cand, cid = ops.ivf_scan(q, torch.tensor([[1, 0]], dtype=torch.int32, device=DEV), start, size, vecs, ids, maxlen)
    want = torch.full((1, 2, maxlen), float("-inf"), dtype=torch.float64, device=DEV)
    wid = torch.full((1, 2, maxlen), -1, device=DEV)
    full = (vecs.double() @ q[0].double())
    want[0, 0, :70], want[0, 1, :n] = full[n:], full[:n]
    wid[0, 0, :70], wid[0, 1, :n] = ids[n:], ids[:n]
    assert torch.equal(cid.view(1, 2, maxlen), wid)
    torch.testing.assert_close(cand.view(1, 2, maxlen).double(), want, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("B,S,H", [(3, 1, 8), (2, 17, 384), (4, 70, 768), (2, 9, 20), (1, 33, 2056)])
def test_pool_normalize_forms(B, S, H):
    g = torch.Generator(device=DEV).manual_seed(S)
    x = torch.randn(B, S, H, generator=g, device=DEV).to(torch.bfloat16)
    lens = torch.randint(1, S + 1, (B,), generator=g, device=DEV, dtype=torch.int32)
    lens[0] = S
    for n in (True, False):
        torch.testing.assert_close(ops.pool_normalize(x, lens, n).double(), ref.pool_norm(x.double(), lens, n).double(),
                                   rtol=1e-5, atol=1e-6)


# ---------------------------------------------------------------------------------------------- decode products, 17..64 rows
@pytest.mark.parametrize("N,K,act", [(16, 64, 0), (80, 192, 0), (2048, 512, 0), (4096, 2048, 0), (4112, 1024, 0),
                                     (6160, 2112, 0), (4096, 4160, ops.ACT_RELU2), (64, 128, 5), (192, 2048, 5), (4224, 4096, 5)])
def test_image_products_17_to_64_rows(N, K, act):
    """Tile-ordered products at 17..64 rows on the rule's own route and at forced splits: odd numbers of row groups and
    chunks, the in-product norm, bias, activation, residual, fp32 results and strided results. bf16 products are exact in
    fp32, so fp32 results differ from 64 bits by the sum's order alone: K 2^-24 of sum |x w| bounds it."""
    C = ops.native()
    g = torch.Generator(device=DEV).manual_seed(N + K)
    w = (torch.randn(N, K, generator=g, device=DEV) / K ** 0.5).bfloat16()
    img = C.shuffle_decode_weight(w)
    bias = torch.randn(N, generator=g, device=DEV).bfloat16()
    No = N // 2 if act == ops.ACT_SWIGLU else N

    def epi(y, r):
        if act == ops.ACT_SWIGLU:
            return torch.nn.functional.silu(y[:, :No]) * y[:, No:]
        y = ref.apply_act(y, act)
        return y if r is None else y + r.double()

    for M in (17, 32, 33, 48, 64):
        x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
        r = torch.randn(M, No, generator=g, device=DEV).bfloat16() if act == 0 else None
        pre = x.double() @ w.double().t()
        rstd = torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + 1e-5)
        bound = (x.double().abs() @ w.double().abs().t()).max().item() * K * 2.0 ** -24 + 1e-6
        for split in (0, 1, 2, 3, 7, 8):
            with ops.tuning(decode_split=split):
                for _ in range(2):  # the second finds the tickets as the first left them
                    y = C.gemm(x, img, None, None, None, 0 if act == ops.ACT_RELU2 else act, True, None, None, 0.0, True)
                e = (y.double() - (epi(pre, None) if act == ops.ACT_SWIGLU else pre)).abs().max().item()
                assert e <= bound * (8 if act == ops.ACT_SWIGLU else 1), (M, split, e, bound)
                out = torch.full((M, No + 8), 7.0, dtype=torch.bfloat16, device=DEV)
                C.gemm(x, img, None, None, bias, act, False, out[:, :No], r, 1e-5, True)
                want = epi(pre * rstd + bias.double(), r)
                # a bf16 rounding of the result and, before a square or a product, the fp32 sum's error
                torch.testing.assert_close(out[:, :No].double(), want, rtol=2.0 ** -8 + 1e-3, atol=4 * bound + 1e-4)
                assert (out[:, No:] == 7).all()


@pytest.mark.parametrize("act", [0, ops.ACT_RELU2, 2, 4])
@pytest.mark.parametrize("N,K,split", [(2064, 2176, 0), (4176, 1088, 0), (4176, 1088, 5), (208, 6144, 8), (3104, 2048, 0), (5136, 1024, 0)])
def test_image_products_17_to_64_rows_epilogues(N, K, split, act):
    """Linear and squared-relu results, whose epilogue is their own, and the others', behind parts of K and without: residuals that come
    four at a time and ones that do not, with and without bias, a last column group that is not whole."""
    C = ops.native()
    g = torch.Generator(device=DEV).manual_seed(N + act)
    w = (torch.randn(N, K, generator=g, device=DEV) / K ** 0.5).bfloat16()
    img, bias = C.shuffle_decode_weight(w), torch.randn(N, generator=g, device=DEV).bfloat16()
    for M in (17, 33, 64):
        x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
        pre = x.double() @ w.double().t()
        bound = (x.double().abs() @ w.double().abs().t()).max().item() * K * 2.0 ** -24 + 1e-6
        for r, b in ((None, None), (torch.randn(M, N, generator=g, device=DEV).bfloat16(), bias),
                     (torch.randn(M, N + 3, generator=g, device=DEV).bfloat16()[:, :N], None)):
            with ops.tuning(decode_split=split):
                y = C.gemm(x, img, None, None, b, act, False, None, r, 0.0, True)
            z = pre if b is None else pre + b.double()
            want = ref.apply_act(z, act) + (0 if r is None else r.double())
            # a bf16 rounding of the result and, before a square, the fp32 sum's error
            torch.testing.assert_close(y.double(), want, rtol=2.0 ** -8 + 1e-4, atol=2 * bound * (1 + z.abs().max().item()) + 1e-5)


# ---------------------------------------------------------------------------------------------- GELU epilogue
@pytest.mark.parametrize("M,N,res", [(65, 256, False), (300, 264, True), (4096, 8, False)])
def test_gelu_epilogue_bits(M, N, res):
    """The tile epilogue's GELU has the bits of the split-K reduction's (erff throughout). A row's input is the sum of the
    three bf16 parts of an fp32 value, times a column's power of two: exact, so both see the same values, from denormal
    results through the negative tail, where the bf16 candidates disagree, to beyond the fitted range."""
    C = ops.native()
    g = torch.Generator(device=DEV).manual_seed(M)
    v = torch.randn(M, generator=g, device=DEV) * torch.where(torch.rand(M, generator=g, device=DEV) < 0.5, 1.0, 4.0)
    v[:8] = torch.tensor([-3.8, -5.2, 5.2, -9.0, 0.0, 1e-30, -2.125, 40.0], device=DEV)
    x = torch.zeros(M, 64, device=DEV, dtype=torch.bfloat16)
    rest = v.clone()
    for k in range(3):
        x[:, k] = rest.bfloat16()
        rest = rest - x[:, k].float()
    w = torch.zeros(N, 64, device=DEV, dtype=torch.bfloat16)
    w[:, :3] = (2.0 ** (torch.arange(N, device=DEV) % 5 - 3).float())[:, None].bfloat16()
    bias = torch.zeros(N, device=DEV, dtype=torch.bfloat16)
    r = torch.randn(M, N, generator=g, device=DEV).bfloat16() if res else None
    y = C.gemm_big(x, w, 0, 0, None, None, bias, 2, 0, 1, None, None, r)
    slabs = torch.empty(M * N, dtype=torch.float32, device=DEV)
    z = C.gemm_splitk(x, w, 1, slabs, bias, 2, None, r)
    assert torch.equal(y.view(torch.int16), z.view(torch.int16))


@pytest.mark.parametrize("M,N,K,act,res", [(1, 8, 64, 0, False), (255, 128, 128, 0, True), (256, 136, 192, 2, False),
                                           (257, 120, 256, 0, False), (513, 264, 64, 2, True), (1300, 1152, 384, 0, True)])
def test_two_workgroup_product_has_the_tile_kernels_bits(M, N, K, act, res):
    """The form with two workgroups per CU multiplies in the order of the 256 x 256 tiles: the same bits, with strided
    operands, around the tile edges and from one K-step on; nothing beyond the columns is written."""
    g = torch.Generator(device=DEV).manual_seed(M + K)

    def r(*s):
        return torch.randn(*s, generator=g, device=DEV).bfloat16()
    x, w, bias = r(M, K + 8)[:, :K], r(N, K + 16)[:, :K] * 0.1, r(N)
    R = r(M, N) if res else None
    out = []
    for duo in (0, 2):
        y = torch.full((M, N + 8), 7.0, dtype=torch.bfloat16, device=DEV)
        with ops.tuning(gemm_duo=duo):
            ops.native().gemm_big(x, w, 0, 0, None, None, bias, act, 0, 1, y[:, :N], None, R)
        assert (y[:, N:] == 7).all()
        out.append(y[:, :N])
    assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))
    want = x.double() @ w.double().t() + bias.double()
    if act:
        want = torch.nn.functional.gelu(want)
    # a bf16 rounding before the residual and one after, on an fp32 sum
    _close(out[1], want + (R.double() if res else 0), rtol=2.0 ** -7, atol=1e-3 * math.sqrt(K))


@pytest.mark.parametrize("form", [2, 3, 4])
@pytest.mark.parametrize("M,N,K,act,res", [(1, 8, 64, 0, False), (63, 64, 128, 2, True), (64, 72, 192, 0, True), (65, 128, 256, 2, False),
                                           (128, 136, 320, 0, False), (129, 120, 384, 2, True), (700, 384, 1536, 0, True),
                                           (1030, 1160, 448, 2, False)])
def test_smaller_tiles_have_the_tile_kernels_bits(form, M, N, K, act, res):
    """Tiles of 64 x 64 to 128 x 128 multiply in the order of the 256 x 256 ones: the same bits, with strided operands, around
    the tile edges, with fewer K-steps than the ring has places and more; nothing beyond the columns is written."""
    g = torch.Generator(device=DEV).manual_seed(M + K)

    def r(*s):
        return torch.randn(*s, generator=g, device=DEV).bfloat16()
    x, w, bias = r(M, K + 8)[:, :K], r(N, K + 16)[:, :K] * 0.1, r(N)
    R = r(M, N) if res else None
    out = []
    for mid in (0, form):
        y = torch.full((M, N + 8), 7.0, dtype=torch.bfloat16, device=DEV)
        with ops.tuning(gemm_duo=0, gemm_mid=mid):
            ops.native().gemm_big(x, w, 0, 0, None, None, bias, act, 0, 1, y[:, :N], None, R)
        assert (y[:, N:] == 7).all()
        out.append(y[:, :N])
    assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))


@pytest.mark.parametrize("M,N,K,act,s", [(65, 384, 384, 0, 1), (300, 384, 1536, 0, 3), (512, 768, 3072, 0, 6), (130, 272, 768, 2, 1),
                                         (500, 272, 1088, 2, 2), (90, 48, 2560, 0, 5), (700, 400, 768, 0, 1), (6000, 768, 1536, 0, 1),
                                         (22000, 768, 1536, 0, 1)])
def test_encoder_products_on_smaller_tiles_are_summed_as_before(M, N, K, act, s):
    """The parts of K in their order up to 512 rows, no parts beyond, whatever tiles the planner takes for a product with a
    bias, or for the rows behind its large tiles."""
    from rag_tl_domainllm_optimizer_amd.ops.linear import small_tiles, splitk_plan
    g = torch.Generator(device=DEV).manual_seed(M)

    def r(*s):
        return torch.randn(*s, generator=g, device=DEV).bfloat16()
    x, w, b = r(M, K), r(N, K) * 0.1, r(N)
    assert splitk_plan(M, N, K, act)[0] == s and small_tiles(M, N, K, act) == (M <= 512)
    got = ops.linear(x, w, b, act="gelu" if act else None)
    with ops.tuning(gemm_duo=0, gemm_mid=0):
        if s > 1:
            want = ops.native().gemm_splitk(x, w, s, torch.empty(s * M * N, device=DEV), b, act, None, None, 256)
        else:
            want = ops.native().gemm_big(x, w, 0, 0, None, None, b, act, 0, 1, None, None, None)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("at", [0, 1, 4])
@pytest.mark.parametrize("M,N,K", [(65, 384, 1536), (300, 272, 1088), (512, 768, 3072)])
def test_split_products_with_a_bias_write_rows_at_any_address(M, N, K, at):
    """Products of 65 to 512 rows with a bias and a split K: out and residual may begin at any element; with and without tiles that sum
    the parts the bits are those of the split product, in strided rows, and nothing beyond the columns is written."""
    from rag_tl_domainllm_optimizer_amd.ops.linear import splitk_plan
    g = torch.Generator(device=DEV).manual_seed(M)

    def r(*s):
        return torch.randn(*s, generator=g, device=DEV).bfloat16()
    x, w, b, R = r(M, K + 8)[:, :K], r(N, K + 16)[:, :K] * 0.1, r(N), r(M, N)
    s = splitk_plan(M, N, K)[0]
    assert s > 1
    want = ops.native().gemm_splitk(x, w, s, torch.empty(s * M * N, device=DEV), b, 0, None, R, 256)

    def rows(t):  # t in rows of N + 16 elements that begin at element `at`
        flat = torch.full((M * (N + 16) + 16,), 7.0, dtype=torch.bfloat16, device=DEV)[at:]
        y = flat[:M * (N + 16)].view(M, N + 16)
        y[:, :N] = t
        return y
    y = rows(torch.zeros_like(R))
    ops.gemm(x, w, bias=b, out=y[:, :N], residual=rows(R)[:, :N])
    assert torch.equal(y[:, :N].view(torch.int16), want.view(torch.int16)) and (y[:, N:] == 7).all()


# ---------------------------------------------------------------------------------------------- encoders without padding
@pytest.mark.parametrize("D,H,bias", [(32, 3, False), (64, 2, False), (64, 12, True), (128, 1, False), (32, 2, True)])
@pytest.mark.parametrize("lens", [[1], [64, 65, 0, 127], [128, 129, 63, 1, 300], [2] * 40])
def test_packed_attention_equals_padded(D, H, bias, lens):
    """Sequences one behind the other against the padded form, around the tile edges. Without a bias the arithmetic per
    row is the same, down to probabilities below 2^-126; the bias is added to the rounded or to the exact scaled score
    (one rounding of an exponent of at most 2^7: 2^-17 of a probability, below the results' bf16)."""
    g = torch.Generator(device=DEV).manual_seed(D + len(lens))
    B, S = len(lens), max(lens)
    n = torch.tensor(lens, device=DEV)
    qkv = torch.randn(B, S, 3 * H * D, generator=g, device=DEV).bfloat16()
    lut = torch.randn(H, 2 * S + 5, generator=g, device=DEV) if bias else None
    rb = S + 3 if bias else 0
    keep = torch.arange(S, device=DEV)[None, :] < n[:, None]
    flat = qkv[keep]
    off = torch.nn.functional.pad(n.cumsum(0), (1, 0))
    cut = lambda t: (t[:, :H * D], t[:, H * D:2 * H * D], t[:, 2 * H * D:])
    got = ops.attention_packed(*cut(flat), off, S, H, D, rel_bias_lut=lut, rb_L=rb)
    want = ops.attention(*cut(qkv.view(B * S, -1)), B, S, S, H, H, D, kv_len=n.int(), rel_bias_lut=lut, rb_L=rb)
    want = want.view(B, S, -1)[keep]
    if bias:
        _close(got, want, rtol=2.0 ** -7, atol=2.0 ** -8)
    else:
        assert torch.equal(got, want)
    x = torch.randn(B, S, 384, generator=g, device=DEV).bfloat16()
    assert torch.equal(ops.pool_normalize_packed(x[keep], off, S), ops.pool_normalize(x, n))


# ---------------------------------------------------------------------------------------------- encoders, few rows
@pytest.mark.parametrize("M,N,K,act,norm", [(1, 16, 64, 0, False), (15, 384, 384, 2, True), (16, 1536, 768, 2, True),
                                            (9, 80, 1600, 0, False), (16, 96, 3072, 2, False), (17, 48, 448, 0, True),
                                            (17, 256, 768, 0, True), (32, 80, 1024, 0, False), (32, 32, 1536, 2, False),
                                            (31, 1152, 576, 0, False), (32, 768, 3072, 0, False), (20, 16, 3072, 0, False)])
def test_few_rows(M, N, K, act, norm):
    """Products of few rows, the norm ahead among them: the bits of the kernels that ``ops.linear``
    takes, whose parts of K they sum: one part to sixteen, parts of uneven length and of none, around the row tiles, strided
    rows."""
    g = torch.Generator(device=DEV).manual_seed(M + K)

    def r(*s, m=1.0):
        return (torch.randn(*s, generator=g, device=DEV) * m).bfloat16()
    x, w, b = r(M, K + 8)[:, :K], r(N, K + 24, m=K ** -0.5)[:, :K], r(N)
    kw = {}
    if norm:
        kw = dict(res=r(M, K), lw=r(K), lb=r(K), eps=1e-5)
    y, xo = ops.native().few_rows(x, w, b, act, **kw)
    if norm:
        assert torch.equal(xo, ops.layer_norm(x.contiguous(), kw["lw"], kw["lb"], 1e-5, residual=kw["res"])[0])
    assert torch.equal(y, ops.linear(xo if norm else x, w, b, act="gelu" if act else None))


@pytest.mark.parametrize("preset", ["minilm-l6", "mpnet-base"])
@pytest.mark.parametrize("lens", [[1], [3, 9, 2], [17, 11], [33], [33, 31], [20, 41, 64, 7], [120] * 7, [125] * 40])
def test_native_encoder_forward_is_the_ops_forward(preset, lens):
    """One native call against the same forward op by op, over the ways it goes (norms in the products up to 32 rows, parts of K
    in smaller tiles up to 512, larger tiles beyond: the same sums, so the same bits), rows placed in another order."""
    from rag_tl_domainllm_optimizer_amd import models
    import dataclasses

    cfg = dataclasses.replace(models.resolve_preset(preset), num_layers=2)
    m = models.SentenceEncoder(cfg, device=DEV, dtype=torch.bfloat16, init=False).eval()
    g = torch.Generator(device=DEV).manual_seed(len(lens))
    with torch.no_grad():
        for name, p in m.named_parameters():
            p.normal_(1.0 if "ln" in name and name.endswith("_w") else 0.0, 0.05, generator=g)
    n = torch.tensor(lens, device=DEV)
    off = torch.nn.functional.pad(n.cumsum(0), (1, 0))
    rows = int(off[-1])
    ids = torch.randint(4, cfg.vocab_size, (rows,), generator=g, device=DEV)
    pos = torch.cat([torch.arange(k, device=DEV) for k in lens]) + m.first_position
    to = torch.randperm(len(lens), generator=g, device=DEV)
    out = torch.full((len(lens) + 1, cfg.hidden_size), 7.0, device=DEV)
    assert m._encode_native(ids, pos, off, max(lens), True, out, to)
    want = m.encode_packed(ids, pos, off, max(lens))
    assert (out[-1] == 7).all()
    assert torch.equal(out[to], want)
    # not for layers of another make: op by op again
    class Other(type(m.layers[0])):
        pass
    m.layers[0].__class__ = Other
    assert not m._encode_native(ids, pos, off, max(lens), True, out, to)
    got = torch.zeros(len(lens), cfg.hidden_size, device=DEV)
    m.encode_packed(ids, pos, off, max(lens), True, got, to)
    assert torch.equal(got[to], want)


def _few_rows_encoder(heads, seed, **kw):
    from rag_tl_domainllm_optimizer_amd import models
    import dataclasses

    cfg = dataclasses.replace(models.resolve_preset("minilm-l6"), num_layers=3, num_heads=heads, **{"head_dim": 384 // heads, **kw})
    m = models.SentenceEncoder(cfg, device=DEV, dtype=torch.bfloat16, init=False).eval()
    g = torch.Generator(device=DEV).manual_seed(seed)
    with torch.no_grad():
        for name, p in m.named_parameters():
            p.normal_(1.0 if "ln" in name and name.endswith("_w") else 0.0, 0.05, generator=g)

    def inputs(lens, gap=0):
        off = gap + torch.nn.functional.pad(torch.tensor(lens, device=DEV).cumsum(0), (1, 0))
        rows = int(off[-1]) + gap
        ids = torch.randint(4, cfg.vocab_size, (rows,), generator=g, device=DEV)
        pos = torch.randint(0, 100, (rows,), generator=g, device=DEV)
        return ids, pos, off, max(lens)
    return m, inputs


# 12 heads of 32, 6 of 64: one launch for the layers; 3 of 128: one by one
@pytest.mark.parametrize("heads,kw", [(12, {}), (6, {}), (3, {}), (6, dict(intermediate_size=1472))])
@pytest.mark.parametrize("lens,gap", [([15], 0), ([16], 0), ([31], 0), ([32], 0), ([48], 0), ([49], 0), ([64], 0), ([1] * 41, 0),
                                      ([0, 5, 0, 33, 0], 0), ([17, 16, 30], 0), ([9, 20], 2), ([2], 31)])
def test_encoder_of_few_rows(heads, kw, lens, gap):
    """Up to 64 rows against the same forward op by op, the same bits: around the 16-row tiles and the 32-query blocks, many texts,
    texts without rows, rows ahead of the first text and behind the last."""
    m, inputs = _few_rows_encoder(heads, len(lens) + heads, **kw)
    ids, pos, off, longest = inputs(lens, gap)
    out = torch.full((len(lens), m.cfg.hidden_size), 7.0, device=DEV)
    assert m._encode_native(ids, pos, off, longest, True, out, torch.arange(len(lens), device=DEV))
    assert torch.equal(out, m.encode_packed(ids, pos, off, longest))


def test_encoder_of_few_rows_replayed_and_on_two_streams():
    """A captured forward gives every replay's inputs their results, with eager calls between; two streams at once theirs."""
    m, inputs = _few_rows_encoder(12, 3)
    cases = [inputs(lens) for lens in ([40], [15], [40], [33, 7], [12, 28])]
    want = [m.encode_packed(*c) for c in cases]
    outs = [torch.zeros_like(w) for w in want]
    tos = [torch.arange(len(w), device=DEV) for w in want]
    ids, pos, off, longest = (t.clone() if torch.is_tensor(t) else t for t in cases[0])
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        m._encode_native(ids, pos, off, longest, True, outs[0], tos[0])
    for k in (0, 2, 0, 2):
        ids.copy_(cases[k][0])
        pos.copy_(cases[k][1])
        m._encode_native(*cases[1], True, outs[1], tos[1])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(outs[0], want[k]) and torch.equal(outs[1], want[1])
    streams = [torch.cuda.Stream() for _ in cases]
    torch.cuda.synchronize()
    for _ in range(20):
        for s, c, o, t in zip(streams, cases, outs, tos):
            with torch.cuda.stream(s):
                m._encode_native(*c, True, o, t)
    torch.cuda.synchronize()
    assert all(torch.equal(o, w) for o, w in zip(outs, want))


@pytest.mark.parametrize("where", ["word_embed", "emb_ln_b", "layers.0.qkv_b", "layers.1.fc1_w", "layers.2.ln2_w"])
def test_encoder_of_few_rows_with_all_ones(where):
    """Words of all ones (NaN) among the parameters: NaN comes out, of no text that they do not reach."""
    m, inputs = _few_rows_encoder(12, 4)
    ids, pos, off, longest = inputs([15, 20])
    ids[:20], ids[20:] = 5, 6
    p = dict(m.named_parameters())[where]
    with torch.no_grad():
        (p[5] if where == "word_embed" else p).view(torch.int16).fill_(-1)
    out = torch.zeros(2, m.cfg.hidden_size, device=DEV)
    assert m._encode_native(ids, pos, off, longest, True, out, torch.arange(2, device=DEV))
    want = m.encode_packed(ids, pos, off, longest)
    assert torch.equal(out.isnan(), want.isnan()) and out[0].isnan().any()
    torch.testing.assert_close(out, want, rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("rows", [64, 128])
@pytest.mark.parametrize("M,K", [(1, 64), (63, 128), (64, 192), (65, 384), (127, 320), (128, 1536), (129, 64), (300, 448), (16400, 384)])
def test_product_and_norm_in_one_launch(M, K, rows):
    """LN(x w^T + b + res) with the bits of product and norm, and close to 64 bits: ends of tiles, fewer K-steps than are fetched ahead, odd
    numbers of them, a NaN, an infinite and a huge row (whose variance overflows) among the others, rows around the result."""
    C = ops.native()
    g = torch.Generator(device=DEV).manual_seed(M + K + rows)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(384, K, generator=g, device=DEV) / K ** 0.5).bfloat16()
    bias, lb = (torch.randn(384, generator=g, device=DEV).bfloat16() for _ in range(2))
    lw = (1 + 0.1 * torch.randn(384, generator=g, device=DEV)).bfloat16()
    res = torch.randn(M, 384, generator=g, device=DEV).bfloat16()
    got = C.linear_norm(x, w, bias, res, lw, lb, 1e-12, rows)
    want = ops.layer_norm(C.gemm_big(x, w, 0, 0, bias=bias), lw, lb, 1e-12, residual=res)[0]
    assert torch.equal(got, want)
    # product and sum are rounded to bf16 (2^-9 of values below 8) ahead of a division by about 1.4, the result (below 8) once more
    h = x.double() @ w.double().t() + bias.double() + res.double()
    ref = torch.nn.functional.layer_norm(h, (384,), lw.double(), lb.double(), 1e-12)
    assert (got.double() - ref).abs().max().item() < 3 * 8 * 2 ** -9
    if M < 60:
        return
    x[5, 3], res[17, 20], res[M - 1] = float("nan"), float("inf"), 1e30 * torch.sign(res[M - 1].float()).bfloat16()
    got = C.linear_norm(x, w, bias, res, lw, lb, 1e-12, rows)
    want2 = ops.layer_norm(C.gemm_big(x, w, 0, 0, bias=bias), lw, lb, 1e-12, residual=res)[0]
    torch.testing.assert_close(got, want2, rtol=0, atol=0, equal_nan=True)
    keep = [i for i in range(min(M - 1, 200)) if i not in (5, 17)]
    assert got[5].isnan().all() and torch.equal(got[keep], want[keep])


# rows of the tiles of the output product (K 384) and of the second feed-forward product (K 1536), 0: product and norm apart
@pytest.mark.parametrize("lens,tiles", [([3999], (0, 0)), ([4000], (64, 0)), ([6407], (64, 0)), ([6407, 1], (64, 64)), ([5000, 11384], (64, 64)),
                                        ([9000, 7385], (128, 128)), ([1] * 500 + [17000], (128, 128))])
def test_encoder_where_products_take_the_norm(lens, tiles):
    """Around the row counts where the output and the second feed-forward product begin to end in the norm and where their tiles
    grow, the bits of the forward op by op."""
    assert tuple(ops.native().linear_norm_tiles(sum(lens), 384, K)[0] for K in (384, 1536)) == tiles
    m, inputs = _few_rows_encoder(12, sum(lens))
    ids, pos, off, longest = inputs(lens)
    out = torch.full((len(lens), m.cfg.hidden_size), 7.0, device=DEV)
    assert m._encode_native(ids, pos, off, longest, True, out, torch.arange(len(lens), device=DEV))
    assert torch.equal(out, m.encode_packed(ids, pos, off, longest))


def test_native_encoder_writes_no_row_beyond_out():
    """Rows counted from the end go there, texts whose row does not exist go nowhere: the rows around out stay as they are."""
    from rag_tl_domainllm_optimizer_amd import models
    import dataclasses

    m = models.SentenceEncoder(dataclasses.replace(models.resolve_preset("minilm-l6"), num_layers=1), device=DEV, dtype=torch.bfloat16).eval()
    lens = [5, 9, 3, 7]
    off = torch.nn.functional.pad(torch.tensor(lens, device=DEV).cumsum(0), (1, 0))
    ids = torch.arange(10, 10 + sum(lens), device=DEV)
    pos = torch.cat([torch.arange(n, device=DEV) for n in lens])
    buf = torch.full((12, m.cfg.hidden_size), 7.0, device=DEV)
    m.encode_packed(ids, pos, off, max(lens), True, buf[4:8], torch.tensor([2, -1, 4, -5], device=DEV))
    want = m.encode_packed(ids, pos, off, max(lens))
    assert torch.equal(buf[6], want[0]) and torch.equal(buf[7], want[1])
    assert (buf[:6] == 7).all() and (buf[8:] == 7).all()


# ---------------------------------------------------------------------------------------------- decode products, 65..128 rows
@pytest.mark.parametrize("N,K,act", [(16, 64, 0), (48, 448, 0), (2048, 1024, 0), (4112, 2112, ops.ACT_RELU2), (33024, 256, 0),
                                     (64, 128, 5), (1056, 1088, 5), (33024, 320, 5)])
def test_image_products_65_to_128_rows(N, K, act):
    """Tile-ordered products at 65..128 rows against 64 bits: odd numbers of row groups and chunks, chosen splits and
    none, unreduced sums, fp32 and strided results. The bound on fp32 results is that of the sum's order."""
    C = ops.native()
    g = torch.Generator(device=DEV).manual_seed(N + K)
    w = (torch.randn(N, K, generator=g, device=DEV) / K ** 0.5).bfloat16()
    shuf = ops.ShufCache()
    No = N // 2 if act == ops.ACT_SWIGLU else N
    for M in (65, 96, 97, 128):
        x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
        pre = x.double() @ w.double().t()
        want = torch.nn.functional.silu(pre[:, :No]) * pre[:, No:] if act == ops.ACT_SWIGLU else ref.apply_act(pre, act)
        bound = (x.double().abs() @ w.double().abs().t()).max().item() * K * 2.0 ** -24 + 1e-6
        out = torch.full((M, No + 8), 7.0, dtype=torch.bfloat16, device=DEV)
        assert ops.image_rows(x, w, shuf, act)
        ops.gemm_image(x, w, shuf, act, out=out[:, :No])
        # a bf16 rounding of the result, and of the pre-activations where a split hands those to the reduction
        torch.testing.assert_close(out[:, :No].double(), want, rtol=2.0 ** -6, atol=4 * bound + 2.0 ** -8)
        assert (out[:, No:] == 7).all()
        if act == 0:
            for s in {1, min(2, K // 64), min(7, K // 64)}:
                slabs = torch.empty(s * M * N, dtype=torch.float32, device=DEV)
                assert C.gemm_image(x, shuf.get(w), 0, False, None, s, slabs, True) is None
                assert (slabs.view(s, M, N).double().sum(0) - pre).abs().max().item() <= bound
            y = C.gemm_image(x, shuf.get(w), 0, True)
            assert (y.double() - pre).abs().max().item() <= bound
    for M in (64, 129):
        x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
        assert not ops.image_rows(x, w, shuf, act)
        with pytest.raises(RuntimeError):
            C.gemm_image(x, shuf.get(w), act)
    with ops.batch_invariant():
        assert not ops.image_rows(torch.zeros(96, K, dtype=torch.bfloat16, device=DEV), w, shuf, act)


@pytest.mark.parametrize("m", [17, 48, 64, 65, 128])
def test_weights_that_row_major_products_refuse(m):
    """Column strides and rows off 16 bytes are refused with an image at hand as without one; rows further apart are not."""
    K, N = 256, 512
    x = torch.ones(m, K, dtype=torch.bfloat16, device=DEV)
    buf = torch.ones(N * (K + 8) + 8, dtype=torch.bfloat16, device=DEV)
    for w in (buf[:N * K].view(K, N).t(), buf[1:1 + N * K].view(N, K), buf[:N * (K + 4)].view(N, K + 4)[:, :K]):
        with pytest.raises(RuntimeError):
            ops.project(x, w, shuf=ops.ShufCache())
        with pytest.raises(RuntimeError):
            ops.act_project(x, w, ops.ACT_RELU2, ops.ShufCache())
    w = buf[:N * (K + 8)].view(N, K + 8)[:, :K]
    assert bool((ops.project(x, w, shuf=ops.ShufCache()) == K).all())


def test_weight_images_across_streams_captures_and_copies():
    """An image that one stream is still laying out is waited for on another, also after the weight has changed; a capture
    without a warm-up leaves no image behind that only its replay fills; copies and pickles start empty."""
    import copy
    import pickle

    g = torch.Generator(device=DEV).manual_seed(5)
    w = (torch.randn(4096, 4096, generator=g, device=DEV) / 64).bfloat16()
    x = torch.randn(100, 4096, generator=g, device=DEV).bfloat16()
    shuf, a, b = ops.ShufCache(), torch.cuda.Stream(), torch.cuda.Stream()

    def check(y):
        torch.testing.assert_close(y.double(), x.double() @ w.double().t(), rtol=2.0 ** -6, atol=2.0 ** -6)

    for _ in range(2):
        torch.cuda.synchronize()
        with torch.cuda.stream(a):
            torch.cuda._sleep(100_000_000)
            shuf.get(w)
        with torch.cuda.stream(b):
            y = ops.project(x, w, shuf=shuf)
        torch.cuda.synchronize()
        check(y)
        w.mul_(-0.5)
    for m in (16, 48, 100):
        shuf = ops.ShufCache()
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            y = ops.project(x[:m], w, shuf=shuf)
        check(torch.cat([ops.project(x[:m], w, shuf=shuf), x.double()[m:] @ w.double().t()]))
        for _ in range(3):
            y.zero_()
            graph.replay()
            torch.cuda.synchronize()
            check(torch.cat([y, x.double()[m:] @ w.double().t()]))
    assert shuf and not copy.deepcopy(shuf) and not copy.copy(shuf) and not pickle.loads(pickle.dumps(shuf))


# ---------------------------------------------------------------------------------------------- norms
@pytest.mark.parametrize("H", [8, 520, 2048, 4096, 5120, 8192, 11008, 13312])
@pytest.mark.parametrize("T", [5, 300])
def test_slab_sums_by_their_number(T, H):
    """One to ten slabs, on either side of the CUs' number: the sum in slab order, rounded once, in the reduction and ahead of a norm;
    the norm of the rounded stream to one rounding (2^-8 of it, and 1e-5 for 32-bit sums)."""
    from rag_tl_domainllm_optimizer_amd.ops.linear import SplitK

    g = torch.Generator(device=DEV).manual_seed(T + H)
    res, w = (torch.randn(n, H, generator=g, device=DEV).bfloat16() for n in (T, 1))
    for ns in (1, 2, 3, 4, 5, 6, 7, 8, 9, 10):
        slabs = torch.randn(ns, T, H, generator=g, device=DEV)
        sk = SplitK(slabs.reshape(-1), ns, T, H, torch.bfloat16)
        total = slabs[0].clone()
        for q in range(1, ns):
            total += slabs[q]
        assert torch.equal(sk.reduce(), total.bfloat16())
        y, h = ops.rms_norm(sk, w[0], 1e-5, res)
        assert torch.equal(h, (total.bfloat16().float() + res.float()).bfloat16())
        x = h.double()
        want = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-5) * w.double()
        assert ((y.double() - want).abs() <= (2.0 ** -8 + 1e-5) * want.abs()).all()


@pytest.mark.parametrize("H", [8, 384, 512, 520, 768, 1024, 1032])
@pytest.mark.parametrize("T", [1, 5, 1023, 1024, 9001])
def test_norm_wave_per_row_bits(H, T):
    """Rows of up to 1024 columns have one bit pattern whichever form the number of rows picks (and up to 512 columns
    that of the split-K form's workgroup a row), with and without the residual sum written."""
    g = torch.Generator(device=DEV).manual_seed(H)
    x, r = (torch.randn(T, H, generator=g, device=DEV).bfloat16() for _ in range(2))
    w, b = (torch.randn(H, generator=g, device=DEV).bfloat16() for _ in range(2))
    C = ops.native()
    for ln in (False, True):
        y, h, rstd, mean = C.norm_fwd(ln, x, r, w, b if ln else None, 1e-5)
        y2, h2, rstd2, _ = C.norm_fwd(ln, x, r, w, b if ln else None, 1e-5, False)
        assert h2 is None and torch.equal(y, y2) and torch.equal(rstd, rstd2)
        ys, hs = C.norm_fwd_slabs(ln, x.float(), 1, T, H, r, w, b if ln else None, 1e-5)[:2]
        assert torch.equal(y, ys) and torch.equal(h, hs)
        hd = h.double()
        want = hd - hd.mean(-1, keepdim=True) if ln else hd
        want = want * torch.rsqrt(want.pow(2).mean(-1, keepdim=True) + 1e-5) * w.double() + (b.double() if ln else 0)
        torch.testing.assert_close(y.double(), want, rtol=2.0 ** -8 + 1e-4, atol=1e-4)


@pytest.mark.parametrize("mode", ["bf16", "fp8", "adapters apart"])
def test_decode_weight_images_only_where_read(mode):
    """A decode of 80 rows lays out images of the weights that it reads through them; a refresh adds none, for fp8 weights or
    adapters that are not merged either."""
    from rag_tl_domainllm_optimizer_amd import models
    from rag_tl_domainllm_optimizer_amd.generation import Generator, SamplingParams
    from rag_tl_domainllm_optimizer_amd.models.config import ModelConfig

    cfg = ModelConfig(arch="mistral", vocab_size=512, hidden_size=512, num_layers=1, num_heads=4, num_kv_heads=1,
                      head_dim=128, intermediate_size=1024, max_position=128, norm_eps=1e-5, name="t-d128")
    m = models.CausalLM(cfg, device=DEV, dtype=torch.bfloat16, seed=6)
    if mode == "fp8":
        m.set_fp8(True)
    elif mode != "bf16":
        m.add_lora(8, 16.0, "all")
    Generator(m, 80, 32, DEV, use_graph=False).generate([[3, 4, 5]] * 80, SamplingParams(max_new_tokens=3, do_sample=False),
                                                         pad_id=0, eos_ids=[-1])
    layer = m.layers[0]
    held = {k for k, c in layer._shufc.items() if c}
    layer.refresh_decode_weights()
    m.refresh_decode_weights(80)
    assert {k for k, c in layer._shufc.items() if c} == held
    if mode == "bf16":
        assert held == {"qkv_plain", "o", "gate_up_plain", "down"}
    elif mode == "fp8":
        assert not held


@pytest.mark.parametrize("n,dtype", [(0, np.int64), (1, np.int32), (131072, np.int64), (131073, np.int64)])
def test_upload_holds_the_source_of_the_call(n, dtype):
    """ops.upload up to its pinned limit and beyond: the values at the call, whatever becomes of the source, behind a busy stream."""
    src = np.arange(2 * n, dtype=dtype)[::2]
    want = src.copy()
    torch.cuda._sleep(2_000_000)
    got = [ops.upload(src, DEV), ops.upload(torch.from_numpy(src), DEV)]
    src += 7
    for g in got:
        assert g.device.type == "cuda" and g.is_contiguous() and np.array_equal(g.cpu().numpy(), want)


def test_upload_under_a_default_device():
    """ops.upload and the tables made with it where new tensors go to the GPU by default, numpy arrays and CPU tensors alike."""
    src = np.arange(1000, dtype=np.int64)
    with torch.device(DEV):
        got = [ops.upload(src, DEV), ops.upload(torch.from_numpy(src), DEV), ops.upload(torch.arange(1000), DEV)]
        batch = RaggedBatch.build([(0, [5, 6, 7], 0), (1, [8] * 40, 3)], DEV)
    for g in got:
        assert g.device.type == "cuda" and torch.equal(g.cpu(), torch.from_numpy(src))
    assert batch.ids.tolist() == [5, 6, 7] + [8] * 40 and batch.pos.tolist() == [0, 1, 2] + list(range(3, 43))


@pytest.mark.parametrize("rows", [64, 96])
@pytest.mark.parametrize("M,K", [(1, 64), (63, 128), (64, 192), (65, 384), (95, 320), (96, 768), (97, 64), (193, 448), (24580, 128)])
def test_product_and_norm_of_768_columns_in_one_launch(M, K, rows):
    """As with 384 columns: the bits of product and norm, close to 64 bits; NaN, infinite and huge rows stay their own."""
    C = ops.native()
    g = torch.Generator(device=DEV).manual_seed(M + K + rows)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(768, K, generator=g, device=DEV) / K ** 0.5).bfloat16()
    bias, lb = (torch.randn(768, generator=g, device=DEV).bfloat16() for _ in range(2))
    lw = (1 + 0.1 * torch.randn(768, generator=g, device=DEV)).bfloat16()
    res = torch.randn(M, 768, generator=g, device=DEV).bfloat16()
    got = C.linear_norm(x, w, bias, res, lw, lb, 1e-12, rows)
    want = ops.layer_norm(C.gemm_big(x, w, 0, 0, bias=bias), lw, lb, 1e-12, residual=res)[0]
    assert torch.equal(got, want)
    # product and sum are rounded to bf16 (2^-9 of values below 8) ahead of a division by about 1.4, the result (below 8) once more
    h = x.double() @ w.double().t() + bias.double() + res.double()
    ref = torch.nn.functional.layer_norm(h, (768,), lw.double(), lb.double(), 1e-12)
    assert (got.double() - ref).abs().max().item() < 3 * 8 * 2 ** -9
    if M < 60:
        return
    x[5, 3], res[17, 700], res[M - 1] = float("nan"), float("inf"), 1e30 * torch.sign(res[M - 1].float()).bfloat16()
    got = C.linear_norm(x, w, bias, res, lw, lb, 1e-12, rows)
    want2 = ops.layer_norm(C.gemm_big(x, w, 0, 0, bias=bias), lw, lb, 1e-12, residual=res)[0]
    torch.testing.assert_close(got, want2, rtol=0, atol=0, equal_nan=True)
    keep = [i for i in range(min(M - 1, 200)) if i not in (5, 17)]
    assert got[5].isnan().all() and torch.equal(got[keep], want[keep])


# 768 columns, K of 768 and 3072: around the row counts where the rule changes between product and norm (0), tiles of 64, of 96, and both (the
# rest in 64 behind leading rows in 96)
@pytest.mark.parametrize("lens,tiles", [([7150], (0, 0)), ([7151], (64, 0)), ([10345], (64, 0)), ([10346], (64, 64)), ([16384], (64, 64)),
                                        ([16385], (96, 0)), ([21760], (96, 96)), ([20000, 4576], (96, 96)), ([24577], (64, 0)),
                                        ([34001], ((64, 24576), (64, 24576))), ([41000], (64, 0)), ([46000], (64, 96))])
def test_encoder_of_768_columns_where_products_take_the_norm(lens, tiles):
    """The bits of the forward op by op."""
    for K, t in zip((768, 3072), tiles):
        assert ops.native().linear_norm_tiles(sum(lens), 768, K) == (t if isinstance(t, tuple) else (t, 0))
    m, inputs = _few_rows_encoder(12, sum(lens), hidden_size=768, intermediate_size=3072, head_dim=64)
    ids, pos, off, longest = inputs(lens)
    out = torch.full((len(lens), m.cfg.hidden_size), 7.0, device=DEV)
    assert m._encode_native(ids, pos, off, longest, True, out, torch.arange(len(lens), device=DEV))
    assert torch.equal(out, m.encode_packed(ids, pos, off, longest))


@pytest.mark.parametrize("nlist,d", [(1, 64), (15, 128), (16, 256), (17, 320), (130, 384), (512, 384), (1000, 768), (300, 2048), (2000, 1088)])
@pytest.mark.parametrize("l2", [False, True])
def test_probes_of_few_queries(nlist, d, l2):
    """The lists that product and top-k find, and the query that rounding alone gives, on both sides of the 16 queries of one launch: repeated
    centroids (ties), a NaN query, queries that are not fp32 or not contiguous, all lists, more than the selection kernel takes."""
    g = torch.Generator(device=DEV).manual_seed(nlist + d)
    cen = torch.randn((nlist + 127) // 128 * 128, d, generator=g, device=DEV).bfloat16()
    cen[nlist // 2] = cen[0]
    pen = torch.randn(nlist, generator=g, device=DEV) if l2 else None
    for nq in (1, 3, 16, 17):
        q = torch.randn(nq, 2 * d, generator=g, device=DEV)
        q[nq - 1, 0] = float("nan")
        for x in (q[:, :d].contiguous(), q[:, :d], q[:, :d].bfloat16(), q[:, 1:d + 1]):
            for k in {1, min(16, nlist), nlist}:
                s = ops.gemm(x.contiguous().bfloat16(), cen, out_f32=True)[:, :nlist]
                if l2:
                    s = s - pen
                qb, got = ops.ivf_probes(x, cen, nlist, k, pen)
                assert torch.equal(qb.view(torch.int16), x.contiguous().bfloat16().view(torch.int16))
                assert got.dtype == torch.int32
                fine = slice(0, nq - 1) if x.isnan().any() else slice(0, nq)
                assert torch.equal(got[fine].long(), ops.topk(s, k)[1][fine])


@pytest.mark.parametrize("Hq,Hkv,D", [(8, 2, 128), (4, 4, 128), (6, 2, 64), (3, 3, 32)])
@pytest.mark.parametrize("S,lens,window", [(5, [5, 1, 3], 0), (64, [64, 63, 1, 0], 0), (129, [129, 0, 66, 128], 40), (300, [7, 300, 65, 200], 0),
                                           (1100, [1100, 1, 900], 500)])
def test_prompt_attention_over_rows_where_they_lie(Hq, Hkv, D, S, lens, window):
    """The bits of the filled grid, attention and gather, and the caches' of its append, pads among them: tiles that are all pads or partly, rows of
    one token and of none, head-packed and other tiles, a window."""
    from rag_tl_domainllm_optimizer_amd.models import packed_index

    B, W = len(lens), (Hq + 2 * Hkv) * D
    g = torch.Generator(device=DEV).manual_seed(S + D)
    start = np.array([S - n for n in lens])
    idx, off = packed_index(start, np.full(B, S), S, torch.device(DEV))
    qkv = torch.randn(int(off[-1]), W + 8, generator=g, device=DEV).bfloat16()[:, :W]
    ks = torch.tensor(start, dtype=torch.int32, device=DEV)
    inv = ops.packed_inverse(idx, B * S)
    first = torch.tensor([int(off[b]) - int(start[b]) for b in range(B)], dtype=torch.int32, device=DEV)
    kc, vc, kc0, vc0 = (torch.full((B, Hkv, S + 3, D), 5.0, device=DEV).bfloat16() for _ in range(4))
    got = ops.prefill_attention_rows(qkv, first, inv, S, Hq, Hkv, D, kc, vc, window, kv_start=ks)
    grid = ops.scatter_rows(qkv, idx, inv, B * S)
    pos = torch.zeros(B * S, dtype=torch.int32, device=DEV)
    ops.rope_qkv_(grid, pos, None, None, Hq, Hkv, D, S=S, k_cache=kc0, v_cache=vc0)
    want = ops.gather_rows(ops.flash_attention_qkv(grid, B, S, Hq, Hkv, D, True, window, kv_start=ks), idx, inv)
    assert torch.equal(got, want) and torch.equal(kc, kc0) and torch.equal(vc, vc0)


@pytest.mark.parametrize("preset", ["tiny-mistral", "tiny-llama", "tiny-opt"])
def test_packed_prefill_of_rows_equals_grid(preset):
    """A whole prompt forward with pads left out and with pads worked on: close (products of other row counts sum in another order), caches of pads zero."""
    from rag_tl_domainllm_optimizer_amd import models
    from rag_tl_domainllm_optimizer_amd.generation import KVCache

    cfg = models.resolve_preset(preset)
    m = models.CausalLM(cfg, device=torch.device(DEV), dtype=torch.bfloat16, seed=0)
    lens, S = [30, 7, 1, 18], 30
    g = torch.Generator().manual_seed(1)
    ids = torch.randint(3, cfg.vocab_size, (len(lens), S), generator=g)
    start = torch.tensor([S - n for n in lens], dtype=torch.int32)
    out = []
    for packed in (None, models.packed_index(start.numpy(), np.full(len(lens), S), S, torch.device(DEV))):
        cache = KVCache(cfg.num_layers, len(lens), cfg.num_kv_heads, 64, cfg.head_dim, torch.device(DEV), torch.bfloat16)
        cache.k.zero_()
        cache.v.zero_()
        out.append((m.prefill(ids.to(DEV), start.to(DEV), cache, packed=packed), cache))
    _close(out[0][0], out[1][0])
    for b, s in enumerate(start.tolist()):
        _close(out[0][1].k[:, b, :, s:S], out[1][1].k[:, b, :, s:S])
        assert not out[1][1].k[:, b, :, :s].any() and not out[1][1].v[:, b, :, :s].any()


@pytest.mark.parametrize("lens,tiles", [([32768], (128, 0)), ([32769], (64, 32768)), ([34000], (64, 32768)), ([20000, 20000], (64, 32768)),
                                        ([49152], (64, 32768)), ([49200], (128, 0))])
def test_encoder_of_384_columns_in_tiles_of_two_sizes(lens, tiles):
    """Around whole rounds of the larger tiles, whose rest goes in smaller ones: the bits of the forward op by op."""
    assert all(ops.native().linear_norm_tiles(sum(lens), 384, K) == tiles for K in (384, 1536))
    m, inputs = _few_rows_encoder(12, sum(lens))
    ids, pos, off, longest = inputs(lens)
    out = torch.full((len(lens), m.cfg.hidden_size), 7.0, device=DEV)
    assert m._encode_native(ids, pos, off, longest, True, out, torch.arange(len(lens), device=DEV))
    assert torch.equal(out, m.encode_packed(ids, pos, off, longest))


def test_encoder_batches_that_go_together():
    """Batches in one forward give what they give one by one; other row counts may sum products in another order: a bf16 rounding or two of
    unit vectors of 384."""
    from rag_tl_domainllm_optimizer_amd.retrieval import Encoder
    from rag_tl_domainllm_optimizer_amd.tokenizer import Tokenizer

    m, _ = _few_rows_encoder(12, 5)
    tok = Tokenizer.synthetic(m.cfg.vocab_size, m.cfg.arch)
    words = tok.words()
    texts = [" ".join(words[(7 * i + k) % len(words)] for k in range(i % 40)) for i in range(200)]
    got = Encoder(m, tok, max_length=64, batch_size=16, max_rows=10 ** 6).encode(texts)
    assert (got - Encoder(m, tok, max_length=64, batch_size=16).encode(texts)).abs().max().item() < 4e-3


@pytest.mark.parametrize("M", [8, 48])
def test_products_captured_first_on_a_stream(M):
    """A stream whose first split product is captured: the workspace it makes is ready for whichever graph is replayed first, beside
    what the graphs' pool held before, and for eager products on the stream."""
    import ctypes

    C = ops.native()
    hip = ctypes.CDLL("libamdhip64.so")
    handle = ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(handle), 1) == 0  # one of torch's might have a workspace; 1: beside the default stream
    s = torch.cuda.ExternalStream(handle.value)
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randn(M, 4096, generator=g, device=DEV).bfloat16()
    w = (torch.randn(2048, 4096, generator=g, device=DEV) / 64).bfloat16()
    img = C.shuffle_decode_weight(w)
    with ops.tuning(decode_split=4):
        want = C.gemm(x, img, None, None, None, 0, False, None, None, 0.0, True)
        pool, junk = torch.cuda.graph_pool_handle(), []
        torch.cuda.synchronize()
        first, graphs, outs = torch.cuda.CUDAGraph(), [], []
        with torch.cuda.graph(first, pool=pool, stream=s):
            junk += [torch.full((1 << 16,), 7, dtype=torch.int32, device=DEV) for _ in range(8)]
        first.replay()
        torch.cuda.synchronize()
        junk.clear()  # back to the pool, with the sevens
        for _ in range(2):
            graphs.append(torch.cuda.CUDAGraph())
            with torch.cuda.graph(graphs[-1], pool=pool, stream=s):
                outs.append(C.gemm(x, img, None, None, None, 0, False, None, None, 0.0, True))
        assert not any(C.decode_ws_dirty_tickets())
        for k in (1, 0, 1):
            with torch.cuda.stream(s):
                assert torch.equal(C.gemm(x, img, None, None, None, 0, False, None, None, 0.0, True), want)
            torch.cuda.synchronize()
            outs[k].fill_(5)
            graphs[k].replay()
            torch.cuda.synchronize()
            assert torch.equal(outs[k], want)


def test_zeros_of_products_are_made_while_capturing():
    """A process whose first product is captured: what products read in place of columns that are not there is zero before the graph is
    replayed, whatever the graph's pool held."""
    import subprocess
    import sys

    code = """
import torch
from rag_tl_domainllm_optimizer_amd import ops
C, dev = ops.native(), "cuda"
x, w = (torch.ones(200, 72, device=dev, dtype=torch.bfloat16) for _ in range(2))
pool, graphs, s = torch.cuda.graph_pool_handle(), [torch.cuda.CUDAGraph() for _ in range(2)], torch.cuda.Stream()
torch.cuda.synchronize()
with torch.cuda.graph(graphs[0], pool=pool, stream=s):
    junk = [torch.full((2048,), 7, dtype=torch.bfloat16, device=dev) for _ in range(512)]
graphs[0].replay()
torch.cuda.synchronize()
del junk
with torch.cuda.graph(graphs[1], pool=pool, stream=s):
    y = C.gemm_big(x, w, 0, 0)
print(C.gemm_big(x, w, 0, 0).unique().tolist())
graphs[1].replay()
torch.cuda.synchronize()
print(y.unique().tolist())
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.split() == ["[72.0]", "[72.0]"], r.stdout + r.stderr[-2000:]


@pytest.mark.parametrize("Hq,Hkv,D", [(8, 2, 128), (4, 4, 128), (6, 2, 64), (3, 3, 32)])
@pytest.mark.parametrize("S,lens,window", [(70, [70, 3, 66, 1], 0), (200, [200, 130, 7, 64], 50)])
def test_prompt_attention_over_rows_of_infinite_values(Hq, Hkv, D, S, lens, window):
    """Infinite and NaN values at a row's first and last token: the grid's results, whose pads are zeros."""
    from rag_tl_domainllm_optimizer_amd.models import packed_index

    B, W = len(lens), (Hq + 2 * Hkv) * D
    g = torch.Generator(device=DEV).manual_seed(S + D)
    start = np.array([S - n for n in lens])
    idx, off = packed_index(start, np.full(B, S), S, torch.device(DEV))
    qkv = torch.randn(int(off[-1]), W, generator=g, device=DEV).bfloat16()
    v = qkv[:, (Hq + Hkv) * D:]
    v[off[:-1], 0], v[off[:-1], D - 1], v[off[1:] - 1, 1] = float("inf"), float("-inf"), float("nan")
    ks = torch.tensor(start, dtype=torch.int32, device=DEV)
    inv = ops.packed_inverse(idx, B * S)
    first = torch.tensor([int(off[b]) - int(start[b]) for b in range(B)], dtype=torch.int32, device=DEV)
    kc, vc = (torch.zeros(B, Hkv, S, D, device=DEV).bfloat16() for _ in range(2))
    got = ops.prefill_attention_rows(qkv, first, inv, S, Hq, Hkv, D, kc, vc, window, kv_start=ks)
    grid = ops.scatter_rows(qkv, idx, inv, B * S)
    want = ops.gather_rows(ops.flash_attention_qkv(grid, B, S, Hq, Hkv, D, True, window, kv_start=ks), idx, inv)
    assert want.isinf().any() and want.isnan().any()
    torch.testing.assert_close(got, want, rtol=0, atol=0, equal_nan=True)


def test_encoder_batch_size_bounds_a_forward():
    """A batch size of the caller's: no forward of more texts, unless rows are allowed; 256, the default: batches together."""
    from rag_tl_domainllm_optimizer_amd.retrieval import Encoder
    from rag_tl_domainllm_optimizer_amd.tokenizer import Tokenizer

    m, _ = _few_rows_encoder(12, 6)
    tok = Tokenizer.synthetic(m.cfg.vocab_size, m.cfg.arch)
    words = tok.words()
    texts = [" ".join(words[(7 * i + k) % len(words)] for k in range(1 + i % 9)) for i in range(600)]
    forward, seen = m._encode_native, []
    m._encode_native = lambda ids, pos, off, *a: seen.append((len(off) - 1, len(ids))) or forward(ids, pos, off, *a)

    def forwards(**kw):
        seen.clear()
        Encoder(m, tok, max_length=64, **kw).encode(texts)
        return list(seen)
    assert max(n for n, _ in forwards(batch_size=16)) == 16
    assert max(n for n, _ in forwards(batch_size=500)) == 500
    assert [n for n, _ in forwards()] == [600] and [n for n, _ in forwards(max_rows=0)] == [256, 256, 88]
    assert len(forwards(batch_size=16, max_rows=1000)) < 600 // 16 and all(r <= 1000 for _, r in forwards(batch_size=16, max_rows=1000))


def test_encoder_of_few_rows_says_that_it_gave_up():
    """A forward whose waits end at once: NaN, and an error from the next forward, from filling an index and where it is asked for, once;
    the forwards after that are as before."""
    from rag_tl_domainllm_optimizer_amd.retrieval import IVFIndex

    m, inputs = _few_rows_encoder(12, 7)
    ids, pos, off, longest = inputs([40, 24])
    to = torch.arange(2, device=DEV)
    want = m.encode_packed(ids, pos, off, longest)
    index = IVFIndex(384, 2, device=DEV)
    index.train(want.repeat(4, 1))

    def given_up():
        out = torch.zeros(2, 384, device=DEV)
        with ops.tuning(encoder_tries=0):
            assert m._encode_native(ids, pos, off, longest, True, out, to)
            torch.cuda.synchronize()
        assert out.isnan().any()
        return out
    for ask in (lambda: m.encode_packed(ids, pos, off, longest, out=torch.empty(2, 384, device=DEV), to=to), lambda: ops.check_lost(DEV)):
        given_up()
        with pytest.raises(RuntimeError, match="gave up"):
            ask()
    bad = given_up()
    with pytest.raises(RuntimeError, match="gave up"):
        index.add(bad)
    assert index.ntotal == 0
    ops.check_lost(DEV)
    out = torch.zeros(2, 384, device=DEV)
    assert m._encode_native(ids, pos, off, longest, True, out, to) and torch.equal(out, want)
