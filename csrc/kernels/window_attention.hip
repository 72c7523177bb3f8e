// Grouped-query attention over a paged K/V cache with a sliding window and kept first tokens, for gfx950:
// query i sees key j <= i with i - j < size or j < keep; scores are (q . k) * scale, optionally softcapped
// (cap * tanh(s / cap)); query / key width D and value width V need not be equal.
//
// Cache: pool [pages][G heads][64 tokens][D + V] (a key row and its value row are one run; the keys of a head
// on a page are one contiguous block), page table [rows][max_pages] int32 (page 0 is never given to a
// request). Only the pages that hold kept or windowed keys are read, whatever the length of the context.
//
//   window_prep     q / k norm over the whole projection, rotation (halves), cache append
//   window_decode   few query tokens per request: (token, key head, partition of its visible tiles), then
//                   partition_merge
//   window_prefill  longer portions: flash attention straight from the pages (a 64-key tile is one page)
//   window_any      any size and fp32: one workgroup per (token, head)
#include "rt_paged.h"

#include <algorithm>

namespace rt {
namespace wa {

using namespace paged;

// ---------------------------------------------------------------------------------------------
// prep
// ---------------------------------------------------------------------------------------------
struct PrepArgs {
  void* proj; long ldp;        // [T, ldp]: q at q_col, k at k_col, v at v_col
  int q_col, k_col, v_col;
  const void* q_norm; const void* k_norm;             // [H * D], [G * D] (null: no norm)
  float eps;
  const float* cosT; const float* sinT; int max_pos;  // [max_pos, half]
  int half;                    // dimension i < half turns with i + half
  const int* row; const int* pos;
  void* pool; const int* tab; int max_pages, n_pages, n_rows;
  int H, G, D, V;
};

template <typename T, int N>
__device__ __forceinline__ void ldn(const T* p, float* o) {
  if constexpr (N == 8) unpack8(*(const uint4*)p, o);
  else o[0] = ld(p);
}
template <typename T, int N>
__device__ __forceinline__ void stn(T* p, const float* o) {
  if constexpr (N == 8) *(uint4*)p = pack8(o);
  else st(p, o[0]);
}

// N consecutive elements per access: 8 (bf16, D, V and half multiples of 8, aligned rows) or 1
template <typename T, int N>
__global__ __launch_bounds__(256) void window_prep_kernel(PrepArgs a) {
  __shared__ float sbuf[8];
  const int t = blockIdx.x, tid = threadIdx.x;
  T* pr = (T*)a.proj + (long)t * a.ldp;
  const int p_raw = a.pos[t], pos = min(max(p_raw, 0), a.max_pos - 1);
  const float* cs = a.cosT + (long)pos * a.half;
  const float* sn = a.sinT + (long)pos * a.half;
  const int row = a.row[t], pg = pos / PAGE;
  const bool ok = row >= 0 && row < a.n_rows && pg < a.max_pages;
  const int page = ok ? a.tab[(long)row * a.max_pages + pg] : -1;
  const bool append = page >= 0 && page < a.n_pages;
  T* dst = (T*)a.pool + ((long)max(page, 0) * a.G * PAGE + pos % PAGE) * (a.D + a.V);  // + head * PAGE * (D + V)
  const long hs = (long)PAGE * (a.D + a.V);

  auto squares = [&](const T* x, int n) {
    float s = 0.f, v[N];
    for (int e = tid * N; e < n; e += 256 * N) {
      ldn<T, N>(x + e, v);
#pragma unroll
      for (int k = 0; k < N; ++k) s += v[k] * v[k];
    }
    return s;
  };
  // one thread normalises and turns both halves of its pairs, so rows may be written in place
  auto turn = [&](T* x, const T* w, int heads, float rstd, bool to_cache) {
    for (int e = tid * N; e < heads * a.D; e += 256 * N) {
      const int h = e / a.D, i = e % a.D;
      if (i >= a.half && i < 2 * a.half) continue;
      T* o = to_cache ? dst + h * hs : x + h * a.D;
      float u[N], wu[N];
      ldn<T, N>(x + e, u);
      if (w) {
        ldn<T, N>(w + e, wu);
#pragma unroll
        for (int k = 0; k < N; ++k) u[k] *= rstd * wu[k];
      }
      if (i < a.half) {
        float v[N], r[N];
        ldn<T, N>(x + e + a.half, v);
        if (w) {
          ldn<T, N>(w + e + a.half, wu);
#pragma unroll
          for (int k = 0; k < N; ++k) v[k] *= rstd * wu[k];
        }
#pragma unroll
        for (int k = 0; k < N; ++k) {
          const float c = cs[i + k], s = sn[i + k];
          r[k] = v[k] * c + u[k] * s;
          u[k] = u[k] * c - v[k] * s;
        }
        if (!to_cache || append) stn<T, N>(o + i + a.half, r);
      }
      if (!to_cache || append) stn<T, N>(o + i, u);
    }
  };
  T* q = pr + a.q_col;
  T* k = pr + a.k_col;
  float rq = 1.f, rk = 1.f;
  if (a.q_norm || a.k_norm) {
    float sq = squares(q, a.H * a.D), sk = squares(k, a.G * a.D);
    sq = wave_sum(sq);
    sk = wave_sum(sk);
    if ((tid & 63) == 0) {
      sbuf[tid >> 6] = sq;
      sbuf[4 + (tid >> 6)] = sk;
    }
    __syncthreads();
    if (a.q_norm) rq = 1.f / sqrtf((sbuf[0] + sbuf[1] + sbuf[2] + sbuf[3]) / (a.H * a.D) + a.eps);
    if (a.k_norm) rk = 1.f / sqrtf((sbuf[4] + sbuf[5] + sbuf[6] + sbuf[7]) / (a.G * a.D) + a.eps);
  }
  turn(q, (const T*)a.q_norm, a.H, rq, false);
  turn(k, (const T*)a.k_norm, a.G, rk, true);
  if (append) {
    const T* v = pr + a.v_col;
    for (int e = tid * N; e < a.G * a.V; e += 256 * N) {
      T* o = dst + e / a.V * hs + a.D + e % a.V;
      if constexpr (N == 8) *(uint4*)o = *(const uint4*)(v + e);
      else *o = v[e];
    }
  }
}

// window_prep_kernel with everything of a token in registers: bf16, 16-byte aligned, at most 256 QJ leads of q, 256 of k and 256
// chunks of v. A lead is a chunk of 8 that turns with its partner or, beyond the rotated part, a chunk alone; a thread takes the
// loads of its leads and their weights at once, beside the token's row and position, then the tables and the page beside the
// squares: three trips to memory where each loop of the other asked for one thing after the other, twice for the rows (32 heads
// of 128, 8 key heads: 1 / 64 / 7854 tokens 6.1 / 6.8 / 61.8 -> 3.9 / 4.4 / 42.7 us, the last at 4.4 TB/s).
template <int QJ>
__global__ __launch_bounds__(256) void window_prep_once_kernel(PrepArgs a) {
  __shared__ float sbuf[8];
  const int t = blockIdx.x, tid = threadIdx.x;
  const int p_raw = a.pos[t], row = a.row[t];
  bf16_t* const pr = (bf16_t*)a.proj + (long)t * a.ldp;
  const int hp = a.half / 8, nl = (a.D - a.half) / 8;  // of a head: pairs, leads
  struct Lead {
    uint4 x, y, wx, wy;  // the lead and its partner, their weights
    int h, i;
    bool on, pair;
  };
  auto fetch = [&](Lead& l, int e, int heads, const bf16_t* x, const void* w) {
    l.on = e < heads * nl;
    const int at = min(e, heads * nl - 1), c = at % nl;
    l.h = at / nl;
    l.pair = c < hp;
    l.i = l.pair ? 8 * c : 8 * (c + hp);
    const int o = l.h * a.D + l.i, y = o + (l.pair ? a.half : 0);
    const bf16_t* wt = w ? (const bf16_t*)w : x;  // not given: unused
    l.x = *(const uint4*)(x + o);
    l.y = *(const uint4*)(x + y);
    l.wx = *(const uint4*)(wt + o);
    l.wy = *(const uint4*)(wt + y);
  };
  Lead q[QJ], k;
#pragma unroll
  for (int j = 0; j < QJ; ++j) fetch(q[j], tid + 256 * j, a.H, pr + a.q_col, a.q_norm);
  fetch(k, tid, a.G, pr + a.k_col, a.k_norm);
  const int nv = a.G * a.V / 8, ve = min(tid, nv - 1) * 8;
  const uint4 v = *(const uint4*)(pr + a.v_col + ve);
  const int pos = min(max(p_raw, 0), a.max_pos - 1), pg = pos / PAGE;
  const bool ok = row >= 0 && row < a.n_rows && pg < a.max_pages;
  const int page = a.tab[ok ? (long)row * a.max_pages + pg : 0];
  const float* cs = a.cosT + (long)pos * a.half;
  const float* sn = a.sinT + (long)pos * a.half;
  struct Turn { float4 c[2], s[2]; };
  auto tables = [&](const Lead& l) {
    const int i = l.pair ? l.i : 0;
    return Turn{{*(const float4*)(cs + i), *(const float4*)(cs + i + 4)}, {*(const float4*)(sn + i), *(const float4*)(sn + i + 4)}};
  };
  Turn tq[QJ];
#pragma unroll
  for (int j = 0; j < QJ; ++j) tq[j] = tables(q[j]);
  const Turn tk = tables(k);

  auto squares = [&](const Lead& l) {
    float s = 0.f, x[8], y[8];
    unpack8(l.x, x);
    unpack8(l.y, y);
#pragma unroll
    for (int e = 0; e < 8; ++e) s += x[e] * x[e] + (l.pair ? y[e] * y[e] : 0.f);
    return l.on ? s : 0.f;
  };
  float rq = 1.f, rk = 1.f;
  if (a.q_norm || a.k_norm) {
    float sq = 0.f, sk = squares(k);
#pragma unroll
    for (int j = 0; j < QJ; ++j) sq += squares(q[j]);
    sq = wave_sum(sq);
    sk = wave_sum(sk);
    if ((tid & 63) == 0) {
      sbuf[tid >> 6] = sq;
      sbuf[4 + (tid >> 6)] = sk;
    }
    __syncthreads();
    if (a.q_norm) rq = 1.f / sqrtf((sbuf[0] + sbuf[1] + sbuf[2] + sbuf[3]) / (a.H * a.D) + a.eps);
    if (a.k_norm) rk = 1.f / sqrtf((sbuf[4] + sbuf[5] + sbuf[6] + sbuf[7]) / (a.G * a.D) + a.eps);
  }
  auto turn = [&](const Lead& l, const Turn& c, bool normed, float rstd, bf16_t* o) {
    float u[8], w[8], x[8], wx[8];
    unpack8(l.x, u);
    unpack8(l.y, x);
    if (normed) {
      unpack8(l.wx, w);
      unpack8(l.wy, wx);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        u[e] *= rstd * w[e];
        x[e] *= rstd * wx[e];
      }
    }
    if (l.pair) {
      const float cc[8] = {c.c[0].x, c.c[0].y, c.c[0].z, c.c[0].w, c.c[1].x, c.c[1].y, c.c[1].z, c.c[1].w};
      const float ss[8] = {c.s[0].x, c.s[0].y, c.s[0].z, c.s[0].w, c.s[1].x, c.s[1].y, c.s[1].z, c.s[1].w};
      float r[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        r[e] = x[e] * cc[e] + u[e] * ss[e];
        u[e] = u[e] * cc[e] - x[e] * ss[e];
      }
      *(uint4*)(o + l.i + a.half) = pack8(r);
    }
    *(uint4*)(o + l.i) = pack8(u);
  };
#pragma unroll
  for (int j = 0; j < QJ; ++j)
    if (q[j].on) turn(q[j], tq[j], a.q_norm, rq, pr + a.q_col + q[j].h * a.D);
  if (ok && page >= 0 && page < a.n_pages) {
    bf16_t* dst = (bf16_t*)a.pool + ((long)page * a.G * PAGE + pos % PAGE) * (a.D + a.V);  // + head * PAGE * (D + V)
    const long hs = (long)PAGE * (a.D + a.V);
    if (k.on) turn(k, tk, a.k_norm, rk, dst + k.h * hs);
    if (tid < nv) *(uint4*)(dst + ve / a.V * hs + a.D + ve % a.V) = v;
  }
}

// what a query at a position sees: [0, kept) and [lo, pos], and the tile lists that cover them
struct Mask {
  int size, keep;  // size: INT_MAX without a window
  __device__ __forceinline__ bool sees(int q, int k) const { return k <= q && (q - k < size || k < keep); }
  __device__ __forceinline__ int lo(int q) const { return q < size ? 0 : q - size + 1; }
};
template <int TILE>
struct Tiles {
  int kept, w0, n;  // tiles over kept keys before the window's first tile, that tile's key, all tiles
  // queries q0 .. q1
  __device__ __forceinline__ Tiles(const Mask& m, int q0, int q1) {
    w0 = m.lo(q0) / TILE * TILE;
    kept = (min(m.keep, w0) + TILE - 1) / TILE;
    n = kept + (q1 - w0) / TILE + 1;
  }
  __device__ __forceinline__ int key(int i) const { return i < kept ? i * TILE : w0 + (i - kept) * TILE; }
};

// score in log2 units: x = q . k
struct Score {
  float mul, cap2;  // without a cap: x * mul; with one: cap2 * tanh(x * scale / cap), mul = 2 log2(e) scale / cap
  __device__ __forceinline__ float operator()(float x) const {
    const float y = x * mul;
    return cap2 > 0.f ? cap2 - 2.f * cap2 * __builtin_amdgcn_rcpf(1.f + fexp2(y)) : y;
  }
};
static Score make_score(float scale, float cap) {
  const float l2e = 1.4426950408889634f;
  return cap > 0.f ? Score{2.f * l2e * scale / cap, cap * l2e} : Score{scale * l2e, 0.f};
}
// Where |x scale / cap| is at most 0.4 for all of a wave's tile, the capped score is t (c0 + c1 t^2 + ..) cap2: minimax over that
// interval, 2.1e-8 from tanh there, where cap2 - 2 cap2 rcp(1 + 2^y) in fp32 is up to 1e-7 off. (2^(s - constant) without a row's
// maximum, which a cap allows, rounds its heaviest probability to bf16, where 2^0 is exact: errors 1.14 to 1.34 times as large.)
constexpr float TANH_T = 0.4f;
struct CapScore {
  float t, c0, c1, c2, c3;  // t = scale / cap, of either sign; c's times cap2
  __device__ __forceinline__ float near(float x) const {
    const float y = x * t, z = y * y;
    return y * fmaf(fmaf(fmaf(c3, z, c2), z, c1), z, c0);
  }
};
static CapScore make_cap_score(float scale, float cap) {
  const double c2 = (double)cap * 1.4426950408889634;
  return {scale / cap, (float)(0.99999957 * c2), (float)(-0.33329726 * c2), (float)(0.13250565 * c2), (float)(-0.04682564 * c2)};
}

// ---------------------------------------------------------------------------------------------
// decode: workgroup = (token, key head with its 16 NH query heads at most, partition), 4 waves
// ---------------------------------------------------------------------------------------------
// The waves take the partition's 16-key tiles in turn, each for itself until the end: an LDS image of its own
// [K: 64 QS columns | V: 64 RT columns] by LDS-DMA, two of them, no barrier. S^T = K Q^T (key on the MFMA row, head on
// the lane), online softmax of 4 scores a lane, O^T += V^T P^T with 16-key MFMAs (P is their B operand as it is);
// the waves' (m, l, O) meet in LDS. With a tile of 32 keys shared by the four waves every wave ran the same softmax
// (H / G of 16 lanes of it needed: 38 of 46 us were its VALU work), with three barriers a tile; and a page's number, loaded
// for each tile, waited for all LDS-DMA under way (loads return in order): the pages of 64 tiles now come at once.
// us, 4 query heads a key head, 128 + 128 columns, before -> this (each at its partitions): 64 rows of 300..1100 keys 50.2 -> 43.5 and no merge, 16 22.6 -> 15.5, 4 of 3000..4000 30 -> 17,
// 200 of 100..600 81.5 -> 70.8, 256 of 60..120 38.8 -> 34.1. 2 or 1 waves a workgroup, more of these on a CU: 44.9 / 52.5, 74.0 / 76.0, 32.6 / 33.3.
// 16 heads of 256 + 256 columns, where every wave reads all of q for itself, are the form's worst: 1 row of 300 keys 9.9 -> 10.3, of
// 4000 keys 17.8 -> 18.2, but 64 of 300..1100 33.9 -> 30.2 and 200 of 100..600 54 -> 41.
// A token's visible tiles are cut in NP equal partitions, so a captured launch with a fixed NP balances every
// length; of one partition the workgroup writes the result. Chunk c of image row r lies in slot c ^ r, or rows are an odd number of 16-B chunks (conflict-free either way).
struct DecArgs {
  const bf16_t* q; long ldq;  // [T, ldq], head h at h * D
  const bf16_t* pool; const int* tab; int max_pages, n_pages, n_rows;
  const int* row; const int* pos;
  float* part; float* ml;     // [T, H, NP, V], [T, H, NP, 2] (max in log2 units, sum)
  bf16_t* out; long ldo; float out_scale;  // of one partition: the result itself, as partition_merge makes it (else null)
  int H, G, D, V, NP, S;      // S: workgroups that share a key head's query heads
  Mask mask;
  Score score;
};

template <int QS, int RT, int NH>
__global__ __launch_bounds__(256, 2) void window_decode_kernel(DecArgs a) {
  constexpr int NW = 4;
  constexpr int CH = 8 * QS + 8 * RT;
  constexpr bool SWZ = CH % 16 == 0;
  constexpr int CPR = SWZ ? CH : CH + 1, ROWB = CPR * 16;
  constexpr int NIT = (16 * CPR + 63) / 64, BUFB = NIT * 1024;  // LDS-DMA instructions of a tile (the last one may be part used)
  constexpr int QF = 2 * QS, LDP = 64 * RT + 4;
  constexpr int RING = NW * 2 * BUFB;                 // two images a wave; at the end 16 heads' O in their place
  static_assert(16 * LDP * 4 <= 2 * BUFB, "a wave's sums fit its images");
  __shared__ __attribute__((aligned(16))) char smem[RING + NW * NH * 16 * 8];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const int bid = xcd_remap(blockIdx.x, gridDim.x);
  const int sub = bid % a.S, part = bid / a.S % a.NP, gh = bid / (a.S * a.NP) % a.G, t = bid / (a.S * a.NP * a.G);
  const int h0 = gh * (a.H / a.G) + 16 * NH * sub, HG = min(a.H / a.G - 16 * NH * sub, 16 * NH);  // query heads h0 .. h0 + HG - 1
  int row = a.row[t], pos = a.pos[t];
  asm volatile("" : "+s"(row), "+s"(pos));           // in one trip, also if the partition is empty
  row = min(max(row, 0), a.n_rows - 1);
  pos = min(max(pos, 0), a.max_pages * PAGE - 1);
  const Tiles<16> tl(a.mask, pos, pos);
  const int per = (tl.n + a.NP - 1) / a.NP;
  const int i0 = part * per, i1 = min(tl.n, i0 + per);
  if (i0 >= i1) {  // nothing for this partition (uniform over the workgroup)
    for (int h = tid; h < HG; h += 64 * NW) {
      float* m = a.ml + (((long)t * a.H + h0 + h) * a.NP + part) * 2;
      m[0] = -INFINITY;
      m[1] = 0.f;
    }
    return;
  }
  const int n = i1 - i0 > w ? (i1 - i0 - w + NW - 1) / NW : 0;  // this wave's tiles: i0 + w + NW j
  auto key_of = [&](int j) { return tl.key(min(i0 + w + NW * j, i1 - 1)); };
  const int* tab = a.tab + (long)row * a.max_pages;
  int pages = tab[key_of(lane) / PAGE];              // of 64 tiles, a tile a lane
  // query fragments: lane holds Q[head r16][32 s + 8 g ..]; heads past the last repeat it (not stored)
  bf16x8 qf[NH][QF];
#pragma unroll
  for (int u = 0; u < NH; ++u) {
    const bf16_t* qp = a.q + (long)t * a.ldq + (long)(h0 + min(16 * u + r16, HG - 1)) * a.D;
#pragma unroll
    for (int s = 0; s < QF; ++s) qf[u][s] = *(const bf16x8*)(qp + min(32 * s + 8 * g, a.D - 8));
  }
  const int W = a.D + a.V;

  // LDS-DMA sources: instruction j covers image chunks 64 j + lane; columns past D (V)
  // repeat the last chunk (the query is zero there, the sums are not stored)
  uint32_t src[NIT];  // element offset from the tile's first cache row
#pragma unroll
  for (int j = 0; j < NIT; ++j) {
    const int c = 64 * j + lane, r = min(c / CPR, 15), cc = SWZ ? c % CPR ^ r : c % CPR;
    const int col = cc < 8 * QS ? min(8 * cc, a.D - 8) : a.D + min(8 * (cc - 8 * QS), a.V - 8);
    src[j] = (uint32_t)(r * W + col);
  }
  char* const mine = smem + w * 2 * BUFB;
  auto stage = [&](int j) {
    if (j % 64 == 0 && j > 0) {
      pages = tab[key_of(j + lane) / PAGE];
      asm volatile("" : "+v"(pages));                // waited for here, not by every tile
    }
    const int page = min(max(__builtin_amdgcn_readlane(pages, j % 64), 0), a.n_pages - 1);
    const bf16_t* base = a.pool + (((long)page * a.G + gh) * PAGE + key_of(j) % PAGE) * W;
    char* to = mine + (j & 1) * BUFB;
#pragma unroll
    for (int k = 0; k < NIT; ++k)
      __builtin_amdgcn_global_load_lds((const void*)(base + src[k]), (lds_void*)(to + k * 1024), 16, 0, 0);
  };

  f32x4 o[NH][4 * RT];
#pragma unroll
  for (int u = 0; u < NH; ++u)
#pragma unroll
    for (int c = 0; c < 4 * RT; ++c) o[u][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m[NH], l[NH];
#pragma unroll
  for (int u = 0; u < NH; ++u) { m[u] = -INFINITY; l[u] = 0.f; }
  if (a.D < 64 * QS) {
#pragma unroll
    for (int u = 0; u < NH; ++u)
#pragma unroll
      for (int s = 0; s < QF; ++s)
        if (32 * s + 8 * g >= a.D) qf[u][s] = bf16x8{};
  }
#pragma unroll
  for (int u = 0; u < NH; ++u)
#pragma unroll
    for (int s = 0; s < QF; ++s) asm volatile("" : "+v"(qf[u][s]));  // waited for ahead of the tiles
  asm volatile("" : "+v"(pages));
  auto slot = [](int r, int c) { return r * ROWB + (SWZ ? c ^ r : c) * 16; };
  const int vr = 4 * g + ((lane >> 2) & 3);          // this lane's part of the transposed reads
  if (n > 0) stage(0);
  if (n > 1) stage(1);
  for (int j = 0; j < n; ++j) {
    const int key0 = key_of(j);
    // this tile's image; the next tile's instructions stay in flight
    if (j + 1 < n) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(NIT) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const char* img = mine + (j & 1) * BUFB;
    f32x4 sp[NH][2];
#pragma unroll
    for (int u = 0; u < NH; ++u) sp[u][0] = sp[u][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < QF; ++s) {
      const bf16x8 kf = *(const bf16x8*)(img + slot(r16, 4 * s + g));
#pragma unroll
      for (int u = 0; u < NH; ++u) sp[u][s & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[u][s], sp[u][s & 1], 0, 0, 0);
    }
    const bool whole = key0 + 15 <= pos && (pos - key0 < a.mask.size || key0 + 15 < a.mask.keep);
    rt_s16x4 pa[NH];
#pragma unroll
    for (int u = 0; u < NH; ++u) {
      f32x4 x = sp[u][0] + sp[u][1];
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = a.score(x[e]);
      if (!whole) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (!a.mask.sees(pos, key0 + 4 * g + e)) x[e] = -INFINITY;
      }
      const float mx = over_groups(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), [](float p, float q) { return fmaxf(p, q); });
      const float mn = fmaxf(m[u], mx);  // finite: every listed tile holds a visible key
      const float alpha = fexp2(m[u] - mn);
      m[u] = mn;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = fexp2(x[e] - mn);
      l[u] = l[u] * alpha + over_groups((x[0] + x[1]) + (x[2] + x[3]), [](float p, float q) { return p + q; });
      pa[u] = __builtin_bit_cast(rt_s16x4, make_uint2(pack2bf(x[0], x[1]), pack2bf(x[2], x[3])));
      // O^T: the head is the lane's column, as in the scores (most tiles bring no new maximum)
      if (__any(alpha != 1.f)) {
#pragma unroll
        for (int c = 0; c < 4 * RT; ++c) o[u][c] *= alpha;
      }
    }
#pragma unroll
    for (int c0 = 0; c0 < 4 * RT; c0 += 8) {
      uint32_t va[8];
      rt_s16x4 v[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) va[c] = lds_addr(img + slot(vr, 8 * QS + 2 * (c0 + c) + ((lane >> 1) & 1)) + (lane & 1) * 8);
      ds_tr16_at8(va, v);
#pragma unroll
      for (int c = 0; c < 8; ++c)
#pragma unroll
        for (int u = 0; u < NH; ++u) o[u][c0 + c] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(v[c], pa[u], o[u][c0 + c], 0, 0, 0);
    }
    if (j + 2 < n) stage(j + 2);  // this image has been read
  }
  // ---- the waves' sums: o[u][c][e] is head h0 + 16 u + r16, value column 16 c + 4 g + e. A wave's go where its own images were,
  // so the waves meet once a head tile, and whoever adds them up weighs them ----
  float2* const mls = (float2*)(smem + RING);        // [wave][head]
  if (g == 0)
#pragma unroll
    for (int u = 0; u < NH; ++u) mls[w * 16 * NH + 16 * u + r16] = make_float2(m[u], l[u]);
  constexpr int OS = 2 * BUFB / 4;                   // floats from wave to wave
#pragma unroll
  for (int u = 0; u < NH; ++u) {
    if (u > 0) __syncthreads();
    if (16 * u + r16 < HG) {
#pragma unroll
      for (int c = 0; c < 4 * RT; ++c) *(f32x4*)((float*)mine + r16 * LDP + 16 * c + 4 * g) = o[u][c];
    }
    __syncthreads();
    const int hn = min(HG - 16 * u, 16), V4 = a.V / 4;  // V % 8 == 0
    for (int e = tid; e < hn * V4; e += 64 * NW) {
      const int h = e / V4, c = e % V4 * 4;
      const long th = (long)t * a.H + h0 + 16 * u + h;
      float2 ml[NW];
      f32x4 x[NW];
#pragma unroll
      for (int k = 0; k < NW; ++k) {
        ml[k] = mls[k * 16 * NH + 16 * u + h];
        x[k] = *(const f32x4*)((float*)smem + k * OS + h * LDP + c);
      }
      float M = ml[0].x, L = 0.f;                    // finite: wave 0 has a tile
#pragma unroll
      for (int k = 1; k < NW; ++k) M = fmaxf(M, ml[k].x);
      f32x4 y;
#pragma unroll
      for (int k = 0; k < NW; ++k) {
#pragma clang fp contract(off)
        const float f = fexp2(ml[k].x - M);          // 0 for a wave without tiles
        L = fmaf(ml[k].y, f, L);
        y = k == 0 ? x[0] * f : y + x[k] * f;
      }
      if (a.out) {
        y *= a.out_scale / L;
        *(uint2*)(a.out + (long)t * a.ldo + (long)(h0 + 16 * u + h) * a.V + c) = make_uint2(pack2bf(y[0], y[1]), pack2bf(y[2], y[3]));
      } else {
        *(f32x4*)(a.part + (th * a.NP + part) * a.V + c) = y;
        if (c == 0) *(float2*)(a.ml + (th * a.NP + part) * 2) = make_float2(M, L);
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// prefill: 128 query rows of one head per workgroup, 4 waves x 32 rows, 64-key tiles = pages
// ---------------------------------------------------------------------------------------------
// Swapped S^T = K Q^T, P straight into the next MFMA (O^T = V^T P^T), double-buffered K / V tiles by LDS-DMA
// straight from the pages, one barrier per tile. Bound by the VALU's work on the scores beside 64 MFMAs a tile: with a
// cap two exponentials and a reciprocal each. So most capped scores take a polynomial for tanh (CapScore); the pages of 64 tiles are read at once instead of a load that every tile waits for; values
// are read four column tiles to a wait instead of two. 2 requests of 3700 tokens, 32 heads of 128, cap 50: 407 -> 324 us
// (550 -> 690 TF/s), of which the order of the tiles 19; without a cap 386 -> 320.
struct PreArgs {
  const bf16_t* q; long ldq;     // [tokens, ldq], head h at h * D, normed and rotated
  const bf16_t* pool; const int* tab; int max_pages, n_pages, n_rows;
  bf16_t* o; long ldo;
  const Seg* segs; const int2* tiles; int n_tiles;   // {segment, first query row / 128}
  int H, G, D, V;
  Mask mask;
  Score score;
  CapScore near;
  float out_scale;
};

// CAP: scores under a cap, see CapScore
template <int DQ, int DV, bool CAP>
__global__ __launch_bounds__(256, 2) void window_prefill_kernel(PreArgs a) {
  constexpr int NQ = DQ / 8, NV = DV / 8, DS = DQ / 32, DT = DV / 16;
  constexpr int KB = 64 * DQ * 2, VB = 64 * DV * 2;
  constexpr int OROW = DV + 8;
  constexpr int TILES = 2 * (KB + VB), OB = 128 * OROW * 2;
  __shared__ __attribute__((aligned(16))) char smem[TILES > OB ? TILES : OB];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const int lin = xcd_remap(blockIdx.x, gridDim.x);
  // the heaviest tiles (first in the list) of all the query heads of a key head, which share an XCD's L2, ahead of the lighter
  const int rep = a.H / a.G, gh = lin / (a.n_tiles * rep), in = lin % (a.n_tiles * rep), h = gh * rep + in % rep;
  const int2 tile = a.tiles[in / rep];
  const Seg sg = a.segs[tile.x];
  const int qblk0 = tile.y * 128, q0 = qblk0 + wid * 32;
  const int pa0 = sg.pos0 + qblk0, pa1 = sg.pos0 + min(qblk0 + 128, sg.q_len) - 1;  // positions of the workgroup
  const Tiles<64> tl(a.mask, pa0, pa1);
  const int* tab = a.tab + (long)min(max(sg.row, 0), a.n_rows - 1) * a.max_pages;
  const int W = a.D + a.V;

  bf16x8 qf[2][DS];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int qr = min(q0 + 16 * u + r16, sg.q_len - 1);
    const bf16_t* qp = a.q + (long)(sg.q_off + qr) * a.ldq + (long)h * a.D;
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      const int c = 32 * s + 8 * g;
      qf[u][s] = c < a.D ? *(const bf16x8*)(qp + c) : bf16x8{};
    }
  }
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int s = 0; s < DS; ++s) asm volatile("" : "+v"(qf[u][s]));

  f32x4 o[2][DT];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int c = 0; c < DT; ++c) o[u][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m[2], l[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) { m[u] = -INFINITY; l[u] = 0.f; }

  // LDS-DMA of one tile: instruction j of this wave fills 1 KiB of the K (V) image; the lane's source chunk
  // undoes the image's swizzle. Columns past D (V) repeat the first chunk (the query is zero there, the
  // values are not stored); slots of the page past the request's keys are finite and masked.
  constexpr int JK = KB / 4096, JV = VB / 4096;
  uint32_t off[JK + JV];
#pragma unroll
  for (int j = 0; j < JK + JV; ++j) {
    const bool v = j >= JK;
    const int e = (4 * (v ? j - JK : j) + wid) * 64 + lane;
    const int key = v ? e / NV : e / NQ;
    const int c = 8 * (v ? vv_chunk<DV>(key, e % NV) : kq_chunk<DQ>(key, e % NQ));
    off[j] = 2 * (uint32_t)(key * W + (v ? a.D + (c < a.V ? c : 0) : (c < a.D ? c : 0)));
  }
  // pages of 64 tiles, one a lane: a load per tile would stand behind the tile's own wait with its latency
  auto pages_from = [&](int i) {
    const int p = tl.key(min(i + lane, tl.n - 1)) / PAGE;
    return min(max(tab[min(p, a.max_pages - 1)], 0), a.n_pages - 1);
  };
  int pages = pages_from(0);
  auto stage = [&](int page, int buf) {
    char* kd = smem + buf * (KB + VB);
    const bf16_t* base = a.pool + ((long)page * a.G + gh) * PAGE * W;
#pragma unroll
    for (int j = 0; j < JK + JV; ++j)
      lds_dma16(base, off[j], kd + (j < JK ? 4 * j : KB / 1024 + 4 * (j - JK)) * 1024 + wid * 1024);
  };
  stage(__builtin_amdgcn_readlane(pages, 0), 0);
  int cur = 0;
  for (int i = 0; i < tl.n; ++i, cur ^= 1) {
    const int kv0 = tl.key(i);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this tile (issued one tile ago)
    asm volatile("s_barrier" ::: "memory");           // ... of every wave; the other buffer is free
    if (i + 1 < tl.n) {
      if (((i + 1) & 63) == 0) pages = pages_from(i + 1);
      stage(__builtin_amdgcn_readlane(pages, (i + 1) & 63), cur ^ 1);
    }
    char* Ks = smem + cur * (KB + VB);
    char* Vs = Ks + KB;
    f32x4 stt[4][2];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) stt[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int s = 0; s < DS; ++s) {
        const bf16x8 kf = *(const bf16x8*)(Ks + kq_off<DQ>(16 * t + r16, 4 * s + g));
#pragma unroll
        for (int u = 0; u < 2; ++u)
          stt[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[u][s], stt[t][u], 0, 0, 0);
      }
    bool close = false;
    if constexpr (CAP) {
      float mx = 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e) mx = fmaxf(mx, fabsf(stt[t][u][e]));
      close = !__any(mx * fabsf(a.near.t) > TANH_T);
    }
    if (close) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e) stt[t][u][e] = a.near.near(stt[t][u][e]);
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e) stt[t][u][e] = a.score(stt[t][u][e]);
    }
    const int w0 = sg.pos0 + q0, w1 = w0 + 31;  // positions of the wave's rows
    if (!(kv0 + 63 <= w0 && (w1 - kv0 < a.mask.size || kv0 + 63 < a.mask.keep))) {  // not all visible
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (!a.mask.sees(w0 + 16 * u + r16, kv0 + 16 * t + 4 * g + e)) stt[t][u][e] = -INFINITY;
    }
    float alpha[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float mx = -INFINITY;
#pragma unroll
      for (int t = 0; t < 4; ++t)
        mx = fmaxf(mx, fmaxf(fmaxf(stt[t][u][0], stt[t][u][1]), fmaxf(stt[t][u][2], stt[t][u][3])));
      const float mn = fmaxf(m[u], over_groups(mx, [](float x, float y) { return fmaxf(x, y); }));
      const float mz = mn == -INFINITY ? 0.f : mn;  // a row may see nothing of its first tiles
      alpha[u] = fexp2(m[u] - mz);
      m[u] = mn;
      float rs = 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float p = fexp2(stt[t][u][e] - mz);
          stt[t][u][e] = p;
          rs += p;
        }
      l[u] = l[u] * alpha[u] + over_groups(rs, [](float x, float y) { return x + y; });
    }
    // O^T: the query is the lane's column, as in the scores (most tiles bring no new maximum)
    if (__any(alpha[0] != 1.f || alpha[1] != 1.f)) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int c = 0; c < DT; ++c) o[u][c] *= alpha[u];
    }
    bf16x8 pa[2][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int u = 0; u < 2; ++u) pa[ks][u] = pack_p(stt[2 * ks][u], stt[2 * ks + 1][u]);
    // transposed reads of four column tiles at a time: rows 16 apart have the same swizzle
    const int key_a = 4 * g + (lane >> 2 & 3), pcol = lane & 3;
#pragma unroll
    for (int c = 0; c < DT; c += 4) {
      uint32_t va[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) va[k] = lds_addr(Vs + vv_off<DV>(key_a, 2 * (c + k) + (pcol >> 1)) + ((pcol & 1) << 3));
      rt_s16x4 v[16];
      ds_tr16_frag4<16 * DV * 2, 32 * DV * 2, 48 * DV * 2>(va[0], va[1], va[2], va[3], v);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const bf16x8 vf = cat4(v[4 * k + 2 * ks], v[4 * k + 2 * ks + 1]);
#pragma unroll
          for (int u = 0; u < 2; ++u) o[u][c + k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pa[ks][u], o[u][c + k], 0, 0, 0);
        }
    }
  }
  __syncthreads();  // the last tile's images become the O staging area
  bf16_t* Os = (bf16_t*)smem;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const float sc = a.out_scale / l[u];  // a position sees itself
    const int r = wid * 32 + 16 * u + r16;
#pragma unroll
    for (int c = 0; c < DT; ++c)
      *(uint2*)(Os + r * OROW + 16 * c + 4 * g) =
          make_uint2(pack2bf(o[u][c][0] * sc, o[u][c][1] * sc), pack2bf(o[u][c][2] * sc, o[u][c][3] * sc));
  }
  __syncthreads();
  for (int e = tid; e < 128 * NV; e += 256) {
    const int r = e / NV, c = (e % NV) * 8;
    if (qblk0 + r < sg.q_len && c < a.V)
      *(uint4*)(a.o + (long)(sg.q_off + qblk0 + r) * a.ldo + (long)h * a.V + c) = *(const uint4*)(Os + r * OROW + c);
  }
}

// ---------------------------------------------------------------------------------------------
// any size and type: one workgroup per (head, token), 256 of its visible keys at a time
// ---------------------------------------------------------------------------------------------
struct AnyArgs {
  const void* q; long ldq;
  const void* pool; const int* tab; int max_pages, n_pages, n_rows;
  const int* row; const int* pos;
  void* o; long ldo;
  int H, G, D, V;
  Mask mask;
  float scale, cap, out_scale;
};

template <typename T>
__global__ __launch_bounds__(256) void window_any_kernel(AnyArgs a) {
  extern __shared__ float sm[];  // q [D], acc [V], p [256], key row offsets [256], sbuf [4]
  float* qs = sm;
  float* acc = qs + a.D;
  float* ps = acc + a.V;
  int* ks = (int*)(ps + 256);
  float* sbuf = (float*)(ks + 256);
  const int h = blockIdx.x, t = blockIdx.y, tid = threadIdx.x, gh = h / (a.H / a.G), W = a.D + a.V;
  const int row = min(max(a.row[t], 0), a.n_rows - 1);
  const int pos = min(max(a.pos[t], 0), a.max_pages * PAGE - 1);
  const int lo = a.mask.lo(pos), kept = min(a.mask.keep, lo), n = kept + pos - lo + 1;
  const int* tab = a.tab + (long)row * a.max_pages;
  for (int c = tid; c < a.D; c += 256) qs[c] = ld((const T*)a.q + (long)t * a.ldq + (long)h * a.D + c);
  for (int c = tid; c < a.V; c += 256) acc[c] = 0.f;
  float m = -INFINITY, l = 0.f;
  __syncthreads();
  for (int j0 = 0; j0 < n; j0 += 256) {
    const int j = j0 + tid;
    float s = -INFINITY;
    if (j < n) {
      const int key = j < kept ? j : lo + j - kept;
      const int page = min(max(tab[key / PAGE], 0), a.n_pages - 1);
      const int at = (page * a.G + gh) * PAGE + key % PAGE;  // pages * G * 64 fits an int (launcher)
      ks[tid] = at;
      const T* kp = (const T*)a.pool + (long)at * W;
      float d = 0.f;
      for (int c = 0; c < a.D; ++c) d = fmaf(qs[c], ld(kp + c), d);
      s = d * a.scale;
      if (a.cap > 0.f) s = a.cap * tanhf(s / a.cap);
    }
    const float mn = fmaxf(m, block_max(s, sbuf));
    const float alpha = expf(m - mn);
    const float p = j < n ? expf(s - mn) : 0.f;
    ps[tid] = p;
    l = l * alpha + block_sum(p, sbuf);
    m = mn;
    __syncthreads();
    const int cnt = min(256, n - j0);
    for (int c = tid; c < a.V; c += 256) {
      float y = acc[c] * alpha;
      for (int k = 0; k < cnt; ++k) y = fmaf(ps[k], ld((const T*)a.pool + (long)ks[k] * W + a.D + c), y);
      acc[c] = y;
    }
    __syncthreads();
  }
  for (int c = tid; c < a.V; c += 256) st((T*)a.o + (long)t * a.ldo + (long)h * a.V + c, acc[c] / l * a.out_scale);
}

static Mask make_mask(int size, int keep) { return Mask{size > 0 ? size : 0x7fffffff, std::max(keep, 0)}; }

}  // namespace wa
}  // namespace rt

using namespace rt;
using namespace rt::wa;

extern "C" int rt_window_prep(int f32, void* proj, long ldp, int q_col, int k_col, int v_col, const void* q_norm,
                              const void* k_norm, float eps, const float* cosT, const float* sinT, int max_pos, int half,
                              const int* row, const int* pos, void* pool, const int* tab, int max_pages, int n_pages,
                              int n_rows, int T, int H, int G, int D, int V, hipStream_t stream) {
  if (T <= 0) return 0;
  if (2 * half > D || max_pos < 1) return -1;
  PrepArgs a{proj, ldp, q_col, k_col, v_col, q_norm, k_norm, eps, cosT, sinT, max_pos, half, row, pos,
             pool, tab, max_pages, n_pages, n_rows, H, G, D, V};
  const bool vec = !f32 && D % 8 == 0 && V % 8 == 0 && half % 8 == 0 && ldp % 8 == 0 && q_col % 8 == 0 && k_col % 8 == 0 &&
                   v_col % 8 == 0 && ((uintptr_t)proj | (uintptr_t)pool | (uintptr_t)q_norm | (uintptr_t)k_norm) % 16 == 0;
  const long leads = (long)H * ((D - half) / 8), k_leads = (long)G * ((D - half) / 8);  // a lead or two a thread; tables in 16-byte loads
  // Where tokens fill the chip several times over a workgroup's idle threads count, and a token of few heads leaves most idle. us,
  // loops / registers: 4 heads and 2 key heads of 64, 700 / 2000 / 8000 tokens 5.7 / 7.4 / 17.4 and 5.2 / 8.5 / 24.0, without norms 4.3 /
  // 5.6 / 11.6 and 4.3 / 6.9 / 19.4; 16 and 4 of 128 (224 items), 8000 tokens 27.9 and 26.9, without norms, where the loops read a
  // row once, 19.9 and 21.5; 20 and 4 (256) 22.9 and 23.2, 24 and 8 37.7 and 33.5
  const bool fills = T <= 768 || leads + k_leads + (long)G * V / 8 >= (q_norm || k_norm ? 224 : 256);
  const bool once = half >= 8 && G > 0 && leads <= 512 && k_leads <= 256 && (long)G * V <= 2048 && n_rows > 0 && max_pages > 0 &&
                    ((uintptr_t)cosT | (uintptr_t)sinT) % 16 == 0 && fills;
  if (f32) hipLaunchKernelGGL((window_prep_kernel<float, 1>), dim3(T), dim3(256), 0, stream, a);
  else if (vec && once) {
    if (leads <= 256) hipLaunchKernelGGL(window_prep_once_kernel<1>, dim3(T), dim3(256), 0, stream, a);
    else hipLaunchKernelGGL(window_prep_once_kernel<2>, dim3(T), dim3(256), 0, stream, a);
  } else if (vec) hipLaunchKernelGGL((window_prep_kernel<bf16_t, 8>), dim3(T), dim3(256), 0, stream, a);
  else hipLaunchKernelGGL((window_prep_kernel<bf16_t, 1>), dim3(T), dim3(256), 0, stream, a);
  RT_LAUNCH_CHECK();
  return 0;
}

extern "C" int rt_window_decode_ok(int H, int G, int D, int V) {
  return G > 0 && H % G == 0 && H / G <= 32 && D % 8 == 0 && V % 8 == 0 && D >= 8 && V >= 8 && D <= 256 && V <= 256;
}

// Workgroups that share the query heads of a key head: one, but one per 16 heads where there are more and more than 128 value
// columns. With two tiles of heads over 256 columns a wave's sums take 256 registers, and the four waves' merge was the longer
// part of a short row: us, a workgroup of 32 heads -> two of 16, 128 + 256 columns, 1 row of 300 keys 12.9 -> 10.1, 16 of 300..1100 17.8 ->
// 14.5, 200 of 100..600 43.2 -> 31.1 (of 4 key heads of 64 + 256, where keys and values are the time, 68 -> 76; before the waves
// had tiles of their own 89)
static int head_groups(int H, int G, int V) { return V > 128 ? (H / G + 15) / 16 : 1; }

// Partitions of a token's tiles that a decode takes of the NP it may: a workgroup per CU. us (without the merge), 8 key heads of
// 128, at 1 / 2 / 4 / 8 partitions: 4 rows of 3000..4000 keys 45 / 27 / 19 / 17, 16 of 300..1100 18.8 / 15.5 / 15.6 / 17.6, 32 24.5 / 26.1 /
// 25.3 / 29.1, 64 43.5 / 44.2 / 44.0 / 50.0, 128 of 100..600 47.2 / 47.8 / 52.6 / 69.3, 256 of 60..120 34 / 42 / 63 / 106; and one needs
// no merge (5 us). The lengths are not known here, only the longest that the cache may hold, which is mostly far beyond them. A
// long row among many short ones is then the time of one workgroup's tiles: 32 rows, one of 4000 keys and 31 of 50..150 41.9 at one
// partition (the tiles of 32 keys shared by the waves took 47.1 with the merge, at four); 64 rows, one of 8000, 83 (93); 16 rows, one
// of 4000, at two partitions 28 (47).
extern "C" int rt_window_decode_parts(int T, int H, int G, int V, int NP) {
  const long groups = std::max(1L, (long)T * G * head_groups(H, G, V)), cus = num_cus();
  return (int)std::min((long)NP, (cus + groups - 1) / groups);
}

// NP of one partition: to out (ldo % 4 == 0, 8-byte aligned), part and ml unused; of more: to part and ml, for partition_merge
extern "C" int rt_window_decode(const void* q, long ldq, const void* pool, const int* tab, int max_pages, int n_pages,
                                int n_rows, const int* row, const int* pos, float* part, float* ml, void* out, long ldo,
                                float out_scale, int T, int H, int G, int D, int V, int NP, int size, int keep, float scale,
                                float cap, hipStream_t stream) {
  if (T <= 0) return 0;
  if (!rt_window_decode_ok(H, G, D, V) || NP < 1 || ldq % 8) return -1;
  if (NP == 1 && (ldo % 4 || (uintptr_t)out % 8)) return -1;
  DecArgs a{(const bf16_t*)q, ldq, (const bf16_t*)pool, tab, max_pages, n_pages, n_rows, row, pos, part, ml,
            NP == 1 ? (bf16_t*)out : nullptr, ldo, out_scale, H, G, D, V, NP, head_groups(H, G, V), make_mask(size, keep),
            make_score(scale, cap)};
  dim3 grid((unsigned)((long)T * G * NP * a.S)), block(256);
#define WD_(QS, RT, NH) hipLaunchKernelGGL((window_decode_kernel<QS, RT, NH>), grid, block, 0, stream, a)
#define WD_V(QS) do { if (V > 128) WD_(QS, 4, 1); else if (H / G > 16) WD_(QS, 2, 2); else WD_(QS, 2, 1); } while (0)
  if (D <= 64) WD_V(1);
  else if (D <= 128) WD_V(2);
  else if (D <= 192) WD_V(3);
  else WD_V(4);
#undef WD_V
#undef WD_
  RT_LAUNCH_CHECK();
  return 0;
}

extern "C" int rt_window_prefill_ok(int D, int V) { return D % 8 == 0 && V % 8 == 0 && D >= 8 && V >= 8 && D <= 256 && V <= 128; }

extern "C" int rt_window_prefill(const void* q, long ldq, const void* pool, const int* tab, int max_pages, int n_pages,
                                 int n_rows, void* o, long ldo, const void* segs, const void* tiles, int n_tiles, int H,
                                 int G, int D, int V, int size, int keep, float scale, float cap, float out_scale,
                                 hipStream_t stream) {
  if (n_tiles <= 0) return 0;
  if (!rt_window_prefill_ok(D, V) || G < 1 || H % G || ldq % 8 || ldo % 8 || (uintptr_t)o % 16) return -1;
  PreArgs a{(const bf16_t*)q, ldq, (const bf16_t*)pool, tab, max_pages, n_pages, n_rows, (bf16_t*)o, ldo, (const Seg*)segs,
            (const int2*)tiles, n_tiles, H, G, D, V, make_mask(size, keep), make_score(scale, cap), CapScore{}, out_scale};
  const bool capped = cap > 0.f;
  if (capped) a.near = make_cap_score(scale, cap);
  dim3 grid((unsigned)((long)n_tiles * H)), block(256);
#define WP_C(DQ, DV, C) hipLaunchKernelGGL((window_prefill_kernel<DQ, DV, C>), grid, block, 0, stream, a)
#define WP_(DQ)                                                          \
  do {                                                                   \
    if (V <= 64) { if (capped) WP_C(DQ, 64, true); else WP_C(DQ, 64, false); } \
    else { if (capped) WP_C(DQ, 128, true); else WP_C(DQ, 128, false); } \
  } while (0)
  if (D <= 64) WP_(64);
  else if (D <= 128) WP_(128);
  else if (D <= 192) WP_(192);
  else WP_(256);
#undef WP_
#undef WP_C
  RT_LAUNCH_CHECK();
  return 0;
}

extern "C" int rt_window_any(int f32, const void* q, long ldq, const void* pool, const int* tab, int max_pages, int n_pages,
                             int n_rows, const int* row, const int* pos, void* o, long ldo, int T, int H, int G, int D,
                             int V, int size, int keep, float scale, float cap, float out_scale, hipStream_t stream) {
  if (T <= 0) return 0;
  if (G < 1 || H % G || (long)n_pages * G * PAGE > 0x7fffffffL) return -1;
  const size_t lds = (size_t)(D + V + 512 + 4) * 4;
  if (lds > 65536) return -2;
  for (int t0 = 0; t0 < T; t0 += 65535) {
    const size_t es = f32 ? 4 : 2;
    AnyArgs a{(const char*)q + (long)t0 * ldq * es, ldq, pool, tab, max_pages, n_pages, n_rows, row + t0, pos + t0,
              (char*)o + (long)t0 * ldo * es, ldo, H, G, D, V, make_mask(size, keep), scale, cap, out_scale};
    dim3 grid(H, std::min(T - t0, 65535));
    if (f32) hipLaunchKernelGGL((window_any_kernel<float>), grid, dim3(256), lds, stream, a);
    else hipLaunchKernelGGL((window_any_kernel<bf16_t>), grid, dim3(256), lds, stream, a);
    RT_LAUNCH_CHECK();
  }
  return 0;
}
