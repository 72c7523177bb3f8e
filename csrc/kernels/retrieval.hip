// Dense-retrieval kernels (SURVEY K12 pool+normalise, K13 flat top-k, K14 IVF list scan).
//
// The bi-encoder's sentence embedding is a masked mean over tokens followed by L2 normalisation
// (sentence-transformers pooling). Search scores are inner products of normalised vectors
// (= cosine), produced by the MFMA GEMM for flat search or by the IVF list scan below; the top-k
// of a row ranks the few scores that reach a bound from its threads' maxima (no full sort of N = 100k scores).
#include "rt_common.h"

#include <algorithm>
#include <climits>

namespace rt {

// x [B, S, H] bf16, lengths [B] (off: text b is rows [off[b], off[b + 1]) of x [rows, H]) -> out [B, H] fp32 (L2-normalised if norm != 0;
// to: text b to row to[b] of out_rows, from the end if negative, nowhere if there is none such). One workgroup a text; a stream
// of its tokens, bound by the loads in flight: 256 texts of 162 x 768 115 -> 15.5 us over 2-byte loads one after
// the other.
__global__ __launch_bounds__(256) void pool_norm_kernel(const bf16_t* __restrict__ x, const int* __restrict__ lengths,
                                                        const long* __restrict__ off, long rows, int S, int H,
                                                        int normalize, float* __restrict__ out, const long* __restrict__ to,
                                                        long out_rows) {
  extern __shared__ float acc[];  // [H]
  __shared__ float sb[4];
  const int b = blockIdx.x;
  const long first = off ? min(max(off[b], 0L), rows) : (long)b * S;
  const int len = off ? (int)(min(max(off[b + 1], first), rows) - first) : lengths ? lengths[b] : S;
  const bf16_t* xb = x + first * H;
  if (H % 8 == 0 && (uintptr_t)x % 16 == 0) {
    // 8 columns a thread in 16-byte loads, 8 tokens' in flight; a column's tokens are summed in order
    for (int c = threadIdx.x; c < H / 8; c += 256) {
      float s[8] = {};
      int t = 0;
      for (; t + 8 <= len; t += 8) {
        uint4 v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = *(const uint4*)(xb + (long)(t + i) * H + 8 * c);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          float f[8];
          unpack8(v[i], f);
#pragma unroll
          for (int e = 0; e < 8; ++e) s[e] += f[e];
        }
      }
      for (; t < len; ++t) {
        float f[8];
        unpack8(*(const uint4*)(xb + (long)t * H + 8 * c), f);
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] += f[e];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[8 * c + e] = s[e] / (float)max(len, 1);
    }
  } else {
    for (int h = threadIdx.x; h < H; h += 256) {
      float s = 0.f;
      for (int t = 0; t < len; ++t) s += bf2f(xb[(long)t * H + h]);
      acc[h] = s / (float)max(len, 1);
    }
  }
  __syncthreads();
  float ss = 0.f;
  for (int h = threadIdx.x; h < H; h += 256) ss += acc[h] * acc[h];
  const float tot = block_sum(ss, sb);
  const float inv = normalize ? 1.f / fmaxf(sqrtf(tot), 1e-12f) : 1.f;
  const long row = !to ? b : to[b] < 0 ? to[b] + out_rows : to[b];
  if (to && (row < 0 || row >= out_rows)) return;  // no row of out
  for (int h = threadIdx.x; h < H; h += 256) out[row * H + h] = acc[h] * inv;
}

__device__ __forceinline__ uint32_t okey(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

constexpr int TOPK_CAND = 1024;  // candidates of a row held in LDS

struct TopkShared {
  unsigned hist[256];
  uint32_t sel;
  unsigned cnt;
  float cv[TOPK_CAND];
  int ci[TOPK_CAND];
};

// where a row's k results go: values and ids, the candidate's index (-1: none) through idmap if there is one
struct TopkOut {
  const long* idmap; int finite;  // of the row
  float* v; long* i;
  __device__ __forceinline__ long id(int idx) const { return idx == 0x7fffffff ? -1 : idmap ? idmap[idx] : idx; }
  __device__ __forceinline__ void put(int at, float val, long id) const {
    v[at] = val;
    i[at] = finite && !(fabsf(val) < INFINITY) ? -1 : id;
  }
};
// the indices alone
struct TopkIndices {
  int* i;
  __device__ __forceinline__ long id(int idx) const { return idx == 0x7fffffff ? -1 : idx; }
  __device__ __forceinline__ void put(int at, float, long id) const { i[at] = (int)id; }
};

// A row with more candidates than the list holds (plateaus, fewer than K finite scores): 4-pass radix select of the K-th
// key, then exactly K entries in cv / ci: the fewer than K above it, and of its ties those of the lowest indices
template <int NT>
__device__ void topk_select(const float* s, int N, int K, TopkShared& sh) {
  unsigned* hist = sh.hist;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  uint32_t prefix = 0, mask = 0;
  unsigned remaining = (unsigned)K;
  for (int shift = 24; shift >= 0; shift -= 8) {
    for (int b = tid; b < 256; b += NT) hist[b] = 0;
    __syncthreads();
    for (int i = tid; i < N; i += NT) {
      const uint32_t key = okey(s[i]);
      if ((key & mask) == prefix) atomicAdd(&hist[(key >> shift) & 255], 1u);
    }
    __syncthreads();
    if (tid == 0) {
      unsigned cum = 0;
      int sel = 0;
      for (int b = 255; b >= 0; --b) {
        if (cum + hist[b] >= remaining) { sel = b; break; }
        cum += hist[b];
      }
      sh.cnt = cum;
      sh.sel = sel;
    }
    __syncthreads();
    remaining -= sh.cnt;
    prefix |= sh.sel << shift;
    mask |= 255u << shift;
    __syncthreads();
  }
  if (tid == 0) sh.cnt = 0;
  __syncthreads();
  for (int i = tid; i < N; i += NT) {
    const float v = s[i];
    if (okey(v) > prefix) {
      const unsigned slot = atomicAdd(&sh.cnt, 1u);
      if (slot < TOPK_CAND) { sh.cv[slot] = v; sh.ci[slot] = i; }
    }
  }
  __syncthreads();
  int at = (int)sh.cnt;
  for (int i0 = 0; i0 < N && at < K; i0 += NT) {
    const int i = i0 + tid;
    const float v = i < N ? s[i] : 0.f;
    const bool tie = i < N && okey(v) == prefix;
    const unsigned long long in_wave = __ballot(tie);
    if (lane == 0) hist[wid] = (unsigned)__popcll(in_wave);
    __syncthreads();
    int slot = at + (int)__popcll(in_wave & ((1ull << lane) - 1ull));
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
      if (w < wid) slot += (int)hist[w];
      at += (int)hist[w];
    }
    if (tie && slot < K) { sh.cv[slot] = v; sh.ci[slot] = i; }
    __syncthreads();
  }
}

// scores [nq, N] fp32 (row stride ld) -> vals/ids [nq, k] sorted descending (ties: lower index first); ids optionally
// mapped through idmap (IVF candidate slot -> document id). Scores of -inf are never returned as hits unless fewer
// than k finite scores exist; `finite`: the id of a score that is not finite is -1.
// One workgroup of NT threads a row, bound by latency. The k-th largest of the threads' own maxima is a lower bound of
// the row's k-th largest score that few surplus elements reach: the threads that hold one place theirs in LDS, and
// every candidate counts the candidates ahead of it, which is its place in the result. Two passes over the row at
// most, no histogram, no sort (four passes and a sort of 1024 before): top 16 of 512 and top 3 of 9600, one row,
// 88 -> 8.3 and 10.8 us each. Loads of both passes go out in blocks: top 3 of 100k, one row and 200 (top 5), 27 -> 20 and 47 -> 30.
// Up to k = 32 the bound is the k-th largest of 64 maxima, a wave's lanes' (32 rounds of one ballot, where 16 of them took 3 us of a
// row's 10; two candidates more at k = 16, 13 at 32); a row of eight elements a thread is read once; and up to 64 candidates, all
// but rows of many ties, are ranked in the registers of one wave: the two above 7.0 -> 5.5 and 10.7 -> 5.4, of 100k 20 -> 13.6
// and 30 -> 23, 65536 rows of 512 56 -> 50.
// Rows with more than TOPK_CAND candidates go through topk_select first.
// NT: a wave where its 64 maxima suffice (k <= 32) and hold 16 elements each at most (k-means assignment: 65536 rows
// of 512), 1024 threads for long rows, 256 between.
template <int NT, typename Out>
__device__ __forceinline__ void topk_row(const float* s, int N, int k, const Out& out) {
  __shared__ TopkShared sh;
  __shared__ uint32_t tmax[NT];
  __shared__ unsigned char keep[TOPK_CAND];
  const int tid = threadIdx.x, lane = tid & 63, K = min(k, N);
  uint32_t km = 0;
  // eight loads in flight, at the end four, those past it of the last element
  auto scan = [&](auto&& use) {
    int i0 = tid;
    for (; i0 + 7 * NT < N; i0 += 8 * NT) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = s[i0 + e * NT];
#pragma unroll
      for (int e = 0; e < 8; ++e) use(v[e], i0 + e * NT);
    }
    for (; i0 < N; i0 += 4 * NT) {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = s[min(i0 + e * NT, N - 1)];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (i0 + e * NT < N) use(v[e], i0 + e * NT);
    }
  };
  // a row of at most eight a thread is read once
  float own[8];
  const bool few = N > 0 && N <= 8 * NT;
  if (few) {
#pragma unroll
    for (int e = 0; e < 8; ++e) own[e] = s[min(tid + e * NT, N - 1)];
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (tid + e * NT < N) km = max(km, okey(own[e]));
  } else {
    scan([&](float v, int) { km = max(km, okey(v)); });
  }
  tmax[tid] = km;
  if (tid == 0) sh.cnt = 0;
  __syncthreads();
  if (tid < 64) {
    uint32_t t[NT / 64], one[1] = {0};
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) {
      t[i] = tmax[lane + 64 * i];
      one[0] = max(one[0], t[i]);
    }
    const uint32_t thr = K <= 32 ? wave_kth(one, K) : K <= NT ? wave_kth(t, K) : 0;
    if (lane == 0) sh.sel = thr;
  }
  __syncthreads();
  const uint32_t thr = sh.sel;
  if (km >= thr) {
    auto take = [&](float v, int i) {
      if (okey(v) >= thr) {
        const unsigned slot = atomicAdd(&sh.cnt, 1u);
        if (slot < TOPK_CAND) { sh.cv[slot] = v; sh.ci[slot] = i; }
      }
    };
    if (few) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (tid + e * NT < N) take(own[e], tid + e * NT);
    } else {
      scan(take);
    }
  }
  __syncthreads();
  int n = (int)sh.cnt;
  if (n > TOPK_CAND) {
    __syncthreads();  // every thread has read cnt
    topk_select<NT>(s, N, K, sh);
    n = K;
  }
  for (int i = K + tid; i < k; i += NT) out.put(i, -INFINITY, -1);
  if (n <= 64) {  // a candidate a lane, as below
    if (tid >= 64) return;
    const bool in = lane < n;
    const float v = in ? sh.cv[lane] : 0.f;
    const int idx = in ? sh.ci[lane] : 0;
    const long id = in ? out.id(idx) : 0;
    const uint32_t raw = okey(v), key = okey(v + 0.f);
    int above = 0, at = 0;
    for (int i = 0; i < n; ++i) above += (uint32_t)__builtin_amdgcn_readlane((int)raw, i) > raw;
    const bool keeps = in && above < K;
    for (unsigned long long left = __ballot(keeps); left; left &= left - 1) {
      const int i = __builtin_ctzll(left);
      const uint32_t o = (uint32_t)__builtin_amdgcn_readlane((int)key, i);
      const int oi = __builtin_amdgcn_readlane(idx, i);
      at += o > key || (o == key && oi < idx);
    }
    if (keeps && at < K) out.put(at, v, id);
    return;
  }
  // those with fewer than K keys above their own, then their places by value and index
  for (int j = tid; j < n; j += NT) {
    const uint32_t key = okey(sh.cv[j]);
    int above = 0;
    for (int i = 0; i < n; ++i) above += okey(sh.cv[i]) > key;
    keep[j] = above < K;
  }
  __syncthreads();
  for (int j = tid; j < n; j += NT)
    if (keep[j]) {
      // x + 0: the zeros of both signs are one value here
      const float v = sh.cv[j];
      const uint32_t key = okey(v + 0.f);
      const int idx = sh.ci[j];
      int at = 0;
      for (int i = 0; i < n; ++i) {
        const uint32_t o = okey(sh.cv[i] + 0.f);
        at += keep[i] && (o > key || (o == key && sh.ci[i] < idx));
      }
      if (at < K) out.put(at, v, out.id(idx));
    }
}

template <int NT>
__global__ __launch_bounds__(NT) void topk_kernel(const float* __restrict__ scores, long ld, int N, int k,
                                                  const long* __restrict__ idmap, long ldmap, int finite,
                                                  float* __restrict__ out_v, long* __restrict__ out_i) {
  const long row = blockIdx.x;
  topk_row<NT>(scores + row * ld, N, k, TopkOut{idmap ? idmap + row * ldmap : nullptr, finite, out_v + row * k, out_i + row * k});
}

// The indices alone, in 32 bits: the lists that a scan probes
template <int NT>
__global__ __launch_bounds__(NT) void topk_index_kernel(const float* __restrict__ scores, long ld, int N, int k, int* __restrict__ out) {
  const long row = blockIdx.x;
  topk_row<NT>(scores + row * ld, N, k, TopkIndices{out + row * k});
}

// Scores of up to 16 queries with the centroids, q cen^T - pen, from fp32 queries, which go on in bf16 to the scan. A workgroup has 16 centroids,
// a wave one of the product's parts of K; parts and groups are summed in the product's order: the same bits. Bound by one trip to
// memory; rounding and product took two launches.
struct CoarseArgs {
  const float* q; int nq, d; const bf16_t* cen; int nlist; const float* pen;
  int parts, grp;
  bf16_t* qb; float* score;
};
__global__ __launch_bounds__(1024) void ivf_coarse_kernel(CoarseArgs a) {
  __shared__ float red[16][4][65];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, r16 = lane & 15;
  const int part = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nc = a.d / 64, c0 = (int)((long)part * nc / a.parts), c1 = (int)((long)(part + 1) * nc / a.parts);
  const bf16_t* const x = a.cen + (16L * blockIdx.x + r16) * a.d + 8 * g;  // rows up to a multiple of 16 are there
  const long qrow = min(r16, a.nq - 1);
  const float* const q = a.q + qrow * a.d + 8 * g;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  constexpr int U = 2;
  for (int c = c0; c < c1; c += U) {
    uint4 xv[U][2];
    float4 qv[U][2][2];
#pragma unroll
    for (int i = 0; i < U; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int k = 64 * min(c + i, c1 - 1) + 32 * h;
        xv[i][h] = *(const uint4*)(x + k);
        qv[i][h][0] = *(const float4*)(q + k);
        qv[i][h][1] = *(const float4*)(q + k + 4);
      }
#pragma unroll
    for (int i = 0; i < U; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (c + i >= c1) continue;
        const float4 lo = qv[i][h][0], hi = qv[i][h][1];
        const uint4 y = make_uint4(pack2bf(lo.x, lo.y), pack2bf(lo.z, lo.w), pack2bf(hi.x, hi.y), pack2bf(hi.z, hi.w));
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, y), __builtin_bit_cast(bf16x8, xv[i][h]), acc, 0, 0, 0);
        if (blockIdx.x == 0 && r16 < a.nq) *(uint4*)(a.qb + qrow * a.d + 64 * (c + i) + 32 * h + 8 * g) = y;
      }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) red[part][r][lane] = acc[r];
  __syncthreads();
  // acc[r] of a lane: query 4 g + r, centroid r16
  if (tid >= 256) return;
  const int r = tid >> 6, query = 4 * g + r, c = 16 * (int)blockIdx.x + r16;
  float v = 0.f, u = 0.f;
  for (int p = 0, in = 0; p < a.parts; ++p) {
    const float t = red[p][r][lane];
    u = in ? u + t : t;
    if (++in == a.grp) {
      v = a.parts == a.grp ? u : v + u;
      in = 0;
    }
  }
  if (query < a.nq && c < a.nlist) a.score[(long)query * a.nlist + c] = a.pen ? v - a.pen[c] : v;
}

// IVF list scan: for query qi and its probe p (list L = probes[qi, p]), score every vector of the
// list (vectors stored contiguously per list from lstart[L], lsize[L] of them; lists may carry
// spare capacity for incremental adds) and write into cand[qi, p*maxlen + j] (+ ids).
// Metric: inner product, or (l2) the negated squared distance 2 q.x - |x|^2 - |q|^2 with |x|^2
// stored per slot — both "higher is better" for the shared top-k. Unused slots get -inf, and so do probes of no list.
struct ScanArgs {
  const bf16_t* q; int nq, d; const int* probes; int nprobe, nlist;
  const int* lstart; const int* lsize; const bf16_t* vecs; const long* ids; const float* sqnorm;
  int l2, maxlen, per;  // per: vectors of a workgroup at least (by list)
  float* cand; long* cand_ids;
};
// 8 elements a lane from a uniform base + off bytes, 0 beyond `bytes` (at most 2^30; FAR lies beyond)
constexpr uint32_t FAR = 0x60000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t scan_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ bf16x8 scan_load(__amdgpu_buffer_rsrc_t r, uint32_t off, int base) {
  return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, off, base, 0));
}

// By probe: one wave per 64 vectors of a (probe, query), one thread per vector, query in LDS: a single query's 16 lists of 200 to
// 800 are a few hundred waves on as many CUs, where one workgroup per list left 240 CUs idle; 8 of a vector's 16-byte
// pieces are in flight (16 lists of 600 x 384: 12.4 -> 8.6 us). A vector's terms are summed in the order of the
// dimensions.
typedef u32x4 __attribute__((aligned(2))) u32x4_any;
__device__ __forceinline__ uint4 load2(const bf16_t* p) { return __builtin_bit_cast(uint4, (u32x4)*(const u32x4_any*)p); }  // vectors at any address
__global__ __launch_bounds__(64) void ivf_probe_kernel(const bf16_t* __restrict__ q, int d, const int* __restrict__ probes,
                                                       int nprobe, int nlist, const int* __restrict__ lstart,
                                                       const int* __restrict__ lsize, const bf16_t* __restrict__ vecs,
                                                       const long* __restrict__ ids, const float* __restrict__ sqnorm,
                                                       int l2, int maxlen, float* __restrict__ cand,
                                                       long* __restrict__ cand_ids) {
  extern __shared__ float qs[];
  const int p = blockIdx.x, qi = blockIdx.y;
  const long j0 = blockIdx.z * 64L, step = gridDim.z * 64L;
  const int L = probes[(long)qi * nprobe + p];
  const bool real = L >= 0 && L < nlist;
  const int b0 = real ? lstart[L] : 0;
  const int len = real ? min(lsize[L], maxlen) : 0;
  float* out = cand + ((long)qi * nprobe + p) * maxlen;
  long* oid = cand_ids + ((long)qi * nprobe + p) * maxlen;
  if (j0 >= len) {
    for (long j = j0 + threadIdx.x; j < maxlen; j += step) { out[j] = -INFINITY; oid[j] = -1; }
    return;
  }
  // |q|^2 in four interleaved parts, added in order
  float part[4] = {};
  for (int i0 = threadIdx.x; i0 < d; i0 += 256) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const int i = i0 + 64 * w;
      if (i >= d) continue;
      const float v = bf2f(q[(long)qi * d + i]);
      qs[i] = v;
      part[w] += v * v;
    }
  }
  float qn = 0.f;
  if (l2) {
#pragma unroll
    for (int w = 0; w < 4; ++w) qn += wave_sum(part[w]);
  }
  __syncthreads();
  for (long j = j0 + threadIdx.x; j < maxlen; j += step) {
    if (j >= len) {
      out[j] = -INFINITY;
      oid[j] = -1;
      continue;
    }
    const bf16_t* vr = vecs + (b0 + j) * d;
    float s = 0.f;
    int c = 0;
    for (; c + 64 <= d; c += 64) {
      uint4 v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = load2(vr + c + 8 * i);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float f[8];
        unpack8(v[i], f);
#pragma unroll
        for (int e = 0; e < 8; ++e) s += f[e] * qs[c + 8 * i + e];
      }
    }
    for (; c < d; c += 8) {
      float f[8];
      unpack8(load2(vr + c), f);
#pragma unroll
      for (int e = 0; e < 8; ++e) s += f[e] * qs[c + e];
    }
    out[j] = l2 ? 2.f * s - sqnorm[b0 + j] - qn : s;
    oid[j] = ids[b0 + j];
  }
}

// The same of 256 < d <= 384 and lists that are even or at most 4096 long: a wave per 16 vectors, whose pieces are all in flight as MFMA
// fragments at once, the query as the other operand's sixteen rows. A single query over 16 lists of 200 and of 780, 7.3 -> 5.2 and 7.5 -> 5.8
// us; many queries over lists of 100 20.3 -> 16.4 (64 x 16 of 4096), 53 -> 49 (256 x 16). Smaller d leaves the wave with too little in flight
// (128: 1.3 to 1.5 times the time), 768 takes half the waves away (1.0 to 1.15 times); one and two queries over skewed
// lists of up to 7909 16.7 against 15.9 and 29.7 against 27.6, over even ones of up to 8735 11.1 against 12.3 and 18.5 against 19.6.
constexpr int PF = 12;
__global__ __launch_bounds__(256, 4) void ivf_probe16_kernel(ScanArgs a) {
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, r16 = lane & 15;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long pr = (long)blockIdx.y * a.nprobe + blockIdx.x;
  const int L = a.probes[pr];
  const bool real = L >= 0 && L < a.nlist;
  const int b0 = real ? a.lstart[L] : 0, len = real ? max(min(a.lsize[L], a.maxlen), 0) : 0;
  const int z0 = blockIdx.z, zn = gridDim.z;
  if (z0 * 64L >= len && len + z0 * 256L >= a.maxlen) return;  // no vectors here and no slots to fill
  float* const out = a.cand + pr * a.maxlen;
  long* const oid = a.cand_ids + pr * a.maxlen;
  for (long j = len + z0 * 256L + tid; j < a.maxlen; j += zn * 256L) {
    out[j] = -INFINITY;
    oid[j] = -1;
  }
  bf16x8 y[PF];
  const auto qr = scan_rsrc(a.q + (long)blockIdx.y * a.d, (uint32_t)a.d * 2);
#pragma unroll
  for (int s = 0; s < PF; ++s) y[s] = scan_load(qr, 16 * g, 64 * s);
  float qq = 0.f;
  if (a.l2) {
#pragma unroll
    for (int s = 0; s < PF; ++s) {
      float f[8];
      unpack8(__builtin_bit_cast(uint4, y[s]), f);
#pragma unroll
      for (int e = 0; e < 8; ++e) qq = fmaf(f[e], f[e], qq);
    }
    qq += __shfl_xor(qq, 16, 64);
    qq += __shfl_xor(qq, 32, 64);
  }
  for (long v0 = z0 * 64L + wid * 16; v0 < len; v0 += zn * 64L) {
    const auto vr = scan_rsrc(a.vecs + (b0 + v0) * a.d, (uint32_t)min(16L, len - v0) * a.d * 2);
    uint32_t vo = (uint32_t)(r16 * a.d + 8 * g) * 2;
    asm volatile("" : "+v"(vo));  // the offsets below are not worth a register each
    bf16x8 x[PF];
#pragma unroll
    for (int s = 0; s < PF; ++s) x[s] = scan_load(vr, 32 * s + 8 * g < a.d ? vo : FAR, 64 * s);
    const long at = b0 + min(v0 + r16, (long)len - 1);
    const long id = a.ids[at];
    const float sq = a.l2 ? a.sqnorm[at] : 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < PF; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(y[s], x[s], acc, 0, 0, 0);
    // every row of the product is the query's: column r16 is vector v0 + r16
    if (g == 0 && v0 + r16 < len) {
      out[v0 + r16] = a.l2 ? 2.f * acc[0] - sq - qq : acc[0];
      oid[v0 + r16] = id;
    }
  }
}

// By list: 64 vectors of a list and more for every query that probes it, found among the probes; a wave multiplies 16 vectors, held as
// MFMA fragments, with 16 queries at a time. Bound by the bytes read and written (12 a candidate), by reading the
// probes where lists are many and short, and by the chain from probe to result where a list has few queries. us, by probe -> by list: 64 queries
// x 16 of 512 lists, 100k vectors of 384 28.6 -> 20.5, 256 queries 84 -> 27; 4 and 12 queries x 16 of 256 lists of up to 7909 48.8 -> 29.9,
// 100 -> 36; 4096 queries x 32 of 4096 lists of about 100 1335 -> 555. (With the probes taken 4096 at a time a list of those
// had one query a round and read its vectors 32 times: 1690.)
constexpr int PAIRS = 4096;
// NF: 32-element fragments of a vector held at once; LONG: a vector has more
template <int NF, bool LONG>
__global__ __launch_bounds__(256, NF == 12 ? 4 : 2) void ivf_list_kernel(ScanArgs a) {
  __shared__ uint32_t pair[PAIRS];  // query * nprobe + probe, from the round's first one
  __shared__ int count;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, r16 = lane & 15;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int L = blockIdx.x;  // nlist stands for no list
  const bool real = L < a.nlist;
  const int b0 = real ? a.lstart[L] : 0, len = real ? max(min(a.lsize[L], a.maxlen), 0) : 0;
  // the list's workgroups, by its vectors and by the slots behind them (a query's are up to 1024 a workgroup: 256 queries x 16 lists, one
  // of 69360 of 200k vectors, 2990 us with one workgroup for a short list, 1840 so); the others need not look for its queries
  const int z0 = blockIdx.z, zn = min((int)gridDim.z, max(max((len + a.per - 1) / a.per, (a.maxlen - len + 1023) / 1024), 1));
  if (z0 >= zn) return;
  // the probes from base on, m of them, that ask for this list: their number, the first PAIRS of them in pair[]
  auto collect = [&](long base, long m) {
    __syncthreads();  // the last pairs and their number have been read
    if (tid == 0) count = 0;
    __syncthreads();
    for (long i0 = tid; i0 < m; i0 += 256 * 16) {
      int l[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) l[e] = a.probes[base + min(i0 + e * 256, m - 1)];
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (i0 + e * 256 < m && (real ? l[e] == L : l[e] < 0 || l[e] >= a.nlist)) {
          const int at = atomicAdd(&count, 1);
          if (at < PAIRS) pair[at] = (uint32_t)(i0 + e * 256);
        }
    }
    __syncthreads();
    return count;
  };
  // a round has all probes, unless more than PAIRS of them ask for this list
  const long all = (long)a.nq * a.nprobe;
  for (long base = 0, step = min(all, 1L << 30); base < all; base += step) {
    int n = collect(base, min(all - base, step));
    if (n > PAIRS) {
      step = PAIRS;
      n = collect(base, min(all - base, step));
    }
    auto pair_of = [&](int k) { return base + pair[k]; };
    for (int k = 0; k < n; ++k) {  // slots behind the list's vectors
      const long o = pair_of(k) * a.maxlen;
      for (long j = len + z0 * 256L + tid; j < a.maxlen; j += zn * 256L) {
        a.cand[o + j] = -INFINITY;
        a.cand_ids[o + j] = -1;
      }
    }
    if (n == 0) continue;
    for (long v0 = z0 * 64L + wid * 16; v0 < len; v0 += zn * 64L) {
      const auto vr = scan_rsrc(a.vecs + (b0 + v0) * a.d, (uint32_t)min(16L, len - v0) * a.d * 2);
      bf16x8 x[NF];
      auto load = [&](int c0) {
        uint32_t vo = (uint32_t)(r16 * a.d + 8 * g) * 2;
        asm volatile("" : "+v"(vo));  // the offsets below are not worth a register each
#pragma unroll
        for (int s = 0; s < NF; ++s) x[s] = scan_load(vr, c0 + 32 * s + 8 * g < a.d ? vo : FAR, (c0 + 32 * s) * 2);
      };
      if constexpr (!LONG) load(0);
      const long at = b0 + min(v0 + r16, (long)len - 1);
      const long id = a.ids[at];
      const float sq = a.l2 ? a.sqnorm[at] : 0.f;
      const auto qr = scan_rsrc(a.q, (uint32_t)a.nq * a.d * 2);
      for (int t = 0; t < n; t += 16) {
        uint32_t qo = (uint32_t)(pair_of(min(t + r16, n - 1)) / a.nprobe * a.d + 8 * g) * 2;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        float qq = 0.f;
        auto part = [&](int c0) {
#pragma unroll
          for (int s0 = 0; s0 < NF; s0 += 4) {
            asm volatile("" : "+v"(qo));
            bf16x8 y[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) y[s] = scan_load(qr, c0 + 32 * (s0 + s) + 8 * g < a.d ? qo : FAR, (c0 + 32 * (s0 + s)) * 2);
#pragma unroll
            for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(y[s], x[s0 + s], acc, 0, 0, 0);
            if (a.l2) {
#pragma unroll
              for (int s = 0; s < 4; ++s) {
                float f[8];
                unpack8(__builtin_bit_cast(uint4, y[s]), f);
#pragma unroll
                for (int e = 0; e < 8; ++e) qq = fmaf(f[e], f[e], qq);
              }
            }
          }
        };
        if constexpr (LONG) {
          for (int c0 = 0; c0 < a.d; c0 += 32 * NF) {
            load(c0);
            part(c0);
          }
        } else {
          part(0);
        }
        if (a.l2) {
          qq += __shfl_xor(qq, 16, 64);
          qq += __shfl_xor(qq, 32, 64);
        }
        // acc[i]: query 4 g + i of the sixteen, vector v0 + r16
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int k = t + 4 * g + i;
          const float qn = a.l2 ? __shfl(qq, 4 * g + i, 64) : 0.f;
          if (k < n && v0 + r16 < len) {
            const long o = pair_of(k) * a.maxlen + v0 + r16;
            a.cand[o] = a.l2 ? 2.f * acc[i] - sq - qn : acc[i];
            a.cand_ids[o] = id;
          }
        }
      }
    }
  }
}

// k-means update: centroid c = mean of the rows order[seg[c] .. seg[c+1]) of x (rows sorted by
// assigned centroid), L2-normalised for the inner-product metric. One workgroup per centroid, a
// column per thread, rows summed in a fixed order (deterministic, no atomics). Empty clusters are
// left untouched (the caller reseeds them). mode bit 0: L2-normalise; bit 1: the plain segment sum
// (the deterministic embedding-table gradient, ops.misc._EmbedFn).
__global__ __launch_bounds__(256) void segment_mean_kernel(const float* __restrict__ x, int d,
                                                           const long* __restrict__ order, const int* __restrict__ seg,
                                                           int mode, float* __restrict__ out) {
  extern __shared__ float col[];  // [d]
  __shared__ float sb[4];
  const int c = blockIdx.x;
  const int r0 = seg[c], r1 = seg[c + 1];
  if (r1 <= r0) return;  // uniform over the block
  const bool normalize = mode & 1;
  const float inv = (mode & 2) ? 1.f : 1.f / (float)(r1 - r0);  // bit 1: plain sum
  float ss = 0.f;
  for (int j = threadIdx.x; j < d; j += 256) {
    float a = 0.f;
    for (int r = r0; r < r1; ++r) a += x[order[r] * (long)d + j];
    a *= inv;
    col[j] = a;
    ss += a * a;
  }
  const float tot = normalize ? block_sum(ss, sb) : 1.f;
  const float scale = normalize ? 1.f / fmaxf(sqrtf(tot), 1e-12f) : 1.f;
  __syncthreads();
  for (int j = threadIdx.x; j < d; j += 256) out[(long)c * d + j] = col[j] * scale;
}

}  // namespace rt

using namespace rt;

extern "C" int rt_pool_norm(const void* x, const int* lengths, const long* off, long rows, int B, int S, int H,
                            int normalize, float* out, const long* to, long out_rows, hipStream_t stream) {
  if (B == 0) return 0;
  hipLaunchKernelGGL(pool_norm_kernel, dim3(B), dim3(256), H * sizeof(float), stream, (const bf16_t*)x, lengths, off, rows,
                     S, H, normalize, out, to, out_rows);
  RT_LAUNCH_CHECK();
  return 0;
}

extern "C" int rt_topk(const float* scores, long ld, long nq, int N, int k, const long* idmap, long ldmap, int finite,
                       float* out_v, long* out_i, hipStream_t stream) {
  if (k > TOPK_CAND / 2) return -1;
  if (nq == 0 || k <= 0) return 0;
#define TOPK_LAUNCH(NT)                                                                                       \
  hipLaunchKernelGGL(topk_kernel<NT>, dim3(nq), dim3(NT), 0, stream, scores, ld, N, k, idmap, ldmap, finite, \
                     out_v, out_i)
  if (k <= 32 && N <= 1024) TOPK_LAUNCH(64);
  else if (k <= 128 && N <= 4096) TOPK_LAUNCH(256);
  else TOPK_LAUNCH(1024);
#undef TOPK_LAUNCH
  RT_LAUNCH_CHECK();
  return 0;
}

extern "C" int rt_topk_index(const float* scores, long ld, long nq, int N, int k, int* out, hipStream_t stream) {
  if (k > TOPK_CAND / 2 || k > N) return -1;
  if (nq == 0 || k <= 0) return 0;
#define TOPK_LAUNCH(NT) hipLaunchKernelGGL(topk_index_kernel<NT>, dim3(nq), dim3(NT), 0, stream, scores, ld, N, k, out)
  if (k <= 32 && N <= 1024) TOPK_LAUNCH(64);
  else if (k <= 128 && N <= 4096) TOPK_LAUNCH(256);
  else TOPK_LAUNCH(1024);
#undef TOPK_LAUNCH
  RT_LAUNCH_CHECK();
  return 0;
}

// score [nq, nlist] and q in bf16, see ivf_coarse_kernel; cen: rows [nlist up to a multiple of 16, d]. -1: not for this kernel.
extern "C" int rt_ivf_coarse(const float* q, int nq, int d, const void* cen, int nlist, const float* pen, int parts, int grp, void* qb,
                             float* score, hipStream_t stream) {
  if (nq < 1 || nq > 16 || d < 64 || d % 64 || nlist < 1 || parts < 4 || parts > 16 || grp < 1 || parts % grp) return -1;
  if ((uintptr_t)q % 16 || (uintptr_t)cen % 16) return -1;
  const CoarseArgs a{q, nq, d, (const bf16_t*)cen, nlist, pen, parts, grp, (bf16_t*)qb, score};
  hipLaunchKernelGGL(ivf_coarse_kernel, dim3((nlist + 15) / 16), dim3(64 * parts), 0, stream, a);
  RT_LAUNCH_CHECK();
  return 0;
}

// Which form a scan takes (total: vectors in all lists, at most). What either takes, in bytes at the rate of a copy: by probe every
// candidate's vector (and 35 more); by list every vector, 300 for its share of a workgroup's chain, 125 a candidate and a look at
// every probe for every list. Fitted to 300 calls of 1 to 20000 queries over 1 to 4096 lists, even and skewed, d of 72 to 1024: none
// of them is slower than by probe. Queries that do not fit a wave's LDS go by list.
extern "C" int rt_ivf_by_list(int nq, int nprobe, int nlist, int d, int maxlen, long total) {
  const double P = (double)nq * nprobe, len = std::min(0.7 * maxlen, (double)total);
  return d > 16384 || (nq > 1 && total * (2. * d + 300) + P * len * 125 + 3.6 * nlist * P + 10e6 < P * len * (2. * d + 35));
}

extern "C" int rt_ivf_scan(const void* q, int nq, int d, const int* probes, int nprobe, int nlist, const int* lstart,
                           const int* lsize, const void* vecs, long total, const long* ids, const float* sqnorm, int l2,
                           int maxlen, float* cand, long* cand_ids, hipStream_t stream) {
  if (d % 8 != 0 || (l2 && !sqnorm)) return -1;
  if (nq == 0 || nprobe == 0) return 0;
  if (maxlen <= 0) return 0;
  if (d > 1 << 24) return -1;
  const bool aligned = (uintptr_t)q % 16 == 0 && (uintptr_t)vecs % 16 == 0;  // else a thread per vector
  const bool by_list = aligned && rt_ivf_by_list(nq, nprobe, nlist, d, maxlen, total);
  // as many queries at once as a grid's second dimension has, or as 32-bit offsets reach
  const long most_q = by_list ? std::min((1L << 30) / (2L * d), (long)INT_MAX) : 65535;
  if (nq > most_q) {
    for (long i = 0; i < nq; i += most_q) {
      const int rc = rt_ivf_scan((const bf16_t*)q + i * d, (int)std::min(most_q, nq - i), d, probes + i * nprobe, nprobe, nlist, lstart, lsize,
                                 vecs, total, ids, sqnorm, l2, maxlen, cand + i * nprobe * maxlen, cand_ids + i * nprobe * maxlen, stream);
      if (rc) return rc;
    }
    return 0;
  }
  // 64 vectors a workgroup up to some six thousand of them; a long list goes round its own
  const int per = by_list ? (int)std::max(64L, (total / 6144 + 63) / 64 * 64) : 64;
  const ScanArgs a{(const bf16_t*)q, nq, d, probes, nprobe, nlist, lstart, lsize, (const bf16_t*)vecs, ids, sqnorm, l2, maxlen, per, cand, cand_ids};
  // a grid's third dimension ends at 65535: longer lists (over 4 million vectors) go round
  const long pieces = std::min((maxlen + per - 1L) / per, 65535L);
  if (!by_list) {
    const dim3 grid(nprobe, nq, (unsigned)pieces);
    if (aligned && d > 256 && d <= 32 * PF && (maxlen <= 4096 || (double)maxlen * nlist <= 2. * total))
      hipLaunchKernelGGL(ivf_probe16_kernel, grid, dim3(256), 0, stream, a);
    else
      hipLaunchKernelGGL(ivf_probe_kernel, grid, dim3(64), d * sizeof(float), stream, a.q, d, probes, nprobe, nlist, lstart, lsize, a.vecs,
                         ids, sqnorm, l2, maxlen, cand, cand_ids);
    RT_LAUNCH_CHECK();
    return 0;
  }
  const dim3 grid(nlist + 1, 1, (unsigned)std::min(pieces, std::max(64L, 16384L / (nlist + 1))));
  if (d <= 384) hipLaunchKernelGGL((ivf_list_kernel<12, false>), grid, dim3(256), 0, stream, a);
  else if (d <= 768) hipLaunchKernelGGL((ivf_list_kernel<24, false>), grid, dim3(256), 0, stream, a);
  else hipLaunchKernelGGL((ivf_list_kernel<12, true>), grid, dim3(256), 0, stream, a);
  RT_LAUNCH_CHECK();
  return 0;
}

extern "C" int rt_segment_mean(const float* x, int d, const long* order, const int* seg, int k, int mode,
                               float* out, hipStream_t stream) {
  if (k == 0) return 0;
  hipLaunchKernelGGL(segment_mean_kernel, dim3(k), dim3(256), d * sizeof(float), stream, x, d, order, seg, mode, out);
  RT_LAUNCH_CHECK();
  return 0;
}
