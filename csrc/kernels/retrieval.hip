// Dense-retrieval kernels (SURVEY K12 pool+normalise, K13 flat top-k, K14 IVF list scan).
//
// The bi-encoder's sentence embedding is a masked mean over tokens followed by L2 normalisation
// (sentence-transformers pooling). Search scores are inner products of normalised vectors
// (= cosine), produced by the MFMA GEMM for flat search or by the IVF list scan below; the top-k
// of a row ranks the few scores that reach a bound from its threads' maxima (no full sort of N = 100k scores).
#include "rt_common.h"

#include <algorithm>

namespace rt {

// x [B, S, H] bf16, lengths [B] (off: text b is rows [off[b], off[b + 1]) of x [rows, H]) -> out [B, H] fp32 (L2-normalised if norm != 0). One workgroup a text; a stream
// of its tokens, bound by the loads in flight: 256 texts of 162 x 768 115 -> 15.5 us over 2-byte loads one after
// the other.
__global__ __launch_bounds__(256) void pool_norm_kernel(const bf16_t* __restrict__ x, const int* __restrict__ lengths,
                                                        const long* __restrict__ off, long rows, int S, int H,
                                                        int normalize, float* __restrict__ out, const long* __restrict__ to) {
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
  for (int h = threadIdx.x; h < H; h += 256) out[(to ? to[b] : (long)b) * H + h] = acc[h] * inv;
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

__device__ __forceinline__ void topk_write(float v, int idx, int k, int at, long row, const long* idmap, long ldmap,
                                           int finite, float* out_v, long* out_i) {
  out_v[row * k + at] = v;
  long id = idx == 0x7fffffff ? -1 : idx;
  if (idmap && id >= 0) id = idmap[row * ldmap + id];
  if (finite && !(fabsf(v) < INFINITY)) id = -1;
  out_i[row * k + at] = id;
}

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
// 88 -> 8.3 and 10.8 us each. Rows with more than TOPK_CAND candidates go through topk_select first.
// NT: a wave where its 64 maxima suffice (k <= 32) and hold 16 elements each at most (k-means assignment: 65536 rows
// of 512), 1024 threads for long rows, 256 between.
template <int NT>
__global__ __launch_bounds__(NT) void topk_kernel(const float* __restrict__ scores, long ld, int N, int k,
                                                  const long* __restrict__ idmap, long ldmap, int finite,
                                                  float* __restrict__ out_v, long* __restrict__ out_i) {
  __shared__ TopkShared sh;
  __shared__ uint32_t tmax[NT];
  __shared__ unsigned char keep[TOPK_CAND];
  const long row = blockIdx.x;
  const float* s = scores + row * ld;
  const int tid = threadIdx.x, lane = tid & 63, K = min(k, N);
  uint32_t km = 0;
  int i0 = tid;
  for (; i0 + 7 * NT < N; i0 += 8 * NT) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = s[i0 + e * NT];
#pragma unroll
    for (int e = 0; e < 8; ++e) km = max(km, okey(v[e]));
  }
  for (; i0 < N; i0 += NT) km = max(km, okey(s[i0]));
  tmax[tid] = km;
  if (tid == 0) sh.cnt = 0;
  __syncthreads();
  if (tid < 64) {
    uint32_t t[NT / 64];
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) t[i] = tmax[lane + 64 * i];
    const uint32_t thr = K <= NT ? wave_kth(t, K) : 0;
    if (lane == 0) sh.sel = thr;
  }
  __syncthreads();
  const uint32_t thr = sh.sel;
  if (km >= thr)
    for (int i = tid; i < N; i += NT) {
      const float v = s[i];
      if (okey(v) >= thr) {
        const unsigned slot = atomicAdd(&sh.cnt, 1u);
        if (slot < TOPK_CAND) { sh.cv[slot] = v; sh.ci[slot] = i; }
      }
    }
  __syncthreads();
  int n = (int)sh.cnt;
  if (n > TOPK_CAND) {
    __syncthreads();  // every thread has read cnt
    topk_select<NT>(s, N, K, sh);
    n = K;
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
      if (at < K) topk_write(v, idx, k, at, row, idmap, ldmap, finite, out_v, out_i);
    }
  for (int i = K + tid; i < k; i += NT) topk_write(-INFINITY, 0x7fffffff, k, i, row, idmap, ldmap, finite, out_v, out_i);
}

// IVF list scan: for query qi and its probe p (list L = probes[qi, p]), score every vector of the
// list (vectors stored contiguously per list from lstart[L], lsize[L] of them; lists may carry
// spare capacity for incremental adds) and write into cand[qi, p*maxlen + j] (+ ids).
// Metric: inner product, or (l2) the negated squared distance 2 q.x - |x|^2 - |q|^2 with |x|^2
// stored per slot — both "higher is better" for the shared top-k. Unused slots get -inf.
// One wave per 64 vectors of a (probe, query), one thread per vector, query in LDS: a single query's 16 lists of 200 to
// 800 are a few hundred waves on as many CUs, where one workgroup per list left 240 CUs idle; 8 of a vector's 16-byte
// pieces are in flight (16 lists of 600 x 384: 12.4 -> 8.6 us). A vector's terms are summed in the order of the
// dimensions.
__global__ __launch_bounds__(64) void ivf_scan_kernel(const bf16_t* __restrict__ q, int d, const int* __restrict__ probes,
                                                      int nprobe, const int* __restrict__ lstart,
                                                      const int* __restrict__ lsize, const bf16_t* __restrict__ vecs,
                                                      const long* __restrict__ ids, const float* __restrict__ sqnorm,
                                                      int l2, int maxlen, float* __restrict__ cand,
                                                      long* __restrict__ cand_ids) {
  extern __shared__ float qs[];
  const int p = blockIdx.x, qi = blockIdx.y;
  const long j0 = blockIdx.z * 64L, step = gridDim.z * 64L;
  const int L = probes[(long)qi * nprobe + p];
  const int b0 = L >= 0 ? lstart[L] : 0;
  const int len = L >= 0 ? min(lsize[L], maxlen) : 0;
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
      for (int i = 0; i < 8; ++i) v[i] = *(const uint4*)(vr + c + 8 * i);
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
      unpack8(*(const uint4*)(vr + c), f);
#pragma unroll
      for (int e = 0; e < 8; ++e) s += f[e] * qs[c + e];
    }
    out[j] = l2 ? 2.f * s - sqnorm[b0 + j] - qn : s;
    oid[j] = ids[b0 + j];
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
                            int normalize, float* out, const long* to, hipStream_t stream) {
  if (B == 0) return 0;
  hipLaunchKernelGGL(pool_norm_kernel, dim3(B), dim3(256), H * sizeof(float), stream, (const bf16_t*)x, lengths, off, rows,
                     S, H, normalize, out, to);
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

extern "C" int rt_ivf_scan(const void* q, int nq, int d, const int* probes, int nprobe, const int* lstart,
                           const int* lsize, const void* vecs, const long* ids, const float* sqnorm, int l2,
                           int maxlen, float* cand, long* cand_ids, hipStream_t stream) {
  if (d % 8 != 0 || (l2 && !sqnorm)) return -1;
  if (nq == 0) return 0;
  if (maxlen <= 0) return 0;
  // a grid's third dimension ends at 65535: longer lists (over 4 million vectors) go round
  const unsigned pieces = (unsigned)std::min((maxlen + 63L) / 64, 65535L);
  hipLaunchKernelGGL(ivf_scan_kernel, dim3(nprobe, nq, pieces), dim3(64), d * sizeof(float), stream, (const bf16_t*)q, d, probes,
                     nprobe, lstart, lsize, (const bf16_t*)vecs, ids, sqnorm, l2, maxlen, cand, cand_ids);
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
