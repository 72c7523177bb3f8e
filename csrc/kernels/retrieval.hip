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
// 88 -> 8.3 and 10.8 us each. Loads of both passes go out in blocks: top 3 of 100k, one row and 200 (top 5), 27 -> 20 and 47 -> 30.
// Rows with more than TOPK_CAND candidates go through topk_select first.
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
  scan([&](float v, int) { km = max(km, okey(v)); });
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
    scan([&](float v, int i) {
      if (okey(v) >= thr) {
        const unsigned slot = atomicAdd(&sh.cnt, 1u);
        if (slot < TOPK_CAND) { sh.cv[slot] = v; sh.ci[slot] = i; }
      }
    });
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
// stored per slot — both "higher is better" for the shared top-k. Unused slots get -inf, and so do probes of no list.
// A wave multiplies 16 vectors, held as MFMA fragments (64 B of 16 vectors a load), with 16 queries at a time; a thread per vector
// had each 16-byte load of a wave touch 64 lines, of which L1 kept none for the next one. BY_LIST: a workgroup takes 64
// vectors of a list for every query that probes it, found among the probes, PAIRS at a time; else for one (query, probe).
// Bound by the bytes read and written (12 a candidate). us, the thread per vector -> this: 64 queries over lists of up to 102108
// vectors of 384 (200k in all) 9500 -> 724, 100 queries over 30k 2473 -> 202, one query over 16 lists of 200 10.5 -> 8.
constexpr int PAIRS = 4096;
struct ScanArgs {
  const bf16_t* q; int nq, d; const int* probes; int nprobe, nlist;
  const int* lstart; const int* lsize; const bf16_t* vecs; const long* ids; const float* sqnorm;
  int l2, maxlen;
  float* cand; long* cand_ids;
};

template <int NF, bool BY_LIST>  // NF: 32-element fragments of a vector held at once
__global__ __launch_bounds__(256) void ivf_scan_kernel(ScanArgs a) {
  __shared__ int pair[BY_LIST ? PAIRS : 1];  // query * nprobe + probe, from the round's first one
  __shared__ int count;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, r16 = lane & 15;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long all = BY_LIST ? (long)a.nq * a.nprobe : 1, first = BY_LIST ? 0 : (long)blockIdx.y * a.nprobe + blockIdx.x;
  const int L = BY_LIST ? blockIdx.x : a.probes[first];  // BY_LIST: nlist stands for no list
  const bool real = L >= 0 && L < a.nlist;
  const int b0 = real ? a.lstart[L] : 0, len = real ? min(a.lsize[L], a.maxlen) : 0;
  const int z0 = blockIdx.z, zn = gridDim.z;
  if (z0 * 64L >= len && len + z0 * 256L >= a.maxlen) return;  // no vectors here and no slots to fill
  for (long base = 0; base < all; base += PAIRS) {
    int n = 1;
    if constexpr (BY_LIST) {
      const int m = (int)min(all - base, (long)PAIRS);
      __syncthreads();  // the last round's pairs have been read
      if (tid == 0) count = 0;
      __syncthreads();
      for (int i0 = tid; i0 < m; i0 += 256 * 8) {
        int l[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) l[e] = a.probes[base + min(i0 + e * 256, m - 1)];
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (i0 + e * 256 < m && (real ? l[e] == L : l[e] < 0 || l[e] >= a.nlist)) pair[atomicAdd(&count, 1)] = i0 + e * 256;
      }
      __syncthreads();
      n = count;
    }
    auto pair_of = [&](int k) { return BY_LIST ? base + pair[k] : first; };
    for (int k = 0; k < n; ++k) {  // slots behind the list's vectors
      const long o = pair_of(k) * a.maxlen;
      for (long j = len + z0 * 256L + tid; j < a.maxlen; j += zn * 256L) {
        a.cand[o + j] = -INFINITY;
        a.cand_ids[o + j] = -1;
      }
    }
    if (n == 0) continue;
    for (long v0 = z0 * 64L + wid * 16; v0 < len; v0 += zn * 64L) {
      const bf16_t* vr = a.vecs + (b0 + min(v0 + r16, (long)len - 1)) * a.d + 8 * g;
      bf16x8 x[NF];
      auto load = [&](int c0) {
#pragma unroll
        for (int s = 0; s < NF; ++s) {
          x[s] = bf16x8{};
          if (c0 + 32 * s + 8 * g < a.d) x[s] = *(const bf16x8*)(vr + c0 + 32 * s);
        }
      };
      load(0);
      long id[4];
      float sq[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {  // of the vectors whose scores the lane holds
        const long at = b0 + min(v0 + 4 * g + i, (long)len - 1);
        id[i] = a.ids[at];
        sq[i] = a.l2 ? a.sqnorm[at] : 0.f;
      }
      for (int t = 0; t < n; t += 16) {
        const long pr = pair_of(min(t + r16, n - 1));
        const bf16_t* qr = a.q + pr / a.nprobe * a.d + 8 * g;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        float qq = 0.f;
        for (int c0 = 0; c0 < a.d; c0 += 32 * NF) {
          if (a.d > 32 * NF && (t > 0 || c0 > 0)) load(c0);
          bf16x8 y[NF];
#pragma unroll
          for (int s = 0; s < NF; ++s) {
            y[s] = bf16x8{};
            if (c0 + 32 * s + 8 * g < a.d) y[s] = *(const bf16x8*)(qr + c0 + 32 * s);
          }
#pragma unroll
          for (int s = 0; s < NF; ++s)
            if (c0 + 32 * s < a.d) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[s], y[s], acc, 0, 0, 0);
          if (a.l2) {
#pragma unroll
            for (int s = 0; s < NF; ++s) {
              float f[8];
              unpack8(__builtin_bit_cast(uint4, y[s]), f);
#pragma unroll
              for (int e = 0; e < 8; ++e) qq = fmaf(f[e], f[e], qq);
            }
          }
        }
        if (a.l2) {
          qq += __shfl_xor(qq, 16, 64);
          qq += __shfl_xor(qq, 32, 64);
        }
        // acc[i]: vector v0 + 4 g + i, query r16 of the sixteen
        if (t + r16 < n && (BY_LIST || r16 == 0)) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const long j = v0 + 4 * g + i;
            if (j < len) {
              a.cand[pr * a.maxlen + j] = a.l2 ? 2.f * acc[i] - sq[i] - qq : acc[i];
              a.cand_ids[pr * a.maxlen + j] = id[i];
            }
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

extern "C" int rt_ivf_scan(const void* q, int nq, int d, const int* probes, int nprobe, int nlist, const int* lstart,
                           const int* lsize, const void* vecs, const long* ids, const float* sqnorm, int l2,
                           int maxlen, float* cand, long* cand_ids, hipStream_t stream) {
  if (d % 8 != 0 || (l2 && !sqnorm) || (uintptr_t)q % 16 || (uintptr_t)vecs % 16) return -1;
  if (nq == 0 || nprobe == 0) return 0;
  if (maxlen <= 0) return 0;
  const ScanArgs a{(const bf16_t*)q, nq, d, probes, nprobe, nlist, lstart, lsize, (const bf16_t*)vecs, ids, sqnorm, l2, maxlen, cand, cand_ids};
  // A list's vectors are read once for all its queries as soon as a list has one on average, or where lists are long: a few
  // then hold most of the vectors, and every query probes them. Search, us, thread per vector / by probe / by list, longest
  // lists of 1000 to 4000: 12 queries 125 / 105 / 81, 20 queries 66 / 77 / 60, 24 queries 118 / 148 / 68; by probe it stays where
  // they are short (8 queries 42 / 42). Long lists go round some thousand workgroups.
  const bool by_list = (long)nq * nprobe >= nlist || (nq > 4 && maxlen > 1024) || (nq > 1 && maxlen > 4096) || nq > 65535;
  const long pieces = (maxlen + 63L) / 64, most = by_list ? 64 : std::max(8192L / ((long)nprobe * nq), 8L);
  const dim3 grid = by_list ? dim3(nlist + 1, 1, (unsigned)std::min(pieces, most)) : dim3(nprobe, nq, (unsigned)std::min(pieces, most));
#define SCAN(NF)                                                                                   \
  do {                                                                                             \
    if (by_list) hipLaunchKernelGGL((ivf_scan_kernel<NF, true>), grid, dim3(256), 0, stream, a);   \
    else hipLaunchKernelGGL((ivf_scan_kernel<NF, false>), grid, dim3(256), 0, stream, a);          \
  } while (0)
  if (d <= 384) SCAN(12);
  else SCAN(24);
#undef SCAN
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
