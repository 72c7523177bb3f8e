// Products of few rows (M <= 64) with weights of an encoder's size, for gfx950: y = act(x W^T + bias), where x may still be
// LN(d + res). One query through all-MiniLM-L6-v2 is 24 such products of about 15 rows, each a few hundred KB of weights: what
// they take is launch, one trip to memory and the reduction over K, not bandwidth.
//
// A workgroup is 8 waves over 16 (K >= 512) or 32 columns; 8 (4) waves split K, so that a wave has 3 to 6 steps of 32 and all of
// its weight loads (MFMA fragments, 16 B a lane straight from the row-major weight) in flight at once. With a norm ahead every
// workgroup normalises the rows itself, two or four to a wave, under those loads (12 KB from L2, where a kernel of its own costs
// a launch and another trip); workgroup 0 also writes them. Partial sums meet in LDS. Bound by latency. 15 rows, us,
// gemm_decode_kernel and the norm ahead -> this: 1152 x 384 6.1 + 2.9 -> 5.2, 1536 x 384 with GELU 6.3 + 2.9 -> 5.9,
// 384 x 384 5.7 -> 4.4, 384 x 1536 11.3 -> 5.7.
#include "rt_common.h"
#include "rt_gelu.h"

#include <algorithm>

namespace rt {
namespace fr {

struct Args {
  const bf16_t* x; long ldx;                // [M, K]; NORM: d
  const bf16_t* res; const bf16_t* lw; const bf16_t* lb; bf16_t* xo; long ldr;  // NORM: res and xo [M, K] (rows ldr)
  const bf16_t* w; long ldw; const bf16_t* bias;  // [N, K], [N] or null
  bf16_t* y; long ldy;
  int M, N, K, act;
  float eps;
};

// RT: row tiles of 16; NW: 16-B vectors of a row a lane normalises (0: no norm ahead)
template <int RT, int NW>
__global__ __launch_bounds__(512) void few_rows_kernel(Args p) {
  constexpr int LDX = NW * 512 + 8;  // K <= 512 NW; an odd number of 16-B chunks where K is a multiple of 16
  __shared__ __attribute__((aligned(16))) bf16_t xs[NW ? RT * 16 * LDX : 8];
  __shared__ f32x4 red[8][RT][64];
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const int steps = p.K / 32, CG = steps >= 16 ? 1 : 2, KS = 8 / CG;
  const int cg = wid / KS, ks = wid % KS;
  const int n0 = (blockIdx.x * CG + cg) * 16;
  const int s0 = ks * steps / KS, s1 = n0 < p.N ? (ks + 1) * steps / KS : s0;
  const bf16_t* const wp = p.w + (long)min(n0 + r16, p.N - 1) * p.ldw + 8 * g;
  constexpr int D = 6;  // weight fragments in flight
  bf16x8 wf[D];
#pragma unroll
  for (int k = 0; k < D; ++k)
    if (s0 + k < s1) wf[k] = *(const bf16x8*)(wp + (s0 + k) * 32);

  if constexpr (NW > 0) {
    // rows of the norm: the arithmetic of norm_rows_kernel
    const int nv = p.K / 8;
    constexpr int RW = RT * 2;  // rows of a wave
    uint4 a[RW][NW], b[RW][NW];
#pragma unroll
    for (int k = 0; k < RW; ++k)
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        const long row = min(wid + 8 * k, p.M - 1);
        const int c = lane + 64 * i;
        if (c < nv) {
          a[k][i] = *(const uint4*)(p.x + row * p.ldx + c * 8);
          b[k][i] = *(const uint4*)(p.res + row * p.ldr + c * 8);
        }
      }
    uint4 wr[NW], br[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i)
      if (lane + 64 * i < nv) {
        wr[i] = *(const uint4*)(p.lw + (lane + 64 * i) * 8);
        br[i] = *(const uint4*)(p.lb + (lane + 64 * i) * 8);
      }
#pragma unroll
    for (int k = 0; k < RW; ++k) {
      const int row = wid + 8 * k;
      float v[NW][8], s[NW];
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        s[i] = 0.f;
        if (lane + 64 * i < nv) {
          float r[8];
          unpack8(a[k][i], v[i]);
          unpack8(b[k][i], r);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            v[i][e] = bf2f(f2bf(v[i][e] + r[e]));
            s[i] += v[i][e];
          }
        }
      }
      auto total = [&]() {
        float t = 0.f;
#pragma unroll
        for (int i = 0; i < NW; ++i) t += wave_sum(s[i]);
        return t;
      };
      const float mean = total() / p.K;
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        s[i] = 0.f;
        if (lane + 64 * i < nv)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float d = v[i][e] - mean;
            s[i] += d * d;
          }
      }
      const float rstd = rsqrtf(total() / p.K + p.eps);
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        const int c = lane + 64 * i;
        if (c < nv) {
          float wv[8], bv[8], o[8];
          unpack8(wr[i], wv);
          unpack8(br[i], bv);
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = fmaf((v[i][e] - mean) * rstd, wv[e], bv[e]);
          const uint4 q = pack8(o);
          *(uint4*)(xs + row * LDX + c * 8) = q;
          if (blockIdx.x == 0 && row < p.M) *(uint4*)(p.xo + row * p.ldr + c * 8) = q;
        }
      }
    }
    __syncthreads();
  }
  f32x4 acc[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s = s0; s < s1; s += D) {
#pragma unroll
    for (int k = 0; k < D; ++k) {
      if (s > s0 && s + k < s1) wf[k] = *(const bf16x8*)(wp + (s + k) * 32);
    }
    bf16x8 xf[D][RT];
#pragma unroll
    for (int k = 0; k < D; ++k)
      if (s + k < s1)
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          const int row = 16 * t + r16, col = (s + k) * 32 + 8 * g;
          if constexpr (NW > 0) xf[k][t] = *(const bf16x8*)(xs + row * LDX + col);
          else xf[k][t] = *(const bf16x8*)(p.x + (long)min(row, p.M - 1) * p.ldx + col);
        }
#pragma unroll
    for (int k = 0; k < D; ++k)
      if (s + k < s1)
#pragma unroll
        for (int t = 0; t < RT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[k], xf[k][t], acc[t], 0, 0, 0);
  }
  // acc[t][e]: row 16 t + r16, column n0 + 4 g + e
#pragma unroll
  for (int t = 0; t < RT; ++t) red[wid][t][lane] = acc[t];
  __syncthreads();
  for (int o = wid; o < CG * RT; o += 8) {
    const int c = o / RT, t = o % RT, row = 16 * t + r16, col = (blockIdx.x * CG + c) * 16 + 4 * g;
    if (row >= p.M || col >= p.N) continue;
    f32x4 v = red[c * KS][t][lane];
    for (int k = 1; k < KS; ++k) v += red[c * KS + k][t][lane];
    if (p.bias) {
      const uint2 b = *(const uint2*)(p.bias + col);
      v += f32x4{__uint_as_float(b.x << 16), __uint_as_float(b.x & 0xffff0000u), __uint_as_float(b.y << 16), __uint_as_float(b.y & 0xffff0000u)};
    }
    const uint2 q = p.act == 2 ? make_uint2(gelu2_bf16(v[0], v[1]), gelu2_bf16(v[2], v[3]))
                               : make_uint2(pack2bf(v[0], v[1]), pack2bf(v[2], v[3]));
    *(uint2*)(p.y + (long)row * p.ldy + col) = q;
  }
}

// x[t] = LN(bf16(word[id] + pos[p]) + type): the embedding of an encoder in one pass, a wave a row. The sum is rounded to bf16
// after each term, as embed_kernel and an addition do; the norm is norm_rows_kernel's without a residual.
template <int NW>
__global__ __launch_bounds__(256) void embed_norm_rows_kernel(const bf16_t* __restrict__ word, const long* __restrict__ ids,
                                                              const bf16_t* __restrict__ pos, const long* __restrict__ pids,
                                                              const bf16_t* __restrict__ type, const bf16_t* __restrict__ w,
                                                              const bf16_t* __restrict__ b, bf16_t* __restrict__ y, int T, int H,
                                                              float eps) {
  const int lane = threadIdx.x & 63, nv = H / 8;
  for (long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6); row < T; row += (long)gridDim.x * 4) {
    const bf16_t* const wp = word + ids[row] * H;
    const bf16_t* const pp = pos + pids[row] * H;
    float v[NW][8], s[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const int c = lane + 64 * i;
      s[i] = 0.f;
      if (c < nv) {
        float q[8];
        unpack8(*(const uint4*)(wp + c * 8), v[i]);
        unpack8(*(const uint4*)(pp + c * 8), q);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = bf2f(f2bf(v[i][e] + q[e]));
        if (type) {
          unpack8(*(const uint4*)(type + c * 8), q);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[i][e] = bf2f(f2bf(v[i][e] + q[e]));
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) s[i] += v[i][e];
      }
    }
    auto total = [&]() {
      float t = 0.f;
#pragma unroll
      for (int i = 0; i < NW; ++i) t += wave_sum(s[i]);
      return t;
    };
    const float mean = total() / H;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      s[i] = 0.f;
      if (lane + 64 * i < nv)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float d = v[i][e] - mean;
          s[i] += d * d;
        }
    }
    const float rstd = rsqrtf(total() / H + eps);
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const int c = lane + 64 * i;
      if (c < nv) {
        float wv[8], bv[8], o[8];
        unpack8(*(const uint4*)(w + c * 8), wv);
        unpack8(*(const uint4*)(b + c * 8), bv);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = fmaf((v[i][e] - mean) * rstd, wv[e], bv[e]);
        *(uint4*)(y + row * H + c * 8) = pack8(o);
      }
    }
  }
}

}  // namespace fr
}  // namespace rt

using namespace rt;

// y = act(x w^T + bias), or act(LN(x + res) w^T + bias) with LN(x + res) to xo (lw given; M <= 32, K <= 1024); act 0 or 2
// (GELU). M <= 64, N % 16 == 0, K % 32 == 0; operands 16-B aligned, leading dimensions multiples of 8. -1: not for this kernel.
extern "C" int rt_few_rows(const void* x, long ldx, const void* res, long ldr, const void* lw, const void* lb, void* xo, const void* w,
                           long ldw, const void* bias, void* y, long ldy, int M, int N, int K, int act, float eps, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 64 || N % 16 || K < 32 || K % 32 || (act != 0 && act != 2) || (lw && (M > 32 || K > 1024 || !lb || !res || !xo))) return -1;
  fr::Args p;
  p.x = (const bf16_t*)x; p.ldx = ldx; p.res = (const bf16_t*)res; p.ldr = ldr;
  p.lw = (const bf16_t*)lw; p.lb = (const bf16_t*)lb; p.xo = (bf16_t*)xo;
  p.w = (const bf16_t*)w; p.ldw = ldw; p.bias = (const bf16_t*)bias; p.y = (bf16_t*)y; p.ldy = ldy;
  p.M = M; p.N = N; p.K = K; p.act = act; p.eps = eps;
  const int cols = K / 32 >= 16 ? 16 : 32;
  const dim3 grid((N + cols - 1) / cols), block(512);
  const int rt = (M + 15) / 16, nw = lw ? (K <= 512 ? 1 : 2) : 0;
#define FR(R, W) hipLaunchKernelGGL((fr::few_rows_kernel<R, W>), grid, block, 0, stream, p)
  switch (rt * 4 + nw) {
    case 4: FR(1, 0); break;
    case 5: FR(1, 1); break;
    case 6: FR(1, 2); break;
    case 8: FR(2, 0); break;
    case 9: FR(2, 1); break;
    case 10: FR(2, 2); break;
    case 12: FR(3, 0); break;
    case 16: FR(4, 0); break;
    default: return -1;
  }
#undef FR
  RT_LAUNCH_CHECK();
  return 0;
}

// y[t] = LN(word[ids[t]] + pos[pids[t]] (+ type)); H % 8 == 0, H <= 1024
extern "C" int rt_embed_norm_rows(const void* word, const long* ids, const void* pos, const long* pids, const void* type,
                                  const void* w, const void* b, void* y, int T, int H, float eps, hipStream_t stream) {
  if (T <= 0) return 0;
  if (H % 8 || H > 1024) return -1;
  const dim3 grid(std::min((T + 3) / 4, 2048)), block(256);
  if (H <= 512)
    hipLaunchKernelGGL(fr::embed_norm_rows_kernel<1>, grid, block, 0, stream, (const bf16_t*)word, ids, (const bf16_t*)pos, pids,
                       (const bf16_t*)type, (const bf16_t*)w, (const bf16_t*)b, (bf16_t*)y, T, H, eps);
  else
    hipLaunchKernelGGL(fr::embed_norm_rows_kernel<2>, grid, block, 0, stream, (const bf16_t*)word, ids, (const bf16_t*)pos, pids,
                       (const bf16_t*)type, (const bf16_t*)w, (const bf16_t*)b, (bf16_t*)y, T, H, eps);
  RT_LAUNCH_CHECK();
  return 0;
}
