// Products of few rows with weights of an encoder's size, for gfx950: y = act(x W^T + bias), where x may still be LN(d + res).
// For encoders that encoder_few.hip does not take (heads of 128, rows of 1024 with 4096 between): a query is four such products a layer, each
// a few hundred KB of weights: what they take is launch, one trip to memory and the reduction over K, not bandwidth.
//
// K is summed in the parts, and the parts in the order, of the kernel that ops.gemm takes for the shape (see Args), so that the
// bits are that kernel's: a text's embedding does not depend on the way it went. The 8 waves of a workgroup are parts x row tiles
// x column groups of 16; a wave has most of its weights (and of x) in flight at once, and partial sums meet in LDS. They come by
// LDS-DMA, eight lanes to a row's 128 B, into places of the wave's own: loads straight in MFMA order, whose adjacent lanes are in
// different rows, keep the CU's address path busy for 64 cycles each, these for 16 (profiles/calls/load_order.txt). With a norm ahead every
// workgroup normalises the rows itself, two or four to a wave, over the weights' trip (12 KB from L2, where a kernel of its own costs a launch and
// another trip); workgroup 0 also writes them.
// Bound by latency. 15 rows, us, gemm_decode_kernel -> MFMA-order loads -> this: 1152 x 384 5.2 -> 4.5 -> 4.0, 384 x 384 (4.5 -> 4.0),
// 384 x 1536 9.8 -> 5.8 -> 4.4, and 2.9 of the norm with it. MiniLM over 15 / 32 rows 157 -> 141 / 201 -> 167, mpnet-base (and with
// wave_reduce) 428 -> 345 / 620 -> 452. From 33 rows on gemm_mid_kernel's tiles are ahead.
#include "rt_common.h"
#include "rt_few_head.h"
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
  int parts, grp;  // K parts of whole 64s, part i from i (K / 64) / parts on; summed in groups of grp, then the groups in order
  int ks, rs;      // of the 8 waves: over parts, over row tiles (powers of two; the rest over column groups of 16)
  float eps;
};

typedef __attribute__((address_space(3))) void lds_void;

// no template: hipcc's host pass drops kernels that call the builtin with dependent arguments
__device__ __forceinline__ void dma16(const bf16_t* from, char* to) { __builtin_amdgcn_global_load_lds(from, (lds_void*)to, 16, 0, 0); }

// RT: row tiles of 16 a wave; NW: 16-B vectors of a row a lane normalises (0: no norm ahead), of up to 16 TR rows
template <int RT, int NW, int TR>
__global__ __launch_bounds__(512, 2) void few_rows_kernel(Args p) {
  constexpr int LDX = NW * 512 + 8;  // K <= 512 NW; an odd number of 16-B chunks where K is a multiple of 16
  // D chunks of 64 k under way a wave: 16 weight rows, and without a norm 16 RT rows of x, of 128 B each
  constexpr int XT = NW ? 0 : RT, CH = (1 + XT) * 2048, D = NW == 0 ? (RT == 1 ? 4 : 3) : NW * TR > 2 ? 4 : 6;
  __shared__ __attribute__((aligned(16))) char ring[8 * D * CH];
  __shared__ __attribute__((aligned(16))) bf16_t xs[NW ? TR * 16 * LDX : 8];
  __shared__ f32x4 red[16][64];  // [part][column group][row tile]
  // <2, 0, 0> takes the CU's LDS to the last byte: without a norm nothing names xs, and it gets no place
  static_assert(sizeof(ring) + (NW ? sizeof(xs) : 0) + sizeof(red) <= 160 * 1024, "the LDS of a CU");
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const int nc = p.K / 64, CG = 8 / (p.ks * p.rs), RTS = p.rs * RT;  // column groups, row tiles of the workgroup
  const int ks = wid % p.ks, rs = wid / p.ks % p.rs, cg = wid / (p.ks * p.rs);
  const int n0 = (blockIdx.x * CG + cg) * 16;
  const bool on = n0 < p.N && rs * RT * 16 < p.M;
  auto begin = [&](int part) { return part * nc / p.parts; };  // in chunks
  // load j of 8 rows: lane -> row 8 j + lane / 8, 16-B slot lane % 8 of it holding k chunk slot ^ (row / 2 % 8)
  const bf16_t *wp[2], *xp[XT ? 2 * XT : 1];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int row = 8 * j + (lane >> 3), kc = ((lane & 7) ^ (row >> 1)) * 8;
    wp[j] = p.w + (long)min(n0 + row, p.N - 1) * p.ldw + kc;
#pragma unroll
    for (int t = 0; t < XT; ++t) xp[2 * t + j] = p.x + (long)min(16 * (rs * RT + t) + row, p.M - 1) * p.ldx + kc;
  }
  char* const mine = ring + wid * D * CH;
  int c0 = 0, c1 = 0;
  if (on && ks < p.parts) { c0 = begin(ks); c1 = begin(ks + 1); }
  auto ask = [&](int c) {
#pragma unroll
    for (int k = 0; k < D; ++k)
      if (c + k < c1)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          dma16(wp[j] + (c + k) * 64, mine + k * CH + j * 1024);
#pragma unroll
          for (int t = 0; t < XT; ++t) dma16(xp[2 * t + j] + (c + k) * 64, mine + k * CH + (2 + 2 * t + j) * 1024);
        }
  };
  if constexpr (NW > 0) {
    // rows of the norm: the arithmetic of norm_rows_kernel
    const int nv = p.K / 8;
    constexpr int RW = TR * 2;  // rows of a wave
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
    ask(c0);  // behind the rows, which the norm waits for
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
  if constexpr (NW == 0) ask(c0);
  for (int part = ks; part < p.parts; part += p.ks) {
    if (part > ks && on) { c0 = begin(part); c1 = begin(part + 1); }
    f32x4 acc[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int c = c0; c < c1; c += D) {
      if (c > c0 || part > ks) ask(c);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      bf16x8 wf[D][2], xf[D][2][RT];
#pragma unroll
      for (int k = 0; k < D; ++k)  // all places, asked for or not: the reads go out together
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const char* const img = mine + k * CH + r16 * 128 + (((4 * h + g) ^ (r16 >> 1)) << 4);
          wf[k][h] = *(const bf16x8*)img;
#pragma unroll
          for (int t = 0; t < RT; ++t) {
            const int row = 16 * (rs * RT + t) + r16, col = min(c + k, c1 - 1) * 64 + h * 32 + 8 * g;
            xf[k][h][t] = *(const bf16x8*)(NW > 0 ? (const char*)(xs + row * LDX + col) : img + (1 + t) * 2048);
          }
        }
#pragma unroll
      for (int k = 0; k < D; ++k)
        if (c + k < c1)
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < RT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[k][h], xf[k][h][t], acc[t], 0, 0, 0);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the next chunks take their place
    }
    // acc[t][e]: row 16 (rs RT + t) + r16, column n0 + 4 g + e
#pragma unroll
    for (int t = 0; t < RT; ++t) red[(part * CG + cg) * RTS + rs * RT + t][lane] = acc[t];
  }
  __syncthreads();
  for (int o = wid; o < CG * RTS; o += 8) {
    const int t = o % RTS, row = 16 * t + r16, col = (blockIdx.x * CG + o / RTS) * 16 + 4 * g;
    if (row >= p.M || col >= p.N) continue;
    f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int b = 0; b < p.parts; b += p.grp) {
      f32x4 u = red[b * CG * RTS + o][lane];
      for (int k = 1; k < p.grp; ++k) u += red[(b + k) * CG * RTS + o][lane];
      v = p.parts == p.grp ? u : v + u;
    }
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
// after each term, as embed_kernel and an addition do; the norm is norm_rows_kernel's without a residual. `unset` and `head`
// (see encoder_few.hip): memory that is set to ones, and a FewHead that is written; with them the rows hold no word of ones, and lie in
// column groups of 16, T up to a multiple of 16 of them each. The arguments fill two lines: with a third it took 4.0 us instead of 3.6.
template <int NW>
__global__ __launch_bounds__(256) void embed_norm_rows_kernel(const bf16_t* __restrict__ word, const long* __restrict__ ids,
                                                              const bf16_t* __restrict__ pos, const long* __restrict__ pids,
                                                              const bf16_t* __restrict__ type, const bf16_t* __restrict__ w,
                                                              const bf16_t* __restrict__ b, bf16_t* __restrict__ y, int T, int H,
                                                              float eps, int n_unset, uint4* __restrict__ unset,
                                                              FewHead* __restrict__ head, unsigned* report, unsigned tries) {
  const int lane = threadIdx.x & 63, nv = H / 8;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n_unset; i += (long)gridDim.x * 256) unset[i] = make_uint4(~0u, ~0u, ~0u, ~0u);
  if (head && blockIdx.x == gridDim.x - 1 && threadIdx.x < 64) {  // a workgroup that has no rows, as a rule
    constexpr int TRIES = offsetof(FewHead, tries) / 4, REPORT = offsetof(FewHead, report) / 4;
    const int t = threadIdx.x;
    const unsigned long to = (unsigned long)report;
    ((unsigned*)head)[t] = t == 0 ? tries == 0 : t == TRIES ? tries : t == REPORT ? (unsigned)to : t == REPORT + 1 ? (unsigned)(to >> 32) : 0;
  }
  for (long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6); row < T; row += (long)gridDim.x * 4) {
    RT_ASSERT(ids[row] >= 0 && pids[row] >= 0);
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
        uint4 q = pack8(o);
        if (head) {
          uint32_t* const u = (uint32_t*)&q;
#pragma unroll
          for (int e = 0; e < 4; ++e) u[e] = u[e] == ~0u ? 0xfffefffeu : u[e];
        }
        *(uint4*)(y + (head ? ((c >> 1) * ((T + 15) & ~15) + row) * 16 + (c & 1) * 8 : row * H + c * 8)) = q;
      }
    }
  }
}

}  // namespace fr
}  // namespace rt

using namespace rt;

// y = act(x w^T + bias), or act(LN(x + res) w^T + bias) with LN(x + res) to xo (lw given; K <= 1024); M <= 32, act 0 or 2
// (GELU). N % 16 == 0, K % 64 == 0; operands 16-B aligned, leading dimensions multiples of 8; up to 8 parts, up to 16 rows 16,
// a multiple of grp. -1: not for this kernel.
extern "C" int rt_few_rows(const void* x, long ldx, const void* res, long ldr, const void* lw, const void* lb, void* xo, const void* w,
                           long ldw, const void* bias, void* y, long ldy, int M, int N, int K, int act, float eps, int parts, int grp,
                           hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 32 || N % 16 || K < 64 || K % 64 || (act != 0 && act != 2) || (lw && (K > 1024 || !lb || !res || !xo))) return -1;
  if (parts < 1 || parts > (M <= 16 ? 16 : 8) || grp < 1 || parts % grp) return -1;
  fr::Args p;
  p.x = (const bf16_t*)x; p.ldx = ldx; p.res = (const bf16_t*)res; p.ldr = ldr;
  p.lw = (const bf16_t*)lw; p.lb = (const bf16_t*)lb; p.xo = (bf16_t*)xo;
  p.w = (const bf16_t*)w; p.ldw = ldw; p.bias = (const bf16_t*)bias; p.y = (bf16_t*)y; p.ldy = ldy;
  p.M = M; p.N = N; p.K = K; p.act = act; p.eps = eps; p.parts = parts; p.grp = grp;
  const int tiles = M <= 16 ? 1 : 2;
  p.ks = parts > 4 ? 8 : parts > 2 ? 4 : parts;
  p.rs = std::min(tiles > 1 ? 4 : 1, 8 / p.ks);  // 17..32 rows in one part: rather idle waves than half the workgroups
  const int rt = std::max(tiles / p.rs, 1), cols = 16 * (8 / (p.ks * p.rs)), nw = lw ? (K <= 512 ? 1 : 2) : 0;
  if (nw && rt != 1) return -1;
  const dim3 grid((N + cols - 1) / cols), block(512);
#define FR(R, W, T) hipLaunchKernelGGL((fr::few_rows_kernel<R, W, T>), grid, block, 0, stream, p)
  if (nw == 1) { if (tiles == 1) FR(1, 1, 1); else FR(1, 1, 2); }
  else if (nw == 2) { if (tiles == 1) FR(1, 2, 1); else FR(1, 2, 2); }
  else if (rt == 1) FR(1, 0, 0);
  else FR(2, 0, 0);
#undef FR
  RT_LAUNCH_CHECK();
  return 0;
}

// y[t] = LN(word[ids[t]] + pos[pids[t]] (+ type)); H % 8 == 0, H <= 1024. unset_bytes: a multiple of 16
extern "C" int rt_embed_norm_rows(const void* word, const long* ids, const void* pos, const long* pids, const void* type,
                                  const void* w, const void* b, void* y, int T, int H, float eps, void* unset, long unset_bytes,
                                  void* head, unsigned* report, unsigned tries, hipStream_t stream) {
  if (T <= 0) return 0;
  if (H % 8 || H > 1024 || unset_bytes / 16 > 0x7fffffffL) return -1;
  const long n = unset ? unset_bytes / 16 : 0;
  const dim3 grid((unsigned)std::min(std::max((T + 3L) / 4, (n + 255) / 256), 2048L)), block(256);
#define EN(W)                                                                                                                 \
  hipLaunchKernelGGL(fr::embed_norm_rows_kernel<W>, grid, block, 0, stream, (const bf16_t*)word, ids, (const bf16_t*)pos, pids, \
                     (const bf16_t*)type, (const bf16_t*)w, (const bf16_t*)b, (bf16_t*)y, T, H, eps, (int)n, (uint4*)unset, (FewHead*)head, \
                     report, tries)
  if (H <= 512) EN(1); else EN(2);
#undef EN
  RT_LAUNCH_CHECK();
  return 0;
}
