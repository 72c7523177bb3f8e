// A sentence encoder's layers over up to 64 rows (a query, a few short texts) in ONE launch, for gfx950.
//
// Launch by launch such a forward is a chain of 5 dependent kernels a layer, each of which waits for its launch, its weights' and
// its rows' trip to memory, and computes for well under a microsecond. Here it is a list of tasks (16 rows of 16 to 64 columns of a
// product with the norm ahead, attention of a few heads, a text's pooling) in an order in which a task needs earlier ones only.
// Workgroups take tasks off a counter, one ahead; a task's weights are on their way to LDS before its rows exist, so what is left
// of the chain is the exchange between workgroups (0.5 us at best) and the arithmetic (the norm 0.7, the others 0.3 to 1).
// Rows go from task to task through memory that holds no result yet: the launch ahead (the embedding) fills it with words no
// result has (two bf16 of all ones, a NaN that a store replaces by another), and a reader asks until none is left. That takes
// no flag, no wait for the stores ahead of one, and no order between words; each word is written once. Reads and writes of it are
// device-scope accesses (sc1). Asking brings a line into the L2 of every XCD that asks, and a store has to take it away from all of
// them: so a wave stores its 16 x 16 results as 512 bytes in a row, lines that nobody else writes (with rows side by side, several
// stores to a line, an exchange took 0.7 to 2 us). Rows that feed a product without a norm lie as the MFMA takes them, and go from memory
// to its operands. Asking more cheaply first (one word, or one wave of a workgroup), or all on one XCD, took longer (106 -> 115, 127).
// A workgroup waits only for tasks that running workgroups have taken before it, so the launch ends with whatever number of them the
// device runs at a time, beside other launches of its kind too; a wait of seconds gives up all the same: the results are NaN, and a word of
// host memory says so.
//
// The arithmetic, its parts of K and their order are few_rows.hip's, attn_packed_kernel's and pool_norm_kernel's: the same bits.
// us, launch by launch -> this, with the embedding: MiniLM over 15 / 32 / 64 rows 133 -> 86 / 158 -> 103 / 190 -> 128, mpnet-base 344 -> 232 /
// 451 -> 329 / 517 -> 475.
#include "rt_common.h"
#include "rt_gelu.h"
#include "rt_few_head.h"

#include <algorithm>
#include <type_traits>

namespace rt {
namespace ef {

constexpr int MAX_LAYERS = 24, WAVES = 8, CHUNK = 2048;  // CHUNK: 16 weight rows x 64 k
constexpr int RING = 48, VPLACE = 8192, UNITS = 4;       // chunks of weights in LDS; a wave's place for values, such waves of a task
constexpr int LDS = 160 * 1024 - 128;                    // a CU's, but for the kernel's own few words: one workgroup a CU
constexpr int RED = 68;                                  // a 16 x 16 result of a part: lane + lane / 16
constexpr uint32_t NONE = 0xffffffffu;                   // no result yet

struct Product {
  int N, K, parts, grp;  // parts of K and their groups: see few_rows.hip
  int ks, cg;            // waves over parts x column groups of 16 (the rest idle)
  int tasks;
};
struct Args {
  const bf16_t* w[MAX_LAYERS][12];  // qkv, o, ln1, fc1, fc2, ln2: a weight and a bias each
  Product p[4];                     // qkv, o, fc1, fc2
  int M, H, F, B, L, heads, tiles;  // tiles: of 16 rows
  int units, att_tasks, layer_tasks, tasks;  // units: heads of a task of attention
  float eps, scale_log2;
  const float* rel_bias; int rb_L;
  const long* off;
  bf16_t* ex;          // rows on their way: x0, then a layer's qkv, a, d1, x1, f, d2, x2; see place()
  unsigned ex_bytes;
  unsigned* next;      // the next task: FewHead, ahead of the rows
  int normalize;
  float* out; const long* to; long out_rows;
  int lds_x, lds_red;  // byte offsets behind the ring
};

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
__device__ __forceinline__ void dma16(const bf16_t* from, char* to) { __builtin_amdgcn_global_load_lds(from, (lds_void*)to, 16, 0, 0); }

constexpr int SC1 = 16;
__device__ __forceinline__ bool there(const u32x4& v) { return v[0] != NONE && v[1] != NONE && v[2] != NONE && v[3] != NONE; }
// v[i] = load(i) until every lane's words are results. Waits are bounded: who has asked in vain `tries` times says so to the launch, which
// gives up (each waiting wave looks every 1024 times), and to the host. Both are beside `lost` and not arguments: the kernel has no register
// for them.
template <int N, typename F>
__device__ __forceinline__ void await(unsigned* lost, u32x4 (&v)[N], F load) {
  for (int tries = 0;; ++tries) {
    asm volatile("" ::: "memory");  // asked anew each time
    bool ok = true;
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = load(i);
#pragma unroll
    for (int i = 0; i < N; ++i) ok = ok && there(v[i]);
    if (__all(ok)) break;
    __builtin_amdgcn_s_sleep(1);
    if ((tries & 1023) == 1023) {
      if (__hip_atomic_load(lost, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
      typedef __attribute__((address_space(4))) const FewHead Head;  // written by the launch before: by scalar loads, into no vector register
      Head* const h = (Head*)(uintptr_t)(lost - 16);
      if ((unsigned)tries >= h->tries) {
        __hip_atomic_store(lost, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(h->report, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
  }
}
__device__ __forceinline__ uint32_t word_of(uint32_t w) { return w == NONE ? 0xfffefffeu : w; }
__device__ __forceinline__ void put8(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t lo, uint32_t hi) {
  __builtin_amdgcn_raw_buffer_store_b64(u32x2{word_of(lo), word_of(hi)}, r, off, 0, SC1);
}
// Byte of a row's column in a block of rows on their way: what a wave stores at once (16 x 16 results) is 512 bytes in a row, whole lines
// of memory that nobody else writes. Rows that are normed lie in column groups of 16, the others (a, f) as the MFMA takes them.
__device__ __forceinline__ uint32_t place(int tiles, int row, int col) { return ((col >> 4) * 16 * tiles + row) * 32 + (col & 15) * 2; }
__device__ __forceinline__ uint32_t place_op(int tiles, int row, int col) {
  return ((col >> 5) * tiles + (row >> 4)) * 1024 + (col >> 3 & 3) * 256 + (row & 15) * 16 + (col & 7) * 2;
}
// row and first column of the four results at 8 lane .. of those 512 bytes, and the lane whose registers they come from
__device__ __forceinline__ int row_at(int lane, bool op) { return op ? lane >> 1 & 15 : lane >> 2; }
__device__ __forceinline__ int quad_at(int lane, bool op) { return op ? (lane >> 5) * 2 + (lane & 1) : lane & 3; }

// LN(d + res) of up to 16 rows from `first` on, two of them a wave, the arithmetic of norm_rows_kernel; to LDS
template <int NW>
__device__ __forceinline__ void norm_rows(unsigned* lost, __amdgpu_buffer_rsrc_t ex, uint32_t d, uint32_t res, const bf16_t* lw, const bf16_t* lb,
                                          int H, int tiles, int first, int n, float eps, char* xs, int wid, int lane) {
  if (2 * wid >= n) return;
  const int nv = H / 8;
  uint4 wr[NW], br[NW];
  int at[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    at[i] = min(lane + 64 * i, nv - 1);
    wr[i] = *(const uint4*)(lw + at[i] * 8);
    br[i] = *(const uint4*)(lb + at[i] * 8);
  }
  constexpr int RW = 2;
  u32x4 dv[RW * NW], rv[RW * NW];
  auto load = [&](uint32_t from, int j) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
        ex, from + place(tiles, first + min(RW * wid + j / NW, n - 1), at[j % NW] * 8), 0, SC1));
  };
  await(lost, rv, [&](int j) { return load(res, j); });  // there for a while
  await(lost, dv, [&](int j) { return load(d, j); });
  float v[RW][NW][8], s[RW][NW], mean[RW], rstd[RW];
#pragma unroll
  for (int k = 0; k < RW; ++k)
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      s[k][i] = 0.f;
      float r[8];
      unpack8(__builtin_bit_cast(uint4, dv[k * NW + i]), v[k][i]);
      unpack8(__builtin_bit_cast(uint4, rv[k * NW + i]), r);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        v[k][i][e] = bf2f(f2bf(v[k][i][e] + r[e]));
        s[k][i] += v[k][i][e];
      }
      if (lane + 64 * i >= nv) s[k][i] = 0.f;
    }
  auto total = [&](int k) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) t += wave_sum(s[k][i]);
    return t;
  };
#pragma unroll
  for (int k = 0; k < RW; ++k) mean[k] = total(k) / H;
#pragma unroll
  for (int k = 0; k < RW; ++k)
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      s[k][i] = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float dd = v[k][i][e] - mean[k];
        s[k][i] += dd * dd;
      }
      if (lane + 64 * i >= nv) s[k][i] = 0.f;
    }
#pragma unroll
  for (int k = 0; k < RW; ++k) rstd[k] = rsqrtf(total(k) / H + eps);
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    float wv[8], bv[8];
    unpack8(wr[i], wv);
    unpack8(br[i], bv);
    const int c = lane + 64 * i;
#pragma unroll
    for (int k = 0; k < RW; ++k) {
      float o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = fmaf((v[k][i][e] - mean[k]) * rstd[k], wv[e], bv[e]);
      if (c < nv && RW * wid + k < n) *(uint4*)(xs + ((RW * wid + k) * (H + 8) + c * 8) * 2) = pack8(o);
    }
  }
}

// 16 TQ queries from q0 on of one head of one text of up to 16 TK rows, by a wave: attn_packed_kernel's first (and only) tile, without
// the keys that count nothing
template <int TK, int TQ, int D, bool RB>
__device__ __forceinline__ void attend(const Args& a, __amdgpu_buffer_rsrc_t ex, uint32_t qkv, uint32_t to, int base, int len, int q0, int h,
                                       char* vs, int lane) {
  constexpr int DS = D / 32, DT = D / 16, KB = (TK + 1) / 2;  // KB: blocks of 32 keys
  const int g = lane >> 4, r16 = lane & 15, H = a.H;
  auto at = [&](int row, int col) { return qkv + place(a.tiles, base + min(row, len - 1), h * D + col); };
  float bias[TK][TQ][4];
  if constexpr (RB) {
#pragma unroll
    for (int t = 0; t < TK; ++t)
#pragma unroll
      for (int u = 0; u < TQ; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int diff = 16 * t + 4 * g + i - (q0 + 16 * u + r16) + a.rb_L - 1;
          bias[t][u][i] = a.rel_bias[(long)h * (2 * a.rb_L - 1) + min(max(diff, 0), 2 * a.rb_L - 2)];
        }
  }
  constexpr int QN = TQ * DS, KN = TK * DS;
  u32x4 f[QN + KN + KB * DT];  // Q, K by 16 rows, V by 32 rows and 16 columns
  await(a.next + 16, f, [&](int j) {
    uint32_t o;
    if (j < QN) o = at(q0 + 16 * (j / DS) + r16, 32 * (j % DS) + 8 * g);
    else if (j < QN + KN) o = at(16 * ((j - QN) / DS) + r16, H + 32 * ((j - QN) % DS) + 8 * g);
    else o = at((j - QN - KN) / DT * 32 + (lane >> 1), 2 * H + 16 * ((j - QN - KN) % DT) + (lane & 1) * 8);
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ex, o, 0, SC1));
  });
#pragma unroll
  for (int j = 0; j < KB * DT; ++j)
    *(u32x4*)(vs + (j / DT * 32 + (lane >> 1)) * 2 * D + 32 * (j % DT) + (lane & 1) * 16) = f[QN + KN + j];
  f32x4 st[TK][TQ];
#pragma unroll
  for (int t = 0; t < TK; ++t)
#pragma unroll
    for (int u = 0; u < TQ; ++u) {
      st[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < DS; ++s)
        st[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, f[QN + t * DS + s]),
                                                          __builtin_bit_cast(bf16x8, f[u * DS + s]), st[t][u], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        st[t][u][i] = RB ? fmaf(st[t][u][i], a.scale_log2, bias[t][u][i]) : st[t][u][i] * a.scale_log2;
        st[t][u][i] = 16 * t + 4 * g + i < len ? st[t][u][i] : -INFINITY;
      }
    }
  bf16x8 pa[KB][TQ];
  float inv[TQ];
#pragma unroll
  for (int u = 0; u < TQ; ++u) {
    float mx = st[0][u][0];
#pragma unroll
    for (int t = 0; t < TK; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) mx = fmaxf(mx, st[t][u][i]);
    const float mn = over_groups(mx, [](float x, float y) { return fmaxf(x, y); });
    const float mu = mn == -INFINITY ? 0.f : mn;
    float rs = 0.f;
    uint32_t w[4 * KB];
    if (TK == 1) w[2] = w[3] = 0;
#pragma unroll
    for (int t = 0; t < TK; ++t) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma clang fp contract(off)
        st[t][u][i] = __builtin_amdgcn_exp2f(st[t][u][i] - mu);
        rs += st[t][u][i];
      }
      w[2 * t] = pack2bf(st[t][u][0], st[t][u][1]);
      w[2 * t + 1] = pack2bf(st[t][u][2], st[t][u][3]);
    }
    const float l = over_groups(rs, [](float x, float y) { return x + y; });
    inv[u] = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
    for (int k = 0; k < KB; ++k) pa[k][u] = __builtin_bit_cast(bf16x8, u32x4{w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]});
  }
#pragma unroll
  for (int c = 0; c < DT; ++c) {
    f32x4 o[TQ];
#pragma unroll
    for (int u = 0; u < TQ; ++u) o[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      uint32_t w[4];  // V[key][16 c + r16] of keys 4 g .. 4 g + 3 of the block and 16 more
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const bf16_t* const p = (const bf16_t*)vs + (32 * kb + 16 * (k / 2) + 4 * g + 2 * (k & 1)) * D + 16 * c + r16;
        w[k] = p[0] | (uint32_t)p[D] << 16;
      }
      const bf16x8 vf = __builtin_bit_cast(bf16x8, u32x4{w[0], w[1], w[2], w[3]});
#pragma unroll
      for (int u = 0; u < TQ; ++u) o[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pa[kb][u], o[u], 0, 0, 0);
    }
    const int r = row_at(lane, true), quad = quad_at(lane, true), src = quad * 16 + r;
#pragma unroll
    for (int u = 0; u < TQ; ++u) {
      const uint32_t lo = __shfl(pack2bf(o[u][0] * inv[u], o[u][1] * inv[u]), src, 64);
      const uint32_t hi = __shfl(pack2bf(o[u][2] * inv[u], o[u][3] * inv[u]), src, 64);
      const int row = q0 + 16 * u + r;
      if (row < len) put8(ex, to + place_op(a.tiles, base + row, h * D + 16 * c + 4 * quad), lo, hi);
    }
  }
}

// NW: 16-B vectors of a row a lane normalises (H <= 512 NW)
template <int NW>
__global__ __launch_bounds__(64 * WAVES, 2) void encoder_few_kernel(Args a) {
  __shared__ __attribute__((aligned(16))) char sm[LDS];  // weights; rows; partial sums
  __shared__ unsigned task_of[2];
  __shared__ float sb[WAVES];
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const int M = a.M, H = a.H;
  char* const xs = sm + a.lds_x;
  f32x4(*const red)[RED] = (f32x4(*)[RED])(sm + a.lds_red);
  const auto ex = __builtin_amdgcn_make_buffer_rsrc(a.ex, 0, (int)a.ex_bytes, 0x00020000);
  const uint32_t MH = 32u * a.tiles * H, MF = 32u * a.tiles * a.F, per = 8 * MH + MF;  // bytes
  unsigned ahead = 0, *const lost = a.next + 16;
  if (tid == 0) ahead = __hip_atomic_fetch_add(a.next, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (int it = 0;; it ^= 1) {
    if (tid == 0) task_of[it] = ahead;
    __syncthreads();
    const unsigned task = __builtin_amdgcn_readfirstlane(task_of[it]);
    if (task >= (unsigned)a.tasks) return;
    if (tid == 0) ahead = __hip_atomic_fetch_add(a.next, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int l = task / a.layer_tasks;
    int i = task - l * a.layer_tasks;
    const uint32_t at = MH + l * per;  // the layer's rows: qkv + 0, a + 3 MH, d1 + 4 MH, x1 + 5 MH, f + 6 MH, d2, x2 behind it
    const uint32_t x_in = l ? at - MH : 0, d_prev = at - 2 * MH, x1_prev = at - per + 5 * MH;
    if (l == a.L) {  // a text's last norm and its pooling, as pool_norm_kernel
      const long first = min(max(a.off[i], 0L), (long)M);
      const int len = (int)(min(max(a.off[i + 1], first), (long)M) - first);
      float* const acc = (float*)red;
      float s[8] = {};
      for (int r = 0; r < len; r += 16) {
        if (r) __syncthreads();
        norm_rows<NW>(lost, ex, d_prev, x1_prev, a.w[l - 1][10], a.w[l - 1][11], H, a.tiles, (int)first + r, min(len - r, 16), a.eps, xs, wid,
                      lane);
        __syncthreads();
        if (tid < H / 8)
          for (int t = 0; t < min(len - r, 16); ++t) {
            float f[8];
            unpack8(*(const uint4*)(xs + (t * (H + 8) + tid * 8) * 2), f);
#pragma unroll
            for (int e = 0; e < 8; ++e) s[e] += f[e];
          }
      }
      if (tid < H / 8)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[8 * tid + e] = s[e] / (float)max(len, 1);
      __syncthreads();
      float ss = 0.f;
      if (tid < 256)
        for (int h = tid; h < H; h += 256) ss += acc[h] * acc[h];
      const float tot = block_sum(ss, sb);
      const float inv = a.normalize ? 1.f / fmaxf(sqrtf(tot), 1e-12f) : 1.f;
      const long row = a.to[i] < 0 ? a.to[i] + a.out_rows : a.to[i];
      if (row >= 0 && row < a.out_rows)
        for (int h = tid; h < H; h += 64 * WAVES) a.out[row * H + h] = acc[h] * inv;
      continue;
    }
    int kind = 0;
    if (i >= a.p[0].tasks) {
      i -= a.p[0].tasks;
      if (i < a.att_tasks) {
        // a text's heads, queries in blocks of 32
        const int blocks = (a.tiles + 1) / 2, unit = i * a.units + wid, x = unit % blocks, h = unit / blocks % a.heads, b = unit / (blocks * a.heads);
        if (wid < a.units && b < a.B) {
          const long first = min(max(a.off[b], 0L), (long)M);
          const int len = (int)(min(max(a.off[b + 1], first), (long)M) - first), D = H / a.heads;
          char* const vs = xs + wid * VPLACE;
          // rows of no text: nothing reads them but the products, which wait for all of theirs
          const int r0 = b == 0 ? (int)first : 0, r1 = b == a.B - 1 ? (int)first + len : M;
          for (int e = lane; e < (r0 + M - r1) * (D / 4); e += 64) {
            const int r = e / (D / 4);
            put8(ex, at + 3 * MH + place_op(a.tiles, r < r0 ? r : r - r0 + r1, h * D + e % (D / 4) * 4), 0u, 0u);
          }
          if (len > 32 * x) {
            auto go = [&](auto d, auto rb) {
              if (len > 32) attend<4, 2, d.value, rb.value>(a, ex, at, at + 3 * MH, (int)first, len, 32 * x, h, vs, lane);
              else if (len > 16) attend<2, 2, d.value, rb.value>(a, ex, at, at + 3 * MH, (int)first, len, 0, h, vs, lane);
              else attend<1, 1, d.value, rb.value>(a, ex, at, at + 3 * MH, (int)first, len, 0, h, vs, lane);
            };
            using D32 = std::integral_constant<int, 32>;
            using D64 = std::integral_constant<int, 64>;
            if (D == 32) { if (a.rel_bias) go(D32(), std::true_type()); else go(D32(), std::false_type()); }
            else { if (a.rel_bias) go(D64(), std::true_type()); else go(D64(), std::false_type()); }
          }
        }
        continue;
      }
      i -= a.att_tasks;
      kind = 1;
      while (i >= a.p[kind].tasks) i -= a.p[kind++].tasks;
    }
    const Product p = a.p[kind];
    const bool norm = kind == 2 || (kind == 0 && l > 0);
    const int wk = kind == 0 ? 0 : kind == 1 ? 2 : kind == 2 ? 6 : 8;
    const bf16_t *const w = a.w[l][wk], *const bias = a.w[l][wk + 1];
    const uint32_t src = kind == 0 ? 0 : kind == 1 ? at + 3 * MH : at + 6 * MH;  // rows of a product without a norm
    const uint32_t dst = kind == 0 ? at : kind == 1 ? at + 4 * MH : kind == 2 ? at + 6 * MH : at + 6 * MH + MF;
    const int nc = p.K / 64, ks = wid % p.ks, cg = wid / p.ks;
    const int m0 = i % a.tiles * 16, m = min(M - m0, 16);  // the task's rows
    i /= a.tiles;
    const int n0 = (i * p.cg + cg) * 16;
    const bool on = cg < p.cg && n0 < p.N && ks < p.parts;
    // the wave's chunks: one part's, or two parts' one behind the other
    auto begin = [&](int part) { return part * nc / p.parts; };
    const int b0 = begin(ks), n_0 = on ? begin(ks + 1) - b0 : 0;
    const int b1 = begin(ks + p.ks), n_k = n_0 + (on && ks + p.ks < p.parts ? begin(ks + p.ks + 1) - b1 : 0);
    auto chunk = [&](int k) { return k < n_0 ? b0 + k : b1 + k - n_0; };
    char* const mine = sm + RING / (p.ks * p.cg) * wid * CHUNK;
    if (on) {
      const bf16_t* wp[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int row = 8 * j + (lane >> 3);
        wp[j] = w + (long)(n0 + row) * p.K + ((lane & 7) ^ (row >> 1)) * 8;
      }
      for (int k = 0; k < n_k; ++k)
#pragma unroll
        for (int j = 0; j < 2; ++j) dma16(wp[j] + chunk(k) * 64, mine + k * CHUNK + j * 1024);
    }
    // this wave's results: column group wid, as their 512 bytes lie in memory
    const int row = row_at(lane, kind == 2), quad = quad_at(lane, kind == 2), col = (i * p.cg + wid) * 16 + 4 * quad;
    const uint2 bb = *(const uint2*)(bias + min(col, p.N - 4));
    if (norm) {
      if (kind == 0) norm_rows<NW>(lost, ex, d_prev, x1_prev, a.w[l - 1][10], a.w[l - 1][11], H, a.tiles, m0, m, a.eps, xs, wid, lane);
      else norm_rows<NW>(lost, ex, at + 4 * MH, x_in, a.w[l][4], a.w[l][5], H, a.tiles, m0, m, a.eps, xs, wid, lane);
    }
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    auto keep = [&](int part) { red[part * p.cg + cg][lane + g] = acc; };
    auto weights = [&](int k, int h) {
      return *(const bf16x8*)(mine + k * CHUNK + r16 * 128 + (((4 * h + g) ^ (r16 >> 1)) << 4));
    };
    if (norm) {  // all waves' rows in one place
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      constexpr int U = 3;
      for (int k0 = 0; k0 < n_k; k0 += U) {
        bf16x8 wf[U][2], xf[U][2];
#pragma unroll
        for (int q = 0; q < U; ++q) {
          const int k = min(k0 + q, n_k - 1);
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            wf[q][h] = weights(k, h);
            xf[q][h] = *(const bf16x8*)(xs + (r16 * (H + 8) + chunk(k) * 64 + h * 32 + 8 * g) * 2);
          }
        }
#pragma unroll
        for (int q = 0; q < U; ++q)
          if (k0 + q < n_k) {
            if (k0 + q == n_0) {
              keep(ks);
              acc = f32x4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[q][h], xf[q][h], acc, 0, 0, 0);
          }
      }
    } else {  // every wave the columns of its own parts, as the MFMA takes them
      const int r = m0 + min(r16, m - 1);
      const uint32_t at = src + (kind ? place_op(a.tiles, r, 8 * g) : place(a.tiles, r, 8 * g));
      // chunks k0 .. k0 + U: no load under a condition
      auto chunks = [&](int k0, auto u) {
        constexpr int U = u.value;
        u32x4 x[2 * U];
        await(lost, x, [&](int j) {
          return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ex, at, (2 * chunk(min(k0 + j / 2, n_k - 1)) + j % 2) * 1024 * a.tiles, SC1));
        });
        if (k0 == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the weights, too
        bf16x8 wf[U][2];
#pragma unroll
        for (int q = 0; q < U; ++q)
#pragma unroll
          for (int h = 0; h < 2; ++h) wf[q][h] = weights(min(k0 + q, n_k - 1), h);
#pragma unroll
        for (int q = 0; q < U; ++q)
          if (k0 + q < n_k) {
            if (k0 + q == n_0) {
              keep(ks);
              acc = f32x4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
              acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[q][h], __builtin_bit_cast(bf16x8, x[2 * q + h]), acc, 0, 0, 0);
          }
      };
      for (int k0 = 0; k0 < n_k; k0 += 6) {
        if (n_k - k0 <= 2) chunks(k0, std::integral_constant<int, 2>());
        else if (n_k - k0 == 3) chunks(k0, std::integral_constant<int, 3>());
        else chunks(k0, std::integral_constant<int, 6>());
      }
    }
    if (n_k) keep(n_k > n_0 ? ks + p.ks : ks);
    __syncthreads();
    if (wid < p.cg && row < m && col < p.N) {
      f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f}, u = v;
      int in = 0;  // of its group
      for (int q0 = 0; q0 < p.parts; q0 += 4) {
        f32x4 r[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) r[q] = red[min(q0 + q, p.parts - 1) * p.cg + wid][quad * 17 + row];
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (q0 + q < p.parts) {
            u = in ? u + r[q] : r[q];
            if (++in == p.grp) {
              v = p.parts == p.grp ? u : v + u;
              in = 0;
            }
          }
      }
      v += f32x4{__uint_as_float(bb.x << 16), __uint_as_float(bb.x & 0xffff0000u), __uint_as_float(bb.y << 16), __uint_as_float(bb.y & 0xffff0000u)};
      const uint32_t y = dst + (kind == 2 ? place_op(a.tiles, m0 + row, col) : place(a.tiles, m0 + row, col));
      if (kind == 2) put8(ex, y, gelu2_bf16(v[0], v[1]), gelu2_bf16(v[2], v[3]));
      else put8(ex, y, pack2bf(v[0], v[1]), pack2bf(v[2], v[3]));
    }
    if (norm && i == 0) {  // the normed rows are a residual, two products on
      for (int e = tid; e < 2 * H; e += 64 * WAVES) {
        const int r = e / 2 % 16, c = e / 32 * 16 + (e & 1) * 8;
        if (r >= m) continue;
        const u32x4 q = *(const u32x4*)(xs + (r * (H + 8) + c) * 2);
        __builtin_amdgcn_raw_buffer_store_b128(u32x4{word_of(q[0]), word_of(q[1]), word_of(q[2]), word_of(q[3])}, ex,
                                               (kind == 0 ? x_in : at + 5 * MH) + place(a.tiles, m0 + r, c), 0, SC1);
      }
    }
  }
}

}  // namespace ef
}  // namespace rt

using namespace rt;

static bool plan(ef::Product& p, int M, int N, int K, int parts, int grp) {
  if (parts < 1 || parts > (M <= 16 ? 16 : 8) || grp < 1 || parts % grp || parts > K / 64) return false;
  p.N = N; p.K = K; p.parts = parts; p.grp = grp;
  p.ks = parts > 4 ? 8 : parts > 2 ? 4 : parts;
  int most = 0;  // chunks of a wave
  for (int k = 0; k < p.ks; ++k) {
    int n = 0;
    for (int q = k; q < parts; q += p.ks) n += (q + 1) * (K / 64) / parts - q * (K / 64) / parts;
    most = std::max(most, n);
  }
  p.cg = K > N ? 1 : std::min(ef::WAVES / p.ks, N == K ? 2 : 4);
  while (p.cg && ef::RING / (p.ks * p.cg) < most) p.cg /= 2;
  if (!p.cg) return false;
  p.tasks = (N / 16 + p.cg - 1) / p.cg * ((M + 15) / 16);
  return true;
}

static int red_bytes(const ef::Product& p) { return p.parts * p.cg * ef::RED * 16; }
// normed rows of a task, or values of attention
static int x_bytes(int H) { return std::max(16 * (H + 8) * 2, ef::UNITS * ef::VPLACE); }

// Bytes of rows on their way (ahead of them a FewHead); 0: not for this kernel. parts: n, grp of qkv, o, fc1, fc2.
extern "C" long rt_encoder_few_bytes(int M, int H, int F, int B, int L, int heads, const int* parts) {
  if (M < 1 || M > 64 || B < 1 || B > 1 << 12 || L < 1 || L > ef::MAX_LAYERS || heads < 1 || H % heads || H % 64 || F % 64 || H > 1024 || F > 1 << 14) return 0;
  if (H / heads != 32 && H / heads != 64) return 0;
  ef::Product p;
  const int N[4] = {3 * H, H, F, H}, K[4] = {H, H, H, F};
  int red = H * 4;
  for (int k = 0; k < 4; ++k) {
    if (!plan(p, M, N[k], K[k], parts[2 * k], parts[2 * k + 1])) return 0;
    red = std::max(red, red_bytes(p));
  }
  if (x_bytes(H) + ef::RING * ef::CHUNK + red > ef::LDS) return 0;
  return 256 + (M + 15) / 16 * 32L * (H + L * (8L * H + F));
}

// x0 in place at ex (behind the head), everything else of it unset (see rt_embed_norm_rows)
extern "C" int rt_encoder_few(const void* const* w, void* ws, long bytes, const long* off, const float* rel_bias, int rb_L, int M, int H, int F,
                              int B, int L, int heads, float eps, float scale, const int* parts, int normalize, float* out, const long* to,
                              long out_rows, hipStream_t stream) {
  if (rt_encoder_few_bytes(M, H, F, B, L, heads, parts) != bytes) return -1;
  ef::Args a;
  for (int l = 0; l < L; ++l)
    for (int k = 0; k < 12; ++k) a.w[l][k] = (const bf16_t*)w[12 * l + k];
  const int N[4] = {3 * H, H, F, H}, K[4] = {H, H, H, F};
  int n = 0;
  for (int k = 0; k < 4; ++k) {
    plan(a.p[k], M, N[k], K[k], parts[2 * k], parts[2 * k + 1]);
    n += a.p[k].tasks;
  }
  a.M = M; a.H = H; a.F = F; a.B = B; a.L = L; a.heads = heads; a.tiles = (M + 15) / 16;
  const int units = B * heads * ((a.tiles + 1) / 2);
  a.units = std::min(ef::UNITS, (units + 31) / 32);
  a.att_tasks = (units + a.units - 1) / a.units;
  a.layer_tasks = n + a.att_tasks;
  a.tasks = L * a.layer_tasks + B;
  a.eps = eps; a.scale_log2 = scale * 1.4426950408889634f;
  a.rel_bias = rel_bias; a.rb_L = rb_L; a.off = off;
  a.next = (unsigned*)ws; a.ex = (bf16_t*)((char*)ws + 256); a.ex_bytes = (unsigned)(bytes - 256);
  a.normalize = normalize; a.out = out; a.to = to; a.out_rows = out_rows;
  a.lds_x = ef::RING * ef::CHUNK;
  a.lds_red = a.lds_x + x_bytes(H);
  const dim3 grid(std::min(num_cus(), a.layer_tasks)), block(64 * ef::WAVES);
  if (H <= 512) hipLaunchKernelGGL(ef::encoder_few_kernel<1>, grid, block, 0, stream, a);
  else hipLaunchKernelGGL(ef::encoder_few_kernel<2>, grid, block, 0, stream, a);
  RT_LAUNCH_CHECK();
  return 0;
}
