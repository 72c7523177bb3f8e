// y = LN(x w^T + bias + res) of rows that a workgroup holds whole: the two products of a post-norm encoder layer that end in a layer norm.
// As two launches the sum went out to memory and back between them, and 384 columns are one and a half tiles of 256: a quarter of the
// matrix work was for columns that are not there; 768 are three tiles of 256, whose rounds leave CUs idle. us, product and norm -> this, by 384
// columns: 28100 rows x 384 33.7 -> 18.8, x 1536 55.5 -> 35.8; 15000 rows 22.6 -> 12.0, 35.1 -> 23.8; 8960 rows 16.6 -> 10.4, 25.5 -> 22.0. By
// 768 columns, in an encoder: 24000 rows x 768 54.9 -> 37.5, x 3072 121 -> 99, 12000 rows 35.9 -> 24.4, 73.6 -> 67. Encoder forward of 1024
// texts (MiniLM) 3775 -> 3446, of mpnet-base over 12000 / 24000 / 49000 rows 3030 -> 2813 / 5150 -> 4790 / 10390 -> 9740.
#include "rt_common.h"

#include <algorithm>

namespace rt {
namespace gn {

typedef __attribute__((address_space(3))) void lds_void;

struct Args {
  const bf16_t* x; long ldx;
  const bf16_t* w; long ldw;
  const bf16_t* bias;  // [N]
  const bf16_t* res; long ldr;
  const bf16_t* lw;
  const bf16_t* lb;
  bf16_t* y; long ldy;
  int M, K;
  float eps;
};

constexpr int AP = 3, BP = 7;  // places for x images (a K-step of the tile's rows) and for w granules (128 of its columns)

// Of the loads that a wave has asked for up to the start of phase p of a K-step, how many may be under way for what is read in that phase to have
// landed? (A granule of w is 2 of them, an x image na.)
constexpr int newer(int np, int p, int na) {
  const int now = 16 * np + p;  // phases count on over the steps; phase b asks for granule b + BP, the second of a step before it for x of step + AP
  auto issued = [&](int from, int to) {  // by phases [from, to)
    int n = 0;
    for (int b = from; b < to; ++b) n += 2 + (b % np == 1 ? na : 0);
    return n;
  };
  int n = issued(now + 1 - BP + 1, now);  // what is newer than the next phase's granule
  if (p == np - 1) {                      // and than the next step's x
    const int m = issued((17 - AP) * np + 1, now) - na;
    n = m < n ? m : n;
  }
  return n;
}

template <int N, int LDS = 0>
__device__ __forceinline__ void wait_but() {
  static_assert(N < 64 && LDS < 16, "counters");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(%1)" ::"n"(N), "n"(LDS) : "memory");
}

// no template: hipcc's host pass drops kernels that call the builtin with dependent arguments
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, char* to, uint32_t off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)to, 16, off, 0, 0, 0);
}

__device__ __forceinline__ void store16(__amdgpu_buffer_rsrc_t r, uint4 v, uint32_t off) {
  typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
  __builtin_amdgcn_raw_buffer_store_b128(u32x4{v.x, v.y, v.z, v.w}, r, off, 0, 0);
}

// A tile is all 128 NP columns of 64 or 128 rows; 8 waves, 8 / WC x WC, of 16 FM x 16 FN. A K-step of 64 is NP phases: the wave's x fragments
// stay for the step, each phase multiplies them by FG of its w fragments (a granule: 128 columns, 16 FG of every wave). While a phase is
// multiplied the next one's fragments are read, and the places that are read out are asked for again: 7 granules and 3 x images ahead.
// Behind the last step nothing is fetched: the same loads go out of range, which fills their places with zeros and keeps the counted waits.
// 96 rows by 768 columns (64 do not fill the matrix cores' time, of 128 neither sums nor rows fit): x fragments come in a burst of 12 a wave at
// the end of a step, 3270 cycles of which the matrix cores work 2320. Cycles a step of 128 / 64 rows by 384 columns: 2090 / 1300, of which the
// matrix cores work 1546 / 773 and the LDS pipe 1790 / 1310 (fragments and DMA), which bounds it. Waves 2 x 4 read the least of 128 rows, 1 x 8
// of 64. w straight from memory to the one wave that multiplies it (1 x 8) took 3200: its lanes lie 16 rows apart, one line a lane.
template <int WC, int FM, int NP>
__global__ __launch_bounds__(512, 2) void gemm_norm_kernel(Args p) {
  constexpr int TM = 8 / WC * 16 * FM, TN = 128 * NP, FG = 8 / WC, FN = FG * NP, NA = (TM + 63) / 64, XI = TM * 128, GR = 128 * 128, LDT = TN + 8;
  static_assert(TM * LDT * 2 <= AP * XI + BP * GR, "the tile fits the places");
  constexpr bool LATE = NP > 4;  // no registers for the epilogue's operands beside the sums
  __shared__ __attribute__((aligned(16))) char smem[AP * XI + BP * GR];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wid / WC, wc = wid % WC;
  const int frow = lane & 15, fq = lane >> 4;
  const int m0 = blockIdx.x * TM, rows = min(TM, p.M - m0), nk = p.K / 64;

  // Instruction o of an image: rows 8 o .. + 7, 128 B each; lane -> row lane / 8, 16-B slot lane % 8 holding k-chunk slot ^ (row / 2) % 8
  const int kc = ((lane & 7) ^ (lane >> 4)) * 16;
  const uint32_t lx[2] = {(uint32_t)(lane >> 3) * (uint32_t)p.ldx * 2 + kc, (uint32_t)(lane >> 3) * (uint32_t)p.ldx * 2 + (kc ^ 64)};
  const uint32_t lw[2] = {(uint32_t)(lane >> 3) * (uint32_t)p.ldw * 2 + kc, (uint32_t)(lane >> 3) * (uint32_t)p.ldw * 2 + (kc ^ 64)};
  const __amdgpu_buffer_rsrc_t Xr = __builtin_amdgcn_make_buffer_rsrc((void*)(p.x + (long)m0 * p.ldx), 0, ((rows - 1) * (int)p.ldx + p.K) * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t Wr = __builtin_amdgcn_make_buffer_rsrc((void*)p.w, 0, ((TN - 1) * (int)p.ldw + p.K) * 2, 0x00020000);
  constexpr uint32_t FAR = 0x80000000u;  // no operand reaches it (launcher)
  auto stage_x = [&](int t, int place) {
    const uint32_t far = (uint32_t)(nk - 1 - t) & FAR;  // beyond the last step
#pragma unroll
    for (int j = 0; j < NA; ++j) {
      const int o = TM == 96 && j ? 8 + (wid & 3) : TM == 128 ? 2 * wid + j : wid;  // 96 rows: the last four by two waves each, the same bytes
      const uint32_t base = (uint32_t)(o * 8 * (int)p.ldx * 2 + t * 128) | far;
      dma16(Xr, smem + place * XI + o * 1024, (TM == 128 ? lx[j] : lx[wid & 1]) + base);
    }
  };
  // granule of phase ph of step t: image row r is column (r / W) 16 FN + W ph + r % W, W = 16 FG
  auto stage_w = [&](int t, int ph, int place) {
    const uint32_t far = (uint32_t)(nk - 1 - t) & FAR;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int o = wid * 2 + j;
      const uint32_t base = (uint32_t)((o / (2 * FG) * 16 * FN + ph * 16 * FG + o % (2 * FG) * 8) * (int)p.ldw * 2 + t * 128) | far;
      dma16(Wr, smem + AP * XI + place * GR + o * 1024, lw[j] + base);
    }
  };

  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 fx[2][FM], fw[2][2][FG];  // k half; of w this phase's and the next one's
  const int sw = (frow >> 1) & 7, c0 = (fq ^ sw) << 4, c1 = ((4 + fq) ^ sw) << 4;
  const int rx = (wr * 16 * FM + frow) * 128, rw = AP * XI + (wc * 16 * FG + frow) * 128;
  auto read_x = [&](int kk, int i, int place) { fx[kk][i] = *(const bf16x8*)(smem + place * XI + rx + i * 2048 + (kk ? c1 : c0)); };
  auto read_w = [&](auto set, int place) {
    constexpr int S = decltype(set)::value;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int j = 0; j < FG; ++j) fw[S][kk][j] = *(const bf16x8*)(smem + place * GR + rw + j * 2048 + (kk ? c1 : c0));
  };

  // For the epilogue: 16 lanes a row, of which a lane has the 16-B vectors nq + 16 m; a wave four rows at a time
  const int nq = lane & 15, nrow = wid * (TM / 8) + (lane >> 4);
  uint2 bias[FN];
  uint4 res[NP], lwr[NP], lbr[NP];
  auto residual = [&](int row) {
#pragma unroll
    for (int m = 0; m < NP; ++m) res[m] = *(const uint4*)(p.res + (long)(m0 + min(row, rows - 1)) * p.ldr + (nq + 16 * m) * 8);
  };
  auto operands = [&]() {
#pragma unroll
    for (int j = 0; j < FN; ++j) bias[j] = *(const uint2*)(p.bias + (FN * wc + j) * 16 + fq * 4);
    residual(nrow);
#pragma unroll
    for (int m = 0; m < NP; ++m) {
      lwr[m] = *(const uint4*)(p.lw + (nq + 16 * m) * 8);
      lbr[m] = *(const uint4*)(p.lb + (nq + 16 * m) * 8);
    }
  };
  if constexpr (!LATE) operands();

  // All of w, each workgroup its share, in whole rows: the products that go through the caches between two of this one leave nothing of
  // w there, and a K-step of it is a line of 128 B from each of TN rows, which all workgroups ask for at the same time, only 7 granules ahead.
  // Its place is one that this wave fills itself later (loads come in in their order). In an encoder, 768 columns: 12000 rows x 3072 101 -> 67
  // us, x 768 32.2 -> 24.4, 24000 rows x 3072 123 -> 99.
  const uint32_t share = (uint32_t)(((long)TN * p.ldw * 2 / gridDim.x + 8191) / 8192);
  for (uint32_t k = 0; k < min(share, 6u); ++k)
    dma16(Wr, smem + (AP - 1) * XI + (TM == 128 ? 2 * wid : wid) * 1024, ((blockIdx.x * share + k) * 8 + wid) * 1024 + lane * 16);
  // what the phases before the first would have asked for
  constexpr int B0 = AP * NP;
  static_assert(B0 - 1 >= BP, "x first");
#pragma unroll
  for (int b = -B0; b < 0; ++b) {
    if ((b + B0 * NP) % NP == 1) stage_x((b - 1) / NP + AP, (b - 1) / NP + AP);
    if (b + BP >= 0) stage_w((b + BP) / NP, (b + BP) % NP, b + BP);
  }
  int t = 0, xp = 0, wp = 0;  // step, the places of its x and of the phase's granule
  wait_but<newer(NP, NP - 1, NA)>();
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  read_w(std::integral_constant<int, 0>{}, 0);
  asm volatile("" ::: "memory");  // w ahead of x, as a step's last phase
#pragma unroll
  for (int i = 0; i < 2 * FM; ++i) read_x(i / FM, i % FM, 0);
  auto phase = [&](auto set, auto ph) {
    constexpr int P = decltype(ph)::value, S = decltype(set)::value;
    // the next fragments' images have landed and this wave has read this phase's granule (and, from the second phase on, the step's x): behind the
    // barrier both hold for all. In the first phase the step's x, 2 FM reads, may be under way: they were asked for behind the granule's
    wait_but<newer(NP, P, NA), P == 0 ? 2 * FM : 0>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    const int wn = wp == BP - 1 ? 0 : wp + 1, xn = xp == AP - 1 ? 0 : xp + 1;
    read_w(std::integral_constant<int, S ^ 1>{}, wn);
    if constexpr (P == NP - 1) asm volatile("" ::: "memory");  // no read of x ahead of these: the next phase's wait counts on it
    if constexpr (P == 1) stage_x(t + AP, xp);
    stage_w(t + (P + BP) / NP, (P + BP) % NP, wp);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int i = 0; i < FM; ++i) {
#pragma unroll
        for (int j = 0; j < FG; ++j)
          acc[i][FG * P + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[S][kk][j], fx[kk][i], acc[i][FG * P + j], 0, 0, 0);
        if constexpr (P == NP - 1) read_x(kk, i, xn);  // the step's last use
      }
    if constexpr (P < NP - 1) {
#pragma unroll
      for (int k = 0; k < 2 * FG; ++k) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
#pragma unroll
      for (int k = 0; k < 2 + (P == 1 ? NA : 0); ++k) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    wp = wn;
    if constexpr (P == NP - 1) {
      ++t;
      xp = xn;
    }
  };
  auto step = [&](auto st) {
    constexpr int S = decltype(st)::value * (NP & 1);
    phase(std::integral_constant<int, S>{}, std::integral_constant<int, 0>{});
    if constexpr (NP > 1) phase(std::integral_constant<int, S ^ 1>{}, std::integral_constant<int, 1>{});
    if constexpr (NP > 2) phase(std::integral_constant<int, S>{}, std::integral_constant<int, 2>{});
    if constexpr (NP > 3) phase(std::integral_constant<int, S ^ 1>{}, std::integral_constant<int, 3>{});
    if constexpr (NP > 4) phase(std::integral_constant<int, S>{}, std::integral_constant<int, 4>{});
    if constexpr (NP > 5) phase(std::integral_constant<int, S ^ 1>{}, std::integral_constant<int, 5>{});
  };
  while (t + 1 < nk) {
    step(std::integral_constant<int, 0>{});
    step(std::integral_constant<int, 1>{});
  }
  if (t < nk) step(std::integral_constant<int, 0>{});

  // acc[i][j][r] = row 16 (FM wr + i) + frow, column 16 (FN wc + j) + 4 fq + r. The products, rounded, as one tile; then the rows, with the
  // sums as norm_rows_kernel has them (the same bits): a vector's 8 columns in their order, the vectors by a butterfly of 32, 16, 8, .. of 64.
  // Rolled, and four rows a wave at a time: code that a workgroup runs once comes in from L2 as it goes. A wave a row took 17200 cycles of 128 rows,
  // everything in registers in straight code 16200, this takes 9800.
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // nothing lands in the places any more
  __syncthreads();
  if constexpr (LATE) operands();
  bf16_t* const tile = (bf16_t*)smem;
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const float b0 = __uint_as_float(bias[j].x << 16), b1 = __uint_as_float(bias[j].x & 0xffff0000u);
    const float b2 = __uint_as_float(bias[j].y << 16), b3 = __uint_as_float(bias[j].y & 0xffff0000u);
#pragma unroll
    for (int i = 0; i < FM; ++i)
      *(uint2*)(tile + (16 * (FM * wr + i) + frow) * LDT + (FN * wc + j) * 16 + fq * 4) =
          make_uint2(pack2bf(acc[i][j][0] + b0, acc[i][j][1] + b1), pack2bf(acc[i][j][2] + b2, acc[i][j][3] + b3));
  }
  __syncthreads();
  const __amdgpu_buffer_rsrc_t Yr = __builtin_amdgcn_make_buffer_rsrc((void*)(p.y + (long)m0 * p.ldy), 0, ((rows - 1) * (int)p.ldy + TN) * 2, 0x00020000);
  auto row_sum = [&](const float (&x)[NP]) {
    static_assert(NP == 2 || NP == 3 || NP == 4 || NP == 6, "vectors of a lane");
    float s, u = 0.f;  // of the first 64 vectors, of the others
    if constexpr (NP >= 4) s = (x[0] + x[2]) + (x[1] + x[3]);
    else if constexpr (NP == 3) s = (x[0] + x[2]) + x[1];
    else s = x[0] + x[1];
    if constexpr (NP == 6) u = x[4] + x[5];
#define GN_DPP(v, ctrl) v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), ctrl, 0xf, 0xf, false))
#define GN_STEP(ctrl) do { GN_DPP(s, ctrl); if constexpr (NP > 4) GN_DPP(u, ctrl); } while (0)
    GN_STEP(0x128);  // row_ror:8
    GN_STEP(0x124);  // row_ror:4: the exchange of lanes 4 apart, now that those 8 apart hold the same
    GN_STEP(0x4e);   // quad_perm [2, 3, 0, 1]
    GN_STEP(0xb1);   // quad_perm [1, 0, 3, 2]
#undef GN_STEP
#undef GN_DPP
    return NP > 4 ? s + u : s;
  };
#pragma unroll 1
  for (int k = 0; k < TM / 8; k += 4) {
    const int row = nrow + k;
    float v[NP][8], s[NP];
#pragma unroll
    for (int m = 0; m < NP; ++m) {
      float r[8];
      unpack8(*(const uint4*)(tile + row * LDT + (nq + 16 * m) * 8), v[m]);
      unpack8(res[m], r);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[m][e] += r[e];
      unpack8(pack8(v[m]), v[m]);
      s[m] = v[m][0];
#pragma unroll
      for (int e = 1; e < 8; ++e) s[m] += v[m][e];
    }
    residual(row + 4);
    const float mean = row_sum(s) / TN;
#pragma unroll
    for (int m = 0; m < NP; ++m) {
      s[m] = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        v[m][e] -= mean;
        s[m] += v[m][e] * v[m][e];
      }
    }
    const float rstd = rsqrtf(row_sum(s) / TN + p.eps);
#pragma unroll
    for (int m = 0; m < NP; ++m) {
      float wv[8], bv[8], o[8];
      unpack8(lwr[m], wv);
      unpack8(lbr[m], bv);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        o[e] = v[m][e] * rstd * wv[e];
        o[e] += bv[e];
      }
      store16(Yr, pack8(o), (uint32_t)row * (uint32_t)p.ldy * 2 + (nq + 16 * m) * 16);  // rows past the last are out of range
    }
  }
}

}  // namespace gn
}  // namespace rt

using namespace rt;

static bool fits(int N, int K) { return (N == 384 || N == 768) && K >= 64 && K % 64 == 0 && (long)N * K * 2 < 0x7fffffffL; }

// Rows of a tile with which rt_gemm_norm beats product and norm, `first` leading rows in larger ones; 0: it doesn't, or the shape is not for it.
// A tile is one chain over K, however few there are: with few rows the product's small tiles in parallel are faster.
// 384 columns: 0.54 us a step of 64 rows and 6 besides (128 rows: 0.9 and 8). Even: 2500 rows at K 128, 3000 at 384, 4500 at 768, 5300 at 1536,
// 10500 at 3072; between an encoder's other kernels of 4000 to 5000 rows both are even at K 384 (a forward of 4500 403 us), 5500 / 8000 464 / 530 -> 456 / 510.
// Tiles of 64 while they are one round of the CUs (16384 rows x 1536 24.7 us, tiles of 128 32.1), then 128 (17000 rows 31.7, tiles of 64 42.6),
// whole rounds of these and the rest in 64 where that is one round more (MiniLM over 34000 rows 1434 -> 1396 us). 768 columns, us within an
// encoder's forward (between other kernels: alone, with w in the caches, both are faster): a round of tiles of 64 takes 10 and 1.18 a step,
// nearly full 14 and 1.25, one of several 6.4 and 1.53; of 96 18 and 1.72. Product and norm: tiles of 256 x 256, whole rounds of them and a
// rest, and 0.78 ns a row. All of one size, or whole rounds of 96 and the rest in 64. Product and norm | this at K 768: 12000 rows 35.9 | 24.4,
// 20000 42.7 | 34.0, 24000 54.9 | 37.5, 28000 59.3 | 49.4, 42000 88 | 73; at K 3072: 12000 73.6 | 67, 20000 89.6 | 90 (not taken), 24000 121 |
// 99, 28000 146 | 160 (not taken), 49000 237 | 204.
extern "C" int rt_gemm_norm_rows(int M, int N, int K, int* first) {
  *first = 0;
  if (!fits(N, K)) return 0;
  const int per64 = 64 * num_cus();
  if (N == 384) {
    if (M < std::max(4000L, 1800 + 3L * K)) return 0;
    const int whole = M / (2 * per64) * 2 * per64;
    if (M - whole > per64) return 128;
    *first = M > whole ? whole : 0;
    return M > whole ? 64 : 128;
  }
  const int per96 = 96 * num_cus(), per256 = num_cus() / 3 * 256;
  auto rounds = [](int rows, int per) { return (rows + per - 1) / per; };
  const double steps = K / 64;
  auto in64 = [&](int rows) {
    const int n = rounds(rows, per64);
    return n > 1 ? n * (6.4 + 1.53 * steps) : 4L * rows <= 3L * per64 ? 10 + 1.18 * steps : 14 + 1.25 * steps;
  };
  const double r96 = 18 + 1.72 * steps, large = 13 + 0.0203 * K, rest = std::min(1., 0.24 + 5e-5 * (M % per256));
  const double apart = (M / per256 + rest) * large + 1.5 + 0.00078 * M;
  const int whole = M / per96;
  const double all64 = in64(M), all96 = rounds(M, per96) * r96, both = whole * r96 + in64(M - whole * per96);
  if (std::min(std::min(all64, all96), both) > apart) return 0;
  if (whole && both < all64 && both < all96) *first = whole * per96;
  return all96 <= all64 && !*first ? 96 : 64;
}

// y = LN(x w^T + bias + res) * lw + lb of M rows, N = 384 or 768 columns, K % 64 == 0; contiguous 16-B aligned rows. rows: of a tile, 64 or 128
// (384 columns) or 96 (768); 0: as rt_gemm_norm_rows says. -1: not for this kernel.
extern "C" int rt_gemm_norm(const void* x, const void* w, const void* bias, const void* res, const void* lw, const void* lb, void* y, int M,
                            int N, int K, float eps, int rows, hipStream_t stream) {
  const int large = N == 384 ? 128 : 96;
  int first = 0;
  if (!rows) rows = rt_gemm_norm_rows(M, N, K, &first);
  if (!fits(N, K) || (rows != 64 && rows != large)) return -1;
  if (M <= 0) return 0;
  auto launch = [&](int m0, int n, int tile) {
    gn::Args p;
    p.x = (const bf16_t*)x + (long)m0 * K; p.ldx = K; p.w = (const bf16_t*)w; p.ldw = K; p.bias = (const bf16_t*)bias;
    p.res = (const bf16_t*)res + (long)m0 * N; p.ldr = N; p.lw = (const bf16_t*)lw; p.lb = (const bf16_t*)lb; p.y = (bf16_t*)y + (long)m0 * N;
    p.ldy = N; p.M = n; p.K = K; p.eps = eps;
    const dim3 grid((n + tile - 1) / tile), block(512);
    if (N == 768 && tile == 64) hipLaunchKernelGGL((gn::gemm_norm_kernel<8, 4, 6>), grid, block, 0, stream, p);
    else if (N == 768) hipLaunchKernelGGL((gn::gemm_norm_kernel<8, 6, 6>), grid, block, 0, stream, p);
    else if (tile == 64) hipLaunchKernelGGL((gn::gemm_norm_kernel<8, 4, 3>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((gn::gemm_norm_kernel<4, 4, 3>), grid, block, 0, stream, p);
  };
  if (first) launch(0, first, large);
  if (M > first) launch(first, M - first, rows);
  RT_LAUNCH_CHECK();
  return 0;
}
