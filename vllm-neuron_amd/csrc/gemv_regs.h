// Token-generation weight stream for 5 .. 32 rows, and for up to 4 where no norm is left to do in front: the activations live in registers.
//
// The kernels of linear_device.h keep the activations in LDS.  From 5 rows on that is what their time goes to: rows x K does not fit
// beside the reduction buffers, so it is staged in chunks between barriers, or streamed beside the weights and read back by every wave.  Here a
// work-group's eight waves split its K-slice and a wave takes its eighth of the activations into registers once, as MFMA operands (4096 deep and 32
// rows: 128 registers a lane).  After that a wave only requests weight tiles, one row-tile ahead, and multiplies them; per row-tile the eight
// partial sums meet in LDS, and the waves take turns at adding them up (in wave order) and running the epilogue, so that no wave has stores
// of every row-tile in front of its requests (vector memory retires in order).  K beyond what fits the registers goes over grid.y: raw sums to
// slabs, added by the next row norm or by splitk_reduce.
// Bound by the weight bytes (117 MB of gate|up of the 8B model in fp8 in 22.7 us at 8 rows, 5.2 TB/s; 27.3 at 32).  us a launch, LDS kernels -> these,
// 8B fp8 at 32 rows: gate|up 35.8 -> 27.3, QKV 23 -> 15.7, and 4.8 for each norm that was a part of them; 7B int8 at 24 rows: gate|up 57.8 -> 30.9.
#pragma once
#include "linear_device.h"

namespace mi {

constexpr int kRegsMaxPasses = 64;   // row-tiles of a work-group: their scales and biases wait in LDS

// HOLD: a work-group takes HOLD row-tiles side by side, and the wave that sums them puts their results together in LDS until it has all: a row's HOLD x 64 bytes
// leave with one request.  For results that go over PCIe, whose packets are what one request writes side by side: 32 rows of 128256 in pieces of 64 bytes
// take 370 us (44 GB/s), of 128 bytes 320, of 256 and more 299 (55 GB/s, a copy 303).  The head of the 8B shape at 32 rows 333 us with four requests of 64 bytes
// from registers, 313 now.
template <int WD, int EPI, int MG, int NK, bool SLAB, int HOLD = 1>
__global__ __launch_bounds__(kGemvWaves * 64) void gemv_regs_kernel(const uint4* __restrict__ W, int NT, int KT, int M, int G,
                                                                   const uint16_t* __restrict__ x, int ldx, EpiArgs e, float* __restrict__ slab) {
  if constexpr (MG == 2) e.next_x = nullptr;          // (up to 16 rows; the registers of 32 leave no room for it)
  constexpr int FR = WD == MI_W_BF16 ? 1 : 2;         // MFMAs per weight tile and column group
  constexpr int NB = NK > 8 ? 2 : 1, BT = NK / NB;    // batches per row-tile, weight tiles per request batch (up to 8 KiB a wave)
  constexpr int TK = WD == MI_W_BF16 ? 32 : 64;
  static_assert(NB * BT == NK, "whole batches");
  __shared__ f32x4_t red[2][kGemvWaves][MG][64];
  __shared__ __attribute__((aligned(16))) float sc_lds[SLAB ? 4 : kRegsMaxPasses * 16], bi_lds[SLAB ? 4 : kRegsMaxPasses * 16];
  __shared__ float rf_lds[SLAB ? 1 : 16 * MG];        // the rows' own factors: 1 / rms where the norm left it to the output
  constexpr int kOutPitch = HOLD * 16 + 4;
  __shared__ __attribute__((aligned(16))) float out_lds[HOLD == 1 ? 4 : 16 * MG * kOutPitch];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int g = lane >> 4, c = lane & 15;
  const int kper = ceil_div(KT, (int)gridDim.y), k_lo = (int)blockIdx.y * kper, k_hi = min(k_lo + kper, KT);
  const int ktw = ceil_div(k_hi - k_lo, kGemvWaves);
  const int kbeg = min(k_lo + wave * ktw, k_hi), kend = min(kbeg + ktw, k_hi), klast = max(kend - 1, k_lo);
  const auto tile_of = [&](int pass) { return HOLD == 1 ? (int)blockIdx.x + pass * G : ((int)blockIdx.x + pass / HOLD * G) * HOLD + pass % HOLD; };
  int passes = ceil_div(ceil_div(NT, HOLD) - (int)blockIdx.x, G) * HOLD;
  if constexpr (HOLD > 1) passes -= max(tile_of(passes - 1) + 1 - NT, 0);       // (the last group may be short)

  // ---- this wave's activations: row c (and 16 + c) of every k-tile it owns; tiles it does not own multiply zeros ----
  u32x4_t xf[NK * FR * MG];
#pragma unroll
  for (int mg = 0; mg < MG; ++mg) {
    const uint16_t* row = x + (size_t)min(mg * 16 + c, M - 1) * ldx + g * (8 * FR);
#pragma unroll
    for (int j = 0; j < NK; ++j) {
      const int kt = min(kbeg + j, klast);
#pragma unroll
      for (int f = 0; f < FR; ++f) xf[(j * FR + f) * MG + mg] = *reinterpret_cast<const u32x4_t*>(row + (size_t)kt * TK + f * 8);
    }
  }
  // The rows' own factors (no residual has one).  Everybody asks, so that no branch waits; in front of the weights, whose second batch would wait for them behind the first
  // (sums of squares over 16 columns, 16 rows of 4096: gate | up of the 8B shape 23.3 us that way, 22.3 now; QKV 10.4 and 9.7; scales and biases asked for up here gained nothing).
  constexpr bool kFactor = !SLAB && EPI != EPI_RESID;
  RowFactor rf;
  float4 ss0, ss1;                                    // 16 rows: 32 threads a row, up to 8 parts each
  const bool parts = e.rs_n > 0.f;
  const int n4 = parts ? e.rs_parts >> 2 : 1, pl = tid & 31;
  if constexpr (kFactor && MG == 1) {
    const float* q = e.row_scale ? e.row_scale : e.scale;
    const float* p4 = parts ? q + (size_t)min(tid >> 5, M - 1) * e.rs_parts : e.scale;
    rf.a = q[e.row_scale && !parts ? min(tid >> 5, M - 1) : 0];
    ss0 = reinterpret_cast<const float4*>(p4)[min(pl, n4 - 1)];
    ss1 = reinterpret_cast<const float4*>(p4)[min(pl + 32, n4 - 1)];
  } else if constexpr (kFactor) {
    rf.request(e.row_scale ? e.row_scale : e.scale, e.row_scale ? min(tid, M - 1) : 0, e.rs_n);   // (a thread a row)
  }
  __builtin_amdgcn_sched_barrier(0);
  // operands of the epilogue of the first row-tile (and column group) that this wave finishes
  constexpr bool kPre = !SLAB && HOLD == 1 && !(EPI == EPI_QKV && MG == 2);   // (two groups' rotary factors would not fit the registers)
  EpiPre<kPre ? EPI : EPI_F32> epre;
  const int pre_pass = wave / MG, pre_m = min(wave % MG * 16 + c, M - 1), pre_n = tile_of(min(pre_pass, passes - 1)) * 16 + g * 4;
  if constexpr (kPre) epi_prefetch<EPI>(e, pre_m, pre_n, epre);
  u32x4_t bufA[BT], bufB[BT];
  const int total = passes * NB;
  auto issue = [&](u32x4_t (&buf)[BT], int i) {
    const int ii = min(i, total - 1), k0 = kbeg + (ii % NB) * BT;      // (behind the last batch, and beyond the slice: no request.  O of the 1B shape 5.2 -> 4.7 us, of the 7B 6.4 -> 6.0)
    stream_batch<MG == 2>(buf, W, tile_of(ii / NB) * KT + k0, i < total ? kend - k0 : 0, lane);
  };
  issue(bufA, 0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < NK; ++j)
    if (kbeg + j >= kend) {
#pragma unroll
      for (int q = 0; q < FR * MG; ++q) xf[j * FR * MG + q] = u32x4_t{0, 0, 0, 0};
    }
  if constexpr (kPre) epi_prefetch_dependent<EPI>(e, pre_n, epre);
  if constexpr (!SLAB) {
    const int n = passes * 16;
#pragma unroll
    for (int q = 0; q < kRegsMaxPasses * 16 / (kGemvWaves * 64); ++q) {
      const int i = tid + q * kGemvWaves * 64;
      if (i < n) {
        const int at = tile_of(i >> 4) * 16 + (i & 15);
        sc_lds[i] = e.scale[at];
        bi_lds[i] = e.bias ? e.bias[at] : 0.f;
      }
    }
    if constexpr (!kFactor) {
      if (tid < 16 * MG) rf_lds[tid] = 1.f;
    } else if constexpr (MG == 1) {
      float ss = pl < n4 ? (ss0.x + ss0.y) + (ss0.z + ss0.w) : 0.f;
      if (pl + 32 < n4) ss += (ss1.x + ss1.y) + (ss1.z + ss1.w);
      ss = group_sum<16>(ss);
      ss += __shfl_xor(ss, 16);
      if (pl == 0) rf_lds[tid >> 5] = !e.row_scale ? 1.f : parts ? rsqrtf(ss / e.rs_n + e.rs_eps) : rf.a;
    } else {
      if (tid < 16 * MG) rf_lds[tid] = e.row_scale ? rf.value(e.rs_n, e.rs_eps) : 1.f;
    }
  }
  issue(bufB, 1);

  f32x4_t acc[MG];
#pragma unroll
  for (int mg = 0; mg < MG; ++mg) acc[mg] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](u32x4_t (&buf)[BT], auto j0) {
#pragma unroll
    for (int u = 0; u < BT; ++u) {
      const u32x4_t w = buf[u];
#pragma unroll
      for (int f = 0; f < FR; ++f) {
        bf16x8_t a;
        if constexpr (WD == MI_W_BF16) a = __builtin_bit_cast(bf16x8_t, w);
        else a = f ? decode8<WD>(w[2], w[3]) : decode8<WD>(w[0], w[1]);
#pragma unroll
        for (int mg = 0; mg < MG; ++mg)
          acc[mg] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8_t, xf[((decltype(j0)::value + u) * FR + f) * MG + mg]), acc[mg], 0, 0, 0);
      }
    }
  };
  // the row-tile's partial sums to LDS; everybody's are there behind the barrier.  Two buffers: a wave reads one before it meets the next barrier,
  // and it is written again behind that one.
  auto meet = [&](int par) {
#pragma unroll
    for (int mg = 0; mg < MG; ++mg) {
      red[par][wave][mg][lane] = acc[mg];
      acc[mg] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto finish = [&](int pass, int par) {
#pragma unroll
    for (int mg = 0; mg < MG; ++mg) {
      if (wave != ((pass / HOLD * MG + mg) & (kGemvWaves - 1))) continue;
      f32x4_t s = red[par][0][mg][lane];
#pragma unroll
      for (int w = 1; w < kGemvWaves; ++w) {
        const f32x4_t t = red[par][w][mg][lane];
        s[0] += t[0]; s[1] += t[1]; s[2] += t[2]; s[3] += t[3];
      }
      const int m = mg * 16 + c, n0 = tile_of(pass) * 16 + g * 4;
      if constexpr (HOLD > 1) {
        static_assert(!SLAB && (EPI == EPI_F32 || EPI == EPI_SOFTCAP), "rows of fp32");
        const float *sc4 = sc_lds + pass * 16 + g * 4, *b4 = bi_lds + pass * 16 + g * 4, rmul = rf_lds[m];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[r] *= sc4[r] * rmul;
          if (e.bias) s[r] += b4[r];
          if constexpr (EPI == EPI_SOFTCAP) s[r] = e.softcap * tanhf(s[r] / e.softcap);
        }
        const int sub = pass % HOLD;
        *reinterpret_cast<f32x4_t*>(out_lds + m * kOutPitch + sub * 16 + g * 4) = s;
        if (sub < HOLD - 1 && pass < passes - 1) continue;
        // (this wave's own; the next group's wave writes here behind a barrier that this one comes to with its results read)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int j = 0; j < HOLD; ++j) {
          const int i = j * 64 + lane, row = mg * 16 + i / (HOLD * 4), q = i % (HOLD * 4);
          const f32x4_t v = *reinterpret_cast<const f32x4_t*>(out_lds + row * kOutPitch + q * 4);
          if (row < M && q < sub * 4 + 4) store_through(e.out_f32, ((uint32_t)row * e.ld_out + (tile_of(pass) - sub) * 16 + q * 4) * 4u, v);
        }
        continue;
      }
      if (m >= M) continue;
      if constexpr (SLAB) {
        *reinterpret_cast<float4*>(slab + ((size_t)blockIdx.y * M + m) * (NT * 16) + n0) = make_float4(s[0], s[1], s[2], s[3]);
      } else {
        const float *sc4 = sc_lds + pass * 16 + g * 4, *b4 = e.bias ? bi_lds + pass * 16 + g * 4 : nullptr, rmul = rf_lds[m];
        bool done = false;
        if constexpr (kPre) {
          if (pass == pre_pass) { epilogue_pre<EPI>(e, m, n0, sc4, b4, s, epre, rmul); done = true; }
        }
        if (!done) epilogue_lds<EPI>(e, m, n0, sc4, b4, s, rmul);
      }
    }
  };
  using First = std::integral_constant<int, 0>;
  using Second = std::integral_constant<int, (NB - 1) * BT>;
  if constexpr (NB == 1) {
    // Pairs, and the odd one behind them: with a branch around the second half hipcc waits for all requests in front of every first half, since on the way around
    // it none of them is younger.  Measured: 7B int8 5 rows gate | up (9 and 10 passes) 25.1 -> 23.3 us, head 136 -> 129, down (one pass, K over 8 slices) 15.1 -> 13.0, O
    // 6.0 -> 5.4; O of the 1B shape at 1 row 4.7 -> 4.3.
    for (int pass = 0; pass + 1 < passes; pass += 2) {
      multiply(bufA, First());
      meet(0);
      issue(bufA, pass + 2);
      finish(pass, 0);
      multiply(bufB, First());
      meet(1);
      issue(bufB, pass + 3);
      finish(pass + 1, 1);
    }
    if (passes & 1) {
      multiply(bufA, First());
      meet(0);
      finish(passes - 1, 0);
    }
  } else {
    for (int pass = 0; pass < passes; ++pass) {
      multiply(bufA, First());
      issue(bufA, 2 * pass + 2);
      multiply(bufB, Second());
      meet(pass & 1);
      issue(bufB, 2 * pass + 3);
      finish(pass, pass & 1);
    }
  }
}

template <int WD, int EPI, int MG, bool SLAB, int HOLD = 1>
static int launch_gemv_regs_k(const LinearW& w, int M, const uint16_t* x, int ldx, const EpiArgs& e, hipStream_t s, int slices, float* slab) {
  const int NT = w.N / 16, KT = w.K / tile_k(WD);
  int num_cu = 0;
  MI_TRY_(device_num_cu(&num_cu));
  const int tiles = ceil_div(ceil_div(KT, slices), kGemvWaves), per = std::max(1, num_cu / slices);
  // every work-group the same number of row-tiles, or one less; at most kRegsMaxPasses
  const int groups = ceil_div(NT, HOLD), G = ceil_div(groups, std::min(kRegsMaxPasses / HOLD, ceil_div(groups, std::min(groups, per))));
  const dim3 grid(G, slices);
  const uint4* W = reinterpret_cast<const uint4*>(w.w);
#define MI_K(NK_) hipLaunchKernelGGL((gemv_regs_kernel<WD, EPI, MG, NK_, SLAB, HOLD>), grid, dim3(kGemvWaves * 64), 0, s, W, NT, KT, M, G, x, ldx, e, slab)
  if (tiles <= 4) MI_K(4);
  else if (tiles == 5) MI_K(5);
  else if (tiles == 6) MI_K(6);
  else if (tiles == 7) MI_K(7);
  else if (tiles == 8) MI_K(8);
  else if constexpr (WD == MI_W_BF16) {
    if (tiles <= 12) MI_K(12);
    else if (tiles <= 14) MI_K(14);
    else MI_K(16);
  }
#undef MI_K
  MI_HIP(hipGetLastError());
  return MI_OK;
}

// Over how many slices K goes: what the registers need at least, and more where whole rows of K would leave CUs idle (2048 x 2048: 128 row-tiles) if the
// sums have a taker.  us: a work-group's weights at 24 GB/s, its rows at 50 GB/s, the slabs both ways, and a launch that adds them where no row norm does.
// (Without the rows' term, us a step: 8B fp8 32 rows 2150, 2099 with it; bf16 24 rows 2323, 2261; 7B int8 24 rows 1820, 1801; Rapodra 20 rows 731, 721.)
template <int WD>
static int gemv_regs_slices(int M, int N, int K, size_t ws_bytes, bool deferred, int num_cu, double* us = nullptr) {
  const int NT = N / 16, KT = K / tile_k(WD);
  int best = 0;
  double best_cost = 0.;
  for (int z = ceil_div(KT, kGemvWaves * regs_max_tiles(WD)); z <= 8; ++z) {
    const int per = ceil_div(KT, z);
    if (z > 1 && ((z - 1) * per >= KT || (size_t)z * M * N * sizeof(float) > ws_bytes)) continue;
    double cost = ceil_div(NT, std::max(1, num_cu / z)) * (per / 24.0 + 0.3) + (double)M * per * tile_k(WD) * 4e-5;
    if (z > 1) cost += (deferred ? 0.5 : 4.5) + z * (double)M * N * 1e-6;
    if (best == 0 || cost < best_cost) { best = z; best_cost = cost; }
  }
  if (us) *us = best_cost;
  return best;
}

template <int WD>
int launch_gemv_regs_wd(const LinearW& w, int M, const uint16_t* x, int ldx, int epi, const EpiArgs& e, hipStream_t s, float* ws, size_t ws_bytes, SlabSum* defer,
                        bool split_as_deferred) {
  int num_cu = 0;
  MI_TRY_(device_num_cu(&num_cu));
  const bool deferred = defer && (epi == EPI_RESID || epi == EPI_F32);
  // (where the norm behind is left to its projection, an unsplit K saves that norm's launch: 4.7 us against the 0.3 - 1 that half-empty CUs cost)
  const int slices = e.next_x ? 1 : gemv_regs_slices<WD>(M, w.N, w.K, ws ? ws_bytes : 0, deferred || split_as_deferred, num_cu);
  MI_CHECK(slices > 0, "gemv_regs: no split of K fits the workspace");
  MI_CHECK(!e.next_x || (epi == EPI_RESID && e.ld_out == w.N && M <= 16 && gemv_regs_holds(w)), "gemv_regs: a norm handed on is for residuals of up to 16 rows side by side, K in one slice");
  MI_CHECK(epi != EPI_RESID || !e.row_scale || slices > 1, "gemv_regs: no residual takes a factor a row");
  MI_CHECK(e.rs_n == 0.f || e.rs_parts == kNormParts || (M <= 16 && slices == 1 && e.rs_parts % 4 == 0 && e.rs_parts > 0 && e.rs_parts <= 256), "gemv_regs: a norm's parts");
  if (slices > 1) {
    MI_TRY_(M <= 16 ? (launch_gemv_regs_k<WD, EPI_F32, 1, true>(w, M, x, ldx, e, s, slices, ws)) : (launch_gemv_regs_k<WD, EPI_F32, 2, true>(w, M, x, ldx, e, s, slices, ws)));
    const SlabSum sum{ws, slices, M, w.N, e.scale, e.bias, e.row_scale, e.rs_n, e.rs_eps};
    if (deferred) { *defer = sum; return MI_OK; }
    return launch_splitk_reduce(sum, epi, e, s);
  }
  // (Logits to the host in groups of four row-tiles where their way, in pieces of 64 bytes, takes as long as the weights do or nearly so; below, single row-tiles deal the weights out more evenly.
  //  Steps of half-depth models, us, single -> four: 8B fp8 6 rows 1123 -> 1121, 9 1199 -> 1188, 16 1403 -> 1382, bf16 5 rows 1710 -> 1714, 12 1839 -> 1856, 14 1870 -> 1877, 16 1940 -> 1919,
  //  7B bf16 12 rows 1665 -> 1668, 14 1714 -> 1686, int8 5 rows 1029 -> 1030, 8 1095 -> 1085, 12 1207 -> 1179, 2048 wide 6 rows 522 -> 522, 16 591 -> 585; groups of two gain half of that.
  //  From 17 rows on all of K that the registers hold (4096) lies above.  Not where less than half of the CUs would have a group: us a launch, 20 - 27 rows, 2048 and 4096 wide, single row-tiles and four: 16384 rows of logits 52.9 and 46.4, 8192 29.5 and 27.2,
  //  fp8 26.4 and 25.8, 4096 21.2 and 24.8)
  const bool four = M * 540 >= w.K * (WD == MI_W_BF16 ? 2 : 1) && w.N / 16 >= 2 * num_cu;
#define MI_R4(EPI_) return M <= 16 ? launch_gemv_regs_k<WD, EPI_, 1, false, 4>(w, M, x, ldx, e, s, 1, nullptr) : launch_gemv_regs_k<WD, EPI_, 2, false, 4>(w, M, x, ldx, e, s, 1, nullptr)
  if (e.far_out && four) {
    if (epi == EPI_F32) MI_R4(EPI_F32);
    if constexpr (WD == MI_W_BF16)
      if (epi == EPI_SOFTCAP) MI_R4(EPI_SOFTCAP);
  }
#undef MI_R4
  // (Far results are stored through: left in L2 they cross PCIe when the weights are done.  Steps of half-depth models, us: 8B fp8 4 rows 1116 -> 1095, 8 rows 1147 -> 1120,
  //  16 rows 1299 -> 1288, 7B int8 5 rows 1138 -> 1088, 2048 wide 2 - 16 rows 0.2 - 3 %; groups of four, 8B fp8 9 rows 1230 -> 1188, 32 rows 1790 -> 1768.  Single row-tiles of 17 and more rows, which only heads of
  //  less than two a CU have, are still left in L2; what going through would give there is little: one layer, 24 rows, left -> through, 4096 wide and 8000 words bf16 101.3 -> 96.6, fp8 103.3 -> 101.6,
  //  4096 words 88.8 -> 87.7 and 92.3 -> 92.7, 2048 wide and 4096 words 82.5 -> 81.6 and 83.2 -> 83.3)
  EpiArgs near = e;
  near.far_out = false;
#define MI_R(EPI_) return M <= 16 ? launch_gemv_regs_k<WD, EPI_, 1, false>(w, M, x, ldx, e, s, 1, nullptr) : launch_gemv_regs_k<WD, EPI_, 2, false>(w, M, x, ldx, near, s, 1, nullptr)
  switch (epi) {
    case EPI_QKV: MI_R(EPI_QKV);
    case EPI_SWIGLU: MI_R(EPI_SWIGLU);
    case EPI_RESID: MI_R(EPI_RESID);
    case EPI_F32: MI_R(EPI_F32);
  }
  if constexpr (WD == MI_W_BF16)
    switch (epi) {
      case EPI_RELU2: MI_R(EPI_RELU2);
      case EPI_GLU_CLIP: MI_R(EPI_GLU_CLIP);
      case EPI_SOFTCAP: MI_R(EPI_SOFTCAP);
    }
#undef MI_R
  set_error("gemv_regs: this epilogue is not built for this weight type");
  return MI_EINVAL;
}

template <int WD>
bool gemv_regs_fits_wd(int M, int N, int K, size_t ws_bytes) {
  int num_cu = 0;
  return device_num_cu(&num_cu) == MI_OK && gemv_regs_slices<WD>(M, N, K, ws_bytes, false, num_cu) > 0;
}

template <int WD>
bool gemv_regs_whole_wd(int M, int N, int K, size_t ws_bytes) {
  int num_cu = 0;
  return device_num_cu(&num_cu) == MI_OK && gemv_regs_slices<WD>(M, N, K, ws_bytes, false, num_cu) == 1;
}

// what the choice of slices takes the launch and the sum of its slices to be, us; 0: no split fits
template <int WD>
double gemv_regs_us_wd(int M, int N, int K, size_t ws_bytes, bool deferred) {
  int num_cu = 0;
  double us = 0.;
  if (device_num_cu(&num_cu) == MI_OK) gemv_regs_slices<WD>(M, N, K, ws_bytes, deferred, num_cu, &us);
  return us;
}

}  // namespace mi
