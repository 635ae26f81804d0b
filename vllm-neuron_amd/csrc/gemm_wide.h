// The wide context-encoding GEMM (launched through linear_kernels.hip, instantiated per weight type).
#pragma once
#include <algorithm>

#include "linear_device.h"
#include "linear_kernels.h"

namespace mi {

// =====================================================================================
// GEMM, wide-N tile with an LDS-DMA ring and two wave groups half a K-step apart (context encoding)
// =====================================================================================
// A 128 x 128 tile pulls 16 KiB of activations + 8 (16) KiB of weights per 64-deep K-step for 2.1 MFLOP.  A CU takes in 55 - 65 GB/s
// once half of it comes from HBM (64 KiB of requests in flight, 1.2 us each; from L2 it takes 125 GB/s), so the tile grows: 128 tokens x 256
// weight rows = 16 + 16 (32) KiB for 4.2 MFLOP, 256 x 256 = 32 + 16 (32) KiB for 8.4.  Smaller ones (32 by 32 to 192 tokens x 128, 192 weight rows) are for
// what those leave idle: a grid of one and a bit rounds, token blocks mostly padding, few tokens, whose K then takes fewer slabs.  Eight waves as 2 (tokens) x 4 (weight
// rows): activation fragments are shared by four waves, weight fragments by two.  Both operands arrive by LDS-DMA
// (global_load_lds, 1 KiB per wave-instruction: the weight tiles land lane-linear = fragment
// order; the activation rows land in an XOR-swizzled image (xs_swz), the swizzle being
// applied to the per-lane SOURCE address) into a ring of stages: all but the one being multiplied are in
// flight, retired by counted vmcnt waits in front of raw barriers -- no ordinary global
// load in the loop, so hipcc has nothing to drain.  A wave's K-step is a READ phase (fragments LDS -> registers, then the requests of a later
// K-step) and a MULTIPLY phase (MFMAs, the weight codes decoded between them), and the two waves of a SIMD are in opposite phases
// (see "Schedule" in the kernel).
// What it holds on full grids (gate|up of the 8B model, 2031 tokens): bf16 1.22, fp8 1.27, int8 1.22 PF/s (1.16 before the codes were decoded
// between the MFMAs), where a library product of 8192^3 in bf16 runs at 1.28 on this card; 128-token blocks 1.13 / 1.18 / 1.05.

// A work-group's tile: BM tokens x 64 NTW weight rows (NTW 16-row tiles for each of the four waves side by side).
template <int WD, int NTW> constexpr int kWideWBytes = NTW * (WD == MI_W_BF16 ? 8 : 4) * 1024;   // the weight rows of a 64-deep K-step
// as many stages as the LDS holds, eight at most
template <int WD, int BM, int NTW, int KD = 1> constexpr int kWideStages = std::min(8, 160 * 1024 / (KD * (kWideWBytes<WD, NTW> + BM * 128)));

// Waits until at most the youngest min(left, MOST) K-steps' DMAs (PER each) of this wave are in flight.
template <int PER, int MOST>
__device__ __forceinline__ void wait_dma(int left) {
  if (left >= MOST) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER * MOST) : "memory");
  else if constexpr (MOST > 0) wait_dma<PER, MOST - 1>(left);
}

// What a work-group needs in front of its first request, in one line of kernel arguments and taken in one go (wide_args): a kernel's arguments come from memory, and hipcc fetches
// each where it is first used.  Divisions are the host's.  (A work-group took 1.6 - 3.1 us to the
// last request of its ring.)  us a launch, before -> now: int8 188 x 4608 in 3 slices 14.2 -> 13.6, x 3584 in 4 12.1 -> 11.6, 18944 deep in 8 33.0 -> 32.4; calls of 32 .. 250 rows 0.8 - 1.3 %, of 1000 tokens and more nothing.
struct WideArgs {
  const uint4* W;
  const uint16_t* x;
  float* slab;
  int NT, KT, T, K, ldx;
  int mtiles, per;           // token blocks; tiles of an XCD
  unsigned by_mtiles;        // 2^32 / mtiles, rounded down
  int kper;                  // K-steps of a slice
};
static_assert(sizeof(WideArgs) <= 64, "a line");
__device__ __forceinline__ void wide_args(const WideArgs& a) {
  asm volatile("" ::"s"(a.W), "s"(a.x), "s"(a.slab), "s"(a.NT), "s"(a.KT), "s"(a.T), "s"(a.K), "s"(a.ldx), "s"(a.mtiles), "s"(a.per), "s"(a.by_mtiles), "s"(a.kper));
}
// ... and what its epilogue needs, asked for behind those requests
template <int EPI, bool SPLIT>
__device__ __forceinline__ void wide_epi_args(const EpiArgs& e) {
  if constexpr (SPLIT) return;
  asm volatile("" ::"s"(e.scale), "s"(e.bias), "s"(e.row_scale));
  if constexpr (EPI == EPI_F32 || EPI == EPI_RESID || EPI == EPI_SOFTCAP) asm volatile("" ::"s"(e.out_f32), "s"(e.ld_out));
  if constexpr (EPI == EPI_RESID) asm volatile("" ::"s"(e.resid_in));
  if constexpr (EPI == EPI_SWIGLU || EPI == EPI_GLU_CLIP || EPI == EPI_RELU2) asm volatile("" ::"s"(e.act_out), "s"(e.ld_act));
  if constexpr (EPI == EPI_QKV) asm volatile("" ::"s"(e.q_out), "s"(e.q_dim), "s"(e.kv_dim), "s"(e.hd), "s"(e.nkv), "s"(e.pos), "s"(e.slots), "s"(e.rope_cos), "s"(e.rope_sin), "s"(e.kpool), "s"(e.vpool), "s"(e.block_size));
}
// The tile of this work-group.  Work-group b runs on XCD b % 8: an XCD takes an eighth of the tiles, one after the other with the token
// blocks of a weight slab in a row, so that a slab comes into its L2 once.  (Every eighth slab to an XCD, as in gemm_kernel, left the XCDs
// up to a slab apart: 44 slabs of 11 token blocks put 66 work-groups on the 32 CUs of four of them, three rounds in place of two.)
template <int BM, int NTW>
__device__ __forceinline__ bool wide_tile(const WideArgs& a, int& m0, int& nt0) {
  const unsigned seq = blockIdx.x >> 3, t = (blockIdx.x & 7) * a.per + seq;
  if (seq >= (unsigned)a.per || t >= (unsigned)(a.mtiles * ceil_div(a.NT, 4 * NTW))) return false;
  unsigned q = __umulhi(t, a.by_mtiles);     // t / mtiles, or one less
  if (t - q * a.mtiles >= (unsigned)a.mtiles) ++q;
  nt0 = (int)q * (4 * NTW);
  m0 = (int)(t - q * a.mtiles) * BM;
  return true;
}
// the K-steps of grid.z slice blockIdx.z: equal ones, the last may be shorter (the launch leaves none empty)
template <bool SPLIT, int KD = 1>
__device__ __forceinline__ void wide_slice(const WideArgs& a, int& ks0, int& nks) {
  const int all = a.K / (64 * KD);
  ks0 = SPLIT ? (int)blockIdx.z * a.kper : 0;
  nks = SPLIT ? min(a.kper, all - ks0) : all;
}

// Slabs are written through while they fit the eight L2s (4 MiB each) with room for the rows and weights that come in beside them: left there, they go out when the kernel
// ends, and the norm behind waits.  us a launch, left -> through: 8 slabs of 188 x 3584 (21.6 MB) 34.3 -> 32.8, 4 of 242 x 4096 (15.9 MB) 31.7 -> 30.2, 3 of 188 x 4608 15.0 -> 14.0, 8 of
// 32 x 4096 8.7 -> 7.5.  Larger ones mostly leave on the way, and pieces of 64 bytes cost more than lines: 2 of 1000 x 4096 (32.8 MB) 107.3 -> 107.9, 2 of 2031 x 4096 181 -> 185.
// Nor where the weights are more than four times the slabs and keep the memory busy to the end: bf16 14336 x 2048, 100 tokens 19.6 -> 20.8, 3584 x 4608 14.7 -> 15.7, fp8 14336 x 4096, 60 tokens
// 17.7 -> 18.2, 100 (4.5 times) 25.5 -> 25.6; 8B bf16, 60 tokens 2127 -> 2155 a call.
constexpr size_t kSlabThroughBytes = (size_t)24 << 20;
__device__ __forceinline__ bool slab_through(int slices, int T, int NT, int K, int weight_bytes) {
  return (size_t)slices * T * NT * 64 <= kSlabThroughBytes && (size_t)K * weight_bytes <= (size_t)16 * slices * T;
}
// a wave's raw accumulators to its K-slice's slab [T][16 NT]
// (One branch for all, and rows behind the last dropped by the descriptor: this code runs once a launch and is fetched from
// memory then.)
template <int NTW, int MT>
__device__ __forceinline__ void store_slab(float* __restrict__ slab, bool through, int T, int NT, int mb, int nb, int g, int c, const f32x4_t (&acc)[NTW][MT]) {
  const auto r = __builtin_amdgcn_make_buffer_rsrc(slab, 0, (uint32_t)T * NT * 64u, 0x00020000);
  const uint32_t at = ((uint32_t)(mb + c) * NT + nb) * 64u + g * 16u;
  const auto put = [&](auto aux) {
#pragma unroll
    for (int i = 0; i < NTW; ++i) {
      if (nb + i >= NT) break;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, acc[i][mt]), r, at + (uint32_t)mt * NT * 1024u + i * 64u, 0, decltype(aux)::value);
    }
  };
  if (through) put(std::integral_constant<int, 16>());
  else put(std::integral_constant<int, 0>());
}

// KD 64-deep parts to a K-step.  A phase (READ or MULTIPLY) costs some 340 cycles of barrier, LDS latency and requests even without its MFMAs; in the smallest tiles
// of one-byte weights that is what a 64-deep K-step takes (us each at 128 work-groups, 64 x 128: fp8 0.325, 128-deep ones 0.294; int8 0.402, 0.326; 128 x 128: int8 0.472, 0.424).
// The K-steps behind which another one is requested run in a loop of their own, without a count of what is left to wait for: us a K-step at 250 work-groups, one loop ->
// two, 256 x 192 fp8 1.27 -> 1.14, int8 1.35 -> 1.20; 192 x 192 int8 1.14 -> 1.02; 64 x 128 fp8 0.388 -> 0.367.
// A wave multiplies BM / 2 tokens x 16 NTW weight rows: NTW BM / 8 accumulator registers (256 x 256: 128, and 246 VGPRs
// with the decoded fragments of one K-step).
// SPLIT: grid.z K-slices write raw fp32 accumulators to slab[z][m][n] (see gemm_a8_kernel).
template <int WD, int EPI, int BM, int NTW, bool SPLIT, int KD>
__global__ __launch_bounds__(512) void gemm_wide_kernel(WideArgs a, EpiArgs e) {
  wide_args(a);
  const uint4* __restrict__ W = a.W;
  const uint16_t* __restrict__ x = a.x;
  float* __restrict__ slab = a.slab;
  const int NT = a.NT, KT = a.KT, T = a.T, K = a.K, ldx = a.ldx;
  constexpr int kW = KD * kWideWBytes<WD, NTW>, kStage = kW + KD * BM * 128, kStages = kWideStages<WD, BM, NTW, KD>;
  static_assert(kStages >= 3, "the two wave groups need three stages");
  // waves as 2 (tokens) x 4 (weight rows), each MT 16-token tiles x NTW 16-row weight tiles (4 x 2 waves would read 16 instead of 20 KiB of
  // fragments per K-step at 256 x 256 but decode every weight code four times instead of twice)
  constexpr int MT = BM / 32, WM = 2;
  constexpr int X0 = (MT + 1) / 2, X1 = MT - X0;                 // 8-row activation pieces per wave and 64-deep part: group 0, group 1
  constexpr int WPH = WD == MI_W_BF16 ? 2 : 1, WPK = KD * WPH;   // 1 KiB weight tiles per 16 rows and 64-deep part, and per K-step
  // the 4 NTW WPK weight tiles and BM / 8 activation pieces of a stage over the waves: group 0 (waves 0-3) may bring one more each than group 1
  constexpr int WP0 = (NTW * WPK + 1) / 2, WP1 = NTW * WPK - WP0;
  constexpr int kDma0 = WP0 + KD * X0, kDma1 = WP1 + KD * X1;   // DMAs per wave and stage
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int g = lane >> 4, c = lane & 15;
  const int wm = wave % WM, wn = wave / WM;
  int m0, ntb;
  if (!wide_tile<BM, NTW>(a, m0, ntb)) return;
  int ks0, nks;                               // this slice's K-steps, from K-step ks0 on
  wide_slice<SPLIT, KD>(a, ks0, nks);

  // this lane's DMA sources: weight tiles wt0 .. (fragment order) and X0 (group 1: X1) 8-row pieces of each 64-deep part of the activation tile
  const int grp = __builtin_amdgcn_readfirstlane(wave >> 2), wt0 = grp == 0 ? WP0 * wave : 4 * WP0 + WP1 * (wave - 4);
  const int xp0 = grp == 0 ? X0 * wave : 4 * X0 + X1 * (wave - 4);
  const uint4* wsrc[WP0];
  const uint16_t* xsrc[KD * X0];
#pragma unroll
  for (int i = 0; i < WP0; ++i) {   // tile (row tile / WPK, k tile % WPK); a group-1 wave without an i-th one does not use it
    const int t = min(wt0 + i, 4 * NTW * WPK - 1);
    wsrc[i] = W + ((size_t)min(ntb + t / WPK, NT - 1) * KT + ks0 * WPK + t % WPK) * 64 + lane;
  }
#pragma unroll
  for (int i = 0; i < KD * X0; ++i) {
    const int r = min(xp0 + i % X0, BM / 8 - 1) * 8 + (lane >> 3), sl = lane & 7;
    xsrc[i] = x + (size_t)min(m0 + r, T - 1) * ldx + (size_t)(ks0 * KD + i / X0) * 64 + ((sl ^ xs_swz<WD>(r)) * 8);   // LDS slot sl of row r holds chunk sl ^ swz(r)
  }
  auto issue = [&](int ks, int stage) {
    unsigned char* st = smem + stage * kStage;
#pragma unroll
    for (int i = 0; i < WP1; ++i) glds16(wsrc[i] + (size_t)ks * WPK * 64, st + (wt0 + i) * 1024);
    if constexpr (WP0 > WP1) {
      if (grp == 0) glds16(wsrc[WP1] + (size_t)ks * WPK * 64, st + (wt0 + WP1) * 1024);
    }
    auto bring_x = [&](int d, int i) { glds16(xsrc[d * X0 + i] + (size_t)ks * (64 * KD), st + kW + d * (BM * 128) + (xp0 + i) * 1024); };
#pragma unroll
    for (int d = 0; d < KD; ++d)
#pragma unroll
      for (int i = 0; i < X1; ++i) bring_x(d, i);
    if constexpr (X0 > X1) {
      if (grp == 0) {
#pragma unroll
        for (int d = 0; d < KD; ++d) bring_x(d, X1);
      }
    }
  };

  f32x4_t acc[NTW][MT];
#pragma unroll
  for (int i = 0; i < NTW; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // Schedule.  A K-step of a wave is two phases: READ (its fragments, 20 KiB at BM = 256, from LDS into registers) and MULTIPLY
  // (2 NTW MT MFMAs from registers).  With one barrier per K-step every wave is in the same phase at the same time, the two waves
  // of a SIMD included, and LDS-read time and MFMA time add up: 1.7 us per K-step at BM = 256 against 1.0 us of MFMAs.  Here
  // the two wave groups (waves 0-3 / 4-7 = the two waves of every SIMD) run half a K-step apart -- group 1 executes one
  // barrier more at the start -- so one group multiplies while the other reads:
  //     physical barrier:      P0        P1        P2        P3        P4  ...
  //     group 0 (waves 0-3):   | READ 0  | MUL 0   | READ 1  | MUL 1   | ...
  //     group 1 (waves 4-7):   |         | READ 0  | MUL 0   | READ 1  | MUL 1 ...
  // Stage k is read in [P2k, P2k+2]; K-step k + kStages - 1 goes into the stage of K-step k - 1 (read until P2k), requested by every wave
  // behind its top barrier of iteration k, kStages - 1 K-steps ahead of its first read.  A wave waits for ITS pieces of a
  // stage before the barrier in front of the stage's first read by anyone (group 0: its top barrier; group 1: its second one).
#pragma unroll
  for (int k = 0; k + 1 < kStages; ++k)
    if (k < nks) issue(k, k);
  wide_epi_args<EPI, SPLIT>(e);
  if (grp == 1) {   // its pieces of stage 0 are in before P0
    wait_dma<kDma1, kStages - 2>(nks - 1);
    __builtin_amdgcn_s_barrier();           // P0
  }
  int cur = 0, fill = kStages - 1;          // the stages of K-step ks and of K-step ks + kStages - 1
  auto step = [&](int ks, auto steady) {
    constexpr bool more = decltype(steady)::value;         // K-step ks + kStages - 1 exists: no counting on the way
    if (grp == 0) {                           // own pieces of stage ks
      if constexpr (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kDma0 * (kStages - 2)) : "memory");
      else wait_dma<kDma0, kStages - 2>(nks - 1 - ks);
    }
    __builtin_amdgcn_s_barrier();           // group 0: P2ks | group 1: P2ks+1 -- either way nobody reads stage ks - 1 any more
    const unsigned char* st = smem + cur * kStage;
    u32x4_t b[KD][2][MT], w[NTW][WPK];
#pragma unroll
    for (int i = 0; i < NTW; ++i)
#pragma unroll
      for (int q = 0; q < WPK; ++q) w[i][q] = reinterpret_cast<const u32x4_t*>(st + (wn * NTW + i) * (WPK * 1024) + lane * 16)[q * 64];
#pragma unroll
    for (int d = 0; d < KD; ++d) {
      const uint4* xs = reinterpret_cast<const uint4*>(st + kW + d * (BM * 128));
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int r = wm * (BM / 2) + mt * 16 + c;
        const int ch0 = WD == MI_W_BF16 ? g : 2 * g, ch1 = WD == MI_W_BF16 ? 4 + g : 2 * g + 1;
        b[d][0][mt] = *reinterpret_cast<const u32x4_t*>(&xs[r * 8 + (ch0 ^ xs_swz<WD>(r))]);
        b[d][1][mt] = *reinterpret_cast<const u32x4_t*>(&xs[r * 8 + (ch1 ^ xs_swz<WD>(r))]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (more) issue(ks + kStages - 1, fill);
    __builtin_amdgcn_sched_barrier(0);
    cur = cur + 1 == kStages ? 0 : cur + 1;
    fill = fill + 1 == kStages ? 0 : fill + 1;
    // the fragments are in registers (the empty asm takes them as operands: the compiler's wait for the reads sits in front of it)
#pragma unroll
    for (int i = 0; i < NTW; ++i)
#pragma unroll
      for (int q = 0; q < WPK; ++q) asm volatile("" : "+v"(w[i][q]));
#pragma unroll
    for (int d = 0; d < KD; ++d)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) { asm volatile("" : "+v"(b[d][0][mt])); asm volatile("" : "+v"(b[d][1][mt])); }
    if (grp == 1) {                           // own pieces of stage ks + 1: group 0 reads it behind the next barrier
      if constexpr (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kDma1 * (kStages - 2)) : "memory");
      else if (ks + 1 < nks) wait_dma<kDma1, kStages - 2>(nks - 2 - ks);
    }
    __builtin_amdgcn_s_barrier();           // group 0: P2ks+1 | group 1: P2ks+2
    __builtin_amdgcn_sched_barrier(0);
    // the codes of weight tile i + 1 are decoded between the MFMAs of tile i, whose 16 cycles leave room for three vector instructions each
    u32x4_t a[2], an[2];
    auto piece = [&](const u32x4_t& v4, int q) { const uint32_t v = v4[q >> 1]; return decode2<WD>(v, q & 1); };
    if constexpr (WD != MI_W_BF16) {
#pragma unroll
      for (int q = 0; q < 8; ++q) a[q >> 2][q & 3] = piece(w[0][0], q);
    }
#pragma unroll
    for (int t = 0; t < KD * NTW; ++t) {
      const int d = t / NTW, i = t % NTW;
      if constexpr (WD == MI_W_BF16) { a[0] = w[i][2 * d]; a[1] = w[i][2 * d + 1]; }
#pragma unroll
      for (int m2 = 0; m2 < 2 * MT; ++m2) {   // both halves one after the other: two MFMAs in a row never meet in an accumulator
        const int h = m2 / MT, mt = m2 % MT;
        acc[i][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a[h]), __builtin_bit_cast(bf16x8_t, b[d][h][mt]), acc[i][mt], 0, 0, 0);
        if constexpr (WD != MI_W_BF16) {
          if (t + 1 < KD * NTW) {
#pragma unroll
            for (int q = m2 * 4 / MT; q < (m2 + 1) * 4 / MT; ++q) an[q >> 2][q & 3] = piece(w[(t + 1) % NTW][(t + 1) / NTW], q);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if constexpr (WD != MI_W_BF16) { a[0] = an[0]; a[1] = an[1]; }
    }
  };
  int ks = 0;
  for (; ks + kStages - 1 < nks; ++ks) step(ks, std::true_type());
  for (; ks < nks; ++ks) step(ks, std::false_type());
  if (grp == 0) __builtin_amdgcn_s_barrier();   // the barrier group 1 executed first
  if constexpr (SPLIT) store_slab<NTW, MT>(slab + (size_t)blockIdx.z * T * (NT * 16), slab_through(gridDim.z, T, NT, K, WD == MI_W_BF16 ? 2 : 1), T, NT, m0 + wm * (BM / 2), ntb + wn * NTW, g, c, acc);
  else epilogue_tile<EPI, NTW, MT>(e, T, NT, m0 + wm * (BM / 2), ntb + wn * NTW, g, c, acc);
}

// The same for bf16 weights at 256 x 256, 256 x 192 and 192 x 256 (tokens x weight rows).  A 64-deep stage of these is 56 - 64 KiB, and the LDS holds
// two; the stagger needs a third.  So a K-step is 32 deep (one weight tile per 16 rows; NTW MT MFMAs a wave), the weights ride in four stages, and the
// activations, whose rows are fetched 128 bytes at a time, in three of 64-deep pairs of K-steps: 160 KiB at 256 x 256.  K-step s requests the weights
// of s + 3 and a part of the rows of the pair behind the next, so what K-step s reads was requested by K-step s - 3 at
// the latest and the DMAs of two K-steps stay in flight.
// us a 64-deep K-step on a full chip: 256 x 256 1.46, the other two 1.2; 128 x 256 by 64 0.83.  12288 x 2048 at 777 tokens: 192 work-groups of 256 x 256 54.8,
// 256 of 256 x 192 48.1, 240 of 192 x 256 46.0.
template <int EPI, int BM, int NTW, bool SPLIT>
__global__ __launch_bounds__(512) void gemm_wide16_kernel(WideArgs a, EpiArgs e) {
  wide_args(a);
  const uint4* __restrict__ W = a.W;
  const uint16_t* __restrict__ x = a.x;
  float* __restrict__ slab = a.slab;
  const int NT = a.NT, KT = a.KT, T = a.T, K = a.K, ldx = a.ldx;
  constexpr int MT = BM / 32, WM = 2, kW = NTW * 4096, kX = BM * 128, kXs = 4 * kW;
  constexpr int XP = BM / 64, XH0 = (XP + 1) / 2, XH1 = XP - XH0;     // 8-row activation pieces per wave and pair, those of its first and its second K-step
  constexpr int WP0 = (NTW + 1) / 2, WP1 = NTW - WP0;                 // weight tiles per wave and K-step: waves 0-3, waves 4-7
  static_assert(4 * kW + 3 * kX <= 160 * 1024, "LDS");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int g = lane >> 4, c = lane & 15;
  const int wm = wave % WM, wn = wave / WM;
  int m0, ntb;
  if (!wide_tile<BM, NTW>(a, m0, ntb)) return;
  int ks0, nks;
  wide_slice<SPLIT>(a, ks0, nks);
  const int s0 = 2 * ks0, n = 2 * nks;        // this slice's 32-deep K-steps

  const int grp = __builtin_amdgcn_readfirstlane(wave >> 2), wt0 = grp == 0 ? WP0 * wave : 4 * WP0 + WP1 * (wave - 4);
  const uint4* wsrc[WP0];
  const uint16_t* xsrc[XP];
#pragma unroll
  for (int i = 0; i < WP0; ++i) wsrc[i] = W + ((size_t)min(ntb + wt0 + i, NT - 1) * KT + s0) * 64 + lane;   // (a group-1 wave without an i-th one does not use it)
#pragma unroll
  for (int i = 0; i < XP; ++i) {
    const int r = (XP * wave + i) * 8 + (lane >> 3), sl = lane & 7;
    xsrc[i] = x + (size_t)min(m0 + r, T - 1) * ldx + (size_t)s0 * 32 + ((sl ^ xs_swz<MI_W_BF16>(r)) * 8);
  }
  auto issue_w = [&](int s) {
#pragma unroll
    for (int i = 0; i < WP1; ++i) glds16(wsrc[i] + (size_t)s * 64, smem + (s & 3) * kW + (wt0 + i) * 1024);
    if constexpr (WP0 > WP1) {
      if (grp == 0) glds16(wsrc[WP1] + (size_t)s * 64, smem + (s & 3) * kW + (wt0 + WP1) * 1024);
    }
  };
  auto issue_x = [&](int p, auto half, int stage) {   // a part of this wave's rows of pair p
    constexpr int lo = decltype(half)::value ? XH0 : 0, hi = decltype(half)::value ? XP : XH0;
#pragma unroll
    for (int q = lo; q < hi; ++q) glds16(xsrc[q] + (size_t)p * 64, smem + kXs + stage * kX + (XP * wave + q) * 1024);
  };
  // own pieces of K-step s are in: the requests of the last two K-steps may be out, fewer of them at the end (w: weight tiles a K-step)
  auto wait_at = [&](int s, auto w) {
    constexpr int w1 = decltype(w)::value;
    const int left = n - 1 - s;
    if (left >= 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * w1 + XP) : "memory");
    else if (left == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * w1 + XH1) : "memory");
    else if (left == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(w1) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };

  f32x4_t acc[NTW][MT];
#pragma unroll
  for (int i = 0; i < NTW; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  using First = std::integral_constant<int, 0>;
  using Second = std::integral_constant<int, 1>;
  using Tiles0 = std::integral_constant<int, WP0>;
  using Tiles1 = std::integral_constant<int, WP1>;
  issue_x(0, First(), 0);
  issue_x(0, Second(), 0);
  issue_w(0);
  issue_w(1);
  if (n > 2) {
    issue_x(1, First(), 1);
    issue_w(2);
    issue_x(1, Second(), 1);
  }
  wide_epi_args<EPI, SPLIT>(e);
  if (grp == 1) {
    wait_at(0, Tiles1());
    __builtin_amdgcn_s_barrier();           // P0
  }
  auto step = [&](int s, auto half, int xcur, int xfill, auto steady) {
    constexpr bool more = decltype(steady)::value;
    if (grp == 0) {
      if constexpr (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * WP0 + XP) : "memory");
      else wait_at(s, Tiles0());
    }
    __builtin_amdgcn_s_barrier();           // group 0: P2s | group 1: P2s+1
    const unsigned char* st = smem + (s & 3) * kW;
    const uint4* xs = reinterpret_cast<const uint4*>(smem + kXs + xcur * kX);
    u32x4_t b[MT], a[NTW];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int r = wm * (BM / 2) + mt * 16 + c;
      b[mt] = *reinterpret_cast<const u32x4_t*>(&xs[r * 8 + ((4 * decltype(half)::value + g) ^ xs_swz<MI_W_BF16>(r))]);
    }
#pragma unroll
    for (int i = 0; i < NTW; ++i) a[i] = *reinterpret_cast<const u32x4_t*>(st + (wn * NTW + i) * 1024 + lane * 16);
    __builtin_amdgcn_sched_barrier(0);
    if (more || s + 3 < n) issue_w(s + 3);
    if (more || (s >> 1) + 2 < (n >> 1)) issue_x((s >> 1) + 2, half, xfill);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) asm volatile("" : "+v"(b[mt]));
#pragma unroll
    for (int i = 0; i < NTW; ++i) asm volatile("" : "+v"(a[i]));
    if (grp == 1) {
      if constexpr (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * WP1 + XP) : "memory");
      else if (s + 1 < n) wait_at(s + 1, Tiles1());
    }
    __builtin_amdgcn_s_barrier();           // group 0: P2s+1 | group 1: P2s+2
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NTW; ++i)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        acc[i][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a[i]), __builtin_bit_cast(bf16x8_t, b[mt]), acc[i][mt], 0, 0, 0);
  };
  int xcur = 0, xfill = 2;
  auto pair = [&](int s, auto steady) {
    step(s, First(), xcur, xfill, steady);
    step(s + 1, Second(), xcur, xfill, steady);
    xcur = xcur == 2 ? 0 : xcur + 1;
    xfill = xfill == 2 ? 0 : xfill + 1;
  };
  int s = 0;
  for (; s + 4 < n; s += 2) pair(s, std::true_type());      // both request, and two K-steps' DMAs are behind what they wait for
  for (; s < n; s += 2) pair(s, std::false_type());
  if (grp == 0) __builtin_amdgcn_s_barrier();   // the barrier group 1 executed first
  if constexpr (SPLIT) store_slab<NTW, MT>(slab + (size_t)blockIdx.z * T * (NT * 16), slab_through(gridDim.z, T, NT, K, 2), T, NT, m0 + wm * (BM / 2), ntb + wn * NTW, g, c, acc);
  else epilogue_tile<EPI, NTW, MT>(e, T, NT, m0 + wm * (BM / 2), ntb + wn * NTW, g, c, acc);
}

// tiles of one-byte weights with 128-deep K-steps: what fits the LDS three times
constexpr bool wide_tile_deep(int wd, int bm, int ntw) { return wd != MI_W_BF16 && 2 * (ntw * 4096 + bm * 128) * 3 <= 160 * 1024; }
// bf16 tiles whose 64-deep stages fit the LDS twice only: 256 x 192, 192 x 256, 256 x 256
constexpr bool wide_tile_by_32(int wd, int bm, int ntw) { return wd == MI_W_BF16 && 3 * (ntw * 8192 + bm * 128) > 160 * 1024; }

template <int WD, int EPI, int BM, int NTW, bool SPLIT>
static int launch_gemm_wide_t(const LinearW& w, int T, const uint16_t* x, int ldx, const EpiArgs& e, hipStream_t s, int KS, float* slab) {
  const int NT = w.N / 16, mtiles = ceil_div(T, BM), per = ceil_div(mtiles * ceil_div(NT, 4 * NTW), 8);
  const dim3 grid(8 * per, 1, KS);
  WideArgs a{reinterpret_cast<const uint4*>(w.w), x, slab, NT, w.K / tile_k(WD), T, w.K, ldx, mtiles, per, mtiles == 1 ? ~0u : (unsigned)((1ull << 32) / mtiles), 0};
  if constexpr (wide_tile_by_32(WD, BM, NTW)) {
    constexpr int lds = 4 * NTW * 4096 + 3 * BM * 128;
    const auto fn = gemm_wide16_kernel<EPI, BM, NTW, SPLIT>;
    MI_TRY_(ensure_dynamic_lds(reinterpret_cast<const void*>(fn), lds));
    a.kper = ceil_div(w.K / 64, KS);
    hipLaunchKernelGGL(fn, grid, dim3(512), lds, s, a, e);
  } else {
    const auto launch = [&](auto deep) {
      constexpr int KD = decltype(deep)::value, lds = kWideStages<WD, BM, NTW, KD> * KD * (kWideWBytes<WD, NTW> + BM * 128);
      const auto fn = gemm_wide_kernel<WD, EPI, BM, NTW, SPLIT, KD>;
      MI_TRY_(ensure_dynamic_lds(reinterpret_cast<const void*>(fn), lds));
      a.kper = ceil_div(w.K / (64 * KD), KS);
      hipLaunchKernelGGL(fn, grid, dim3(512), lds, s, a, e);
      return (int)MI_OK;
    };
    // 128-deep K-steps where a phase would be shorter than its reads: weights of a byte in the smallest tiles, if no slice of K stays empty by them
    bool deep = false;
    if constexpr (wide_tile_deep(WD, BM, NTW)) {
      deep = w.K % 128 == 0 && (KS - 1) * ceil_div(w.K / 128, KS) < w.K / 128;
      if (deep) MI_TRY_(launch(std::integral_constant<int, 2>()));
    }
    if (!deep) MI_TRY_(launch(std::integral_constant<int, 1>()));
  }
  MI_HIP(hipGetLastError());
  return MI_OK;
}

template <int WD, int BM, int NTW>
static int launch_gemm_wide_bm(const LinearW& w, int T, const uint16_t* x, int ldx, int epi, const EpiArgs& e, hipStream_t s,
                               int KS, float* ws, SlabSum* defer) {
  MI_CHECK(e.rs_n == 0.f || BM == 32 || KS > 1, "gemm_wide: the parts of a norm are for blocks of 32 tokens");
  if (KS > 1) {
    MI_TRY_((launch_gemm_wide_t<WD, EPI_F32, BM, NTW, true>(w, T, x, ldx, e, s, KS, ws)));
    const SlabSum sum{ws, KS, T, w.N, e.scale, e.bias, e.row_scale, e.rs_n, e.rs_eps};
    if (defer && (epi == EPI_RESID || epi == EPI_F32)) { *defer = sum; return MI_OK; }
    return launch_splitk_reduce(sum, epi, e, s);
  }
#define MI_GW(EPI_) return launch_gemm_wide_t<WD, EPI_, BM, NTW, false>(w, T, x, ldx, e, s, 1, nullptr)
  switch (epi) {
    case EPI_QKV: MI_GW(EPI_QKV);
    case EPI_SWIGLU: MI_GW(EPI_SWIGLU);
    case EPI_RESID: MI_GW(EPI_RESID);
    case EPI_F32: MI_GW(EPI_F32);
  }
  if constexpr (WD == MI_W_BF16)
    switch (epi) {
      case EPI_RELU2: MI_GW(EPI_RELU2);
      case EPI_GLU_CLIP: MI_GW(EPI_GLU_CLIP);
      case EPI_SOFTCAP: MI_GW(EPI_SOFTCAP);
      case EPI_HEADS_KV: MI_GW(EPI_HEADS_KV);
    }
#undef MI_GW
  set_error("gemm_wide: this epilogue is not built for this weight type");
  return MI_EINVAL;
}

// bm x 64 ntw tiles, K over ks slices (ks > 1: ws holds them)
template <int WD>
int launch_gemm_wide_wd(const LinearW& w, int T, const uint16_t* x, int ldx, int epi, const EpiArgs& e, hipStream_t s, int bm, int ntw, int ks, float* ws,
                        SlabSum* defer) {
#define MI_GT(BM_, NTW_) \
  if (bm == BM_ && ntw == NTW_) return launch_gemm_wide_bm<WD, BM_, NTW_>(w, T, x, ldx, epi, e, s, ks, ws, defer)
  MI_GT(32, 2); MI_GT(32, 3); MI_GT(32, 4);
  MI_GT(64, 2); MI_GT(64, 3); MI_GT(64, 4);
  MI_GT(96, 2); MI_GT(96, 3); MI_GT(96, 4);
  MI_GT(128, 2); MI_GT(128, 3); MI_GT(128, 4);
  MI_GT(160, 2); MI_GT(160, 3); MI_GT(160, 4);
  MI_GT(192, 2); MI_GT(192, 3); MI_GT(192, 4);
  MI_GT(256, 2); MI_GT(256, 3); MI_GT(256, 4);
#undef MI_GT
  set_error("gemm_wide: no such tile");
  return MI_EINVAL;
}

}  // namespace mi
