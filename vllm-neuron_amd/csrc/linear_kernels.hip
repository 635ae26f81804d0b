// Weight-quantized linear layers for gfx950 (MI355X).
//
//   y[m, n] = (sum_k x[m, k] * q[n, k]) * scale[n] (+ bias[n])      q in {e4m3fn, int8, bf16}
//
// Replaces the NxDI quantized Column/RowParallel linears the reference reaches through
// /root/reference/vllm_neuron/worker/neuronx_distributed_model_loader.py:339-348, with the
// quantization keys of loader.py:886-898.
//
// Storage: the library owns the weights, so they are kept in the shape the matrix cores
// want.  A tile is 16 output rows x 64 bytes of K (fp8/int8; 32 elements for bf16) = 1 KiB
// laid out lane-linear: lane l holds the 16 bytes of row (l & 15), k-chunk (l >> 4).  One
// 16-byte load per lane is then (a) a perfectly coalesced 1 KiB wave read and (b) exactly
// the A operand of v_mfma_f32_16x16x32_bf16 after an in-register fp8->bf16 decode (two
// k-steps per load for the 1-byte types).  Tiles of one 16-row group are contiguous along K,
// so a wave streams a dense byte range.
//
// Token generation of up to 4 rows, where no norm was handed on and gemv_few_rows_in_regs says no: the kernels of linear_device.h — pure weight streaming, HBM-bound.  x lives in LDS in
//   fragment order; every wave streams a K-slice of one row-tile with 2 x 8 KiB in flight;
//   the MFMA does the dot products AND the cross-lane reduction; waves combine through LDS
//   in a fixed order (deterministic, no atomics).  5 .. 32 rows, and up to 4 behind a norm that was handed on: gemv_regs.h, x in registers.
// Context encoding: gemm_wide.h; gemm_kernel here (128 x 128 tile, x through swizzled LDS, W straight
//   from global in fragment order) for what that does not take.
//
// All share one epilogue on D[n = 4g + r][m = c] (lane = 16 g + c): dequant scale, bias,
// then fp32 store | RoPE + q/KV-pool scatter | SwiGLU.

#include <cmath>

#include "linear_kernels.h"

#include "gemm_wide.h"
#include "linear_device.h"

namespace mi {

// instantiated in gemv_bf16.hip / gemv_f8.hip / gemv_i8.hip
template <int WD>
int launch_gemv_wd(const LinearW& w, int M, int pro, const ProArgs& p, int epi, const EpiArgs& e, hipStream_t s);
extern template int launch_gemv_wd<MI_W_BF16>(const LinearW&, int, int, const ProArgs&, int, const EpiArgs&, hipStream_t);
extern template int launch_gemv_wd<MI_W_F8E4M3>(const LinearW&, int, int, const ProArgs&, int, const EpiArgs&, hipStream_t);
extern template int launch_gemv_wd<MI_W_INT8>(const LinearW&, int, int, const ProArgs&, int, const EpiArgs&, hipStream_t);

template <int WD>
int launch_gemv_regs_wd(const LinearW& w, int M, const uint16_t* x, int ldx, int epi, const EpiArgs& e, hipStream_t s, float* ws, size_t ws_bytes, SlabSum* defer, bool split_as_deferred);
template <int WD> bool gemv_regs_fits_wd(int M, int N, int K, size_t ws_bytes);
template <int WD> double gemv_regs_us_wd(int M, int N, int K, size_t ws_bytes, bool deferred);

static bool gemv_regs_fits(const LinearW& w, int M, size_t ws_bytes) {
  switch (w.wd) {
    case MI_W_BF16: return gemv_regs_fits_wd<MI_W_BF16>(M, w.N, w.K, ws_bytes);
    case MI_W_F8E4M3: return gemv_regs_fits_wd<MI_W_F8E4M3>(M, w.N, w.K, ws_bytes);
    case MI_W_INT8: return gemv_regs_fits_wd<MI_W_INT8>(M, w.N, w.K, ws_bytes);
  }
  return false;
}
template <int WD> bool gemv_regs_whole_wd(int M, int N, int K, size_t ws_bytes);
bool gemv_regs_whole(const LinearW& w, int M, size_t ws_bytes) {
  switch (w.wd) {
    case MI_W_BF16: return gemv_regs_whole_wd<MI_W_BF16>(M, w.N, w.K, ws_bytes);
    case MI_W_F8E4M3: return gemv_regs_whole_wd<MI_W_F8E4M3>(M, w.N, w.K, ws_bytes);
    case MI_W_INT8: return gemv_regs_whole_wd<MI_W_INT8>(M, w.N, w.K, ws_bytes);
  }
  return false;
}
bool gemv_regs_holds(const LinearW& w) { return ceil_div(w.K / tile_k(w.wd), kGemvWaves) <= regs_max_tiles(w.wd); }
// From 5 rows on (us per call; the LDS kernels with the norm in front of them / these behind a norm kernel; contexts of 500, TinyLlama 200):
//   8B fp8, 16 layers:  8 rows 1472 / 1332, 16 rows 1758 / 1527, 32 rows 2282 / 2117;   4 rows 1191 / 1277
//   8B bf16:            8 rows 1949 / 1857, 24 rows 2526 / 2298
//   7B int8, 14 layers: 5 rows 1454 / 1330, 14 rows 1699 / 1446, 24 rows 2332 / 1789
//   TinyLlama bf16:     1 row 876 / 1034, 16 rows 1389 / 1210, 30 rows 1501 / 1450
//   16 layers of width 256 / 512 / 1024 / 1536, bf16: 5 rows 572 / 467, 604 / 538, 637 / 556, 745 / 673; 32 rows 739 / 604, 790 / 626, 850 / 667, 1001 / 926
// Up to 4 rows the norm inside the weight stream's kernel and its two to eight waves per row-tile win, unless the projection in front has handed that norm on (run_linear).
bool gemv_in_regs(const LinearW& w, int M, size_t ws_bytes) { return M >= 5 && M <= 32 && gemv_regs_fits(w, M, ws_bytes); }
// Up to 4 rows of bf16 activations (nothing to fuse in front).  They win where a wave's weights of a row-tile are one batch of requests and each work-group has one
// row-tile (the chain to the first request is shorter: no staging) or eight and more (the tiles follow each other without a barrier on the way), and, where the sums have a
// taker, on rows of at most half the CUs: K goes over the other half.  us a launch at 1 / 4 rows, LDS kernels -> these: 2048 x 2048 bf16 5.3 / 5.5 -> 4.3 / 4.3 with a
// taker, 4.9 / 5.2 without; 2048 x 7680 bf16 9.0 / 9.3 -> 8.2 / 8.6 and 2048 x 14336 13.8 / 14.4 -> 12.5 / 12.7 with one; 4096 x 4096 fp8 7.4 -> 6.5, int8 7.7 -> 7.1;
// 32768 x 2048 bf16 26.2 -> 23.7.  In whole calls, us a layer, rule off and on in turn: 2048 wide fp8 1.0 .. 1.3 of 33 - 37, int8 1.4 .. 1.7 of 35 - 39, bf16 nothing to 0.3; 3584 wide fp8 0.6 .. 1.3
// of 70, 4096 wide bf16 1 .. 2 of 93, the others nothing to 0.6 (two models of the same weights differ by 0.3).  Not between: 8192 x 2048 bf16 8.1 -> 9.3, 15360 x 2048 12.7 -> 13.4, 5120 x 4096 fp8 7.1 -> 7.5; nor K in two batches: 3584 x 3584 bf16 7.6 -> 7.7.
bool gemv_few_rows_in_regs(const LinearW& w, int M, size_t ws_bytes, bool deferred) {
  int cus = 0;
  if (M < 1 || M > 4 || device_num_cu(&cus) != MI_OK) return false;
  const int NT = w.N / 16;
  if (ceil_div(w.K / tile_k(w.wd), kGemvWaves) <= 8 && (NT <= cus || NT >= 8 * cus)) return true;
  return deferred && 2 * NT <= cus && gemv_regs_fits(w, M, ws_bytes);
}
static int gemm_wide_mode() {   // MI355X_GEMM_WIDE: 0 never, 1 whenever the shape allows, unset: by size
  static const int m = [] { const char* v = getenv("MI355X_GEMM_WIDE"); return v ? atoi(v) : -1; }();
  return m;
}
static int gemm_wide_bm() {      // MI355X_GEMM_WIDE_BM: 128 / 256 forces the token block (default: by grid size)
  static const int m = [] { const char* v = getenv("MI355X_GEMM_WIDE_BM"); const int b = v ? atoi(v) : 0; return b == 128 || b == 256 ? b : 0; }();
  return m;
}
int launch_gemv_regs(const LinearW& w, int M, const uint16_t* x, int ldx, int epi, const EpiArgs& e, hipStream_t s, float* ws, size_t ws_bytes, SlabSum* defer,
                     bool split_as_deferred) {
  if (defer) *defer = SlabSum();
  MI_CHECK(M >= 1 && M <= 32 && w.N % 16 == 0 && w.K % 64 == 0 && ldx % 8 == 0, "gemv_regs: 1 .. 32 rows, N % 16 == 0, K % 64 == 0, row stride a multiple of 8");
  switch (w.wd) {
    case MI_W_BF16: return launch_gemv_regs_wd<MI_W_BF16>(w, M, x, ldx, epi, e, s, ws, ws_bytes, defer, split_as_deferred);
    case MI_W_F8E4M3: return launch_gemv_regs_wd<MI_W_F8E4M3>(w, M, x, ldx, epi, e, s, ws, ws_bytes, defer, split_as_deferred);
    case MI_W_INT8: return launch_gemv_regs_wd<MI_W_INT8>(w, M, x, ldx, epi, e, s, ws, ws_bytes, defer, split_as_deferred);
  }
  set_error("gemv_regs: bad weight dtype");
  return MI_EINVAL;
}

size_t gemv_lds_bytes(int M, int K) { return gemv_image_lds_bytes(M, K); }
bool gemv_fits(int M, int K) { (void)K; return gemv_rows_fit(M); }

int launch_gemv(const LinearW& w, int M, int pro, const ProArgs& p, int epi, const EpiArgs& e, hipStream_t s) {
  MI_CHECK(M >= 1 && M <= 16, "gemv: M must be 1..16");
  MI_CHECK(!e.next_x || (epi == EPI_RESID && e.ld_out == w.N), "gemv: a norm handed on is for residuals, rows side by side");
  MI_CHECK(w.N % 16 == 0 && w.K % 64 == 0, "gemv: N % 16 == 0 and K % 64 == 0 required");
  switch (w.wd) {
    case MI_W_BF16: return launch_gemv_wd<MI_W_BF16>(w, M, pro, p, epi, e, s);
    case MI_W_F8E4M3: return launch_gemv_wd<MI_W_F8E4M3>(w, M, pro, p, epi, e, s);
    case MI_W_INT8: return launch_gemv_wd<MI_W_INT8>(w, M, pro, p, epi, e, s);
  }
  set_error("gemv: bad weight dtype");
  return MI_EINVAL;
}

// =====================================================================================
// GEMM (context encoding)
// =====================================================================================
// Work-group tile 128 (n) x 128 (m); 4 waves as 2 (n) x 2 (m), each 64 x 64 = 4 x 4 MFMA tiles.
// x tile [128 m][64 k] bf16 through LDS (16-byte chunks XOR-swizzled by row); W fragments
// straight from the pre-tiled global image.
constexpr int kBM = 128, kBN = 128, kBK = 64;


// SPLIT: grid.z K-slices write raw fp32 accumulators to slab[z][m][n] (see gemm_a8_kernel).
// Registers are kept under 170 per lane so that three work-groups share a CU (the same lesson as
// the FP8 GEMM): the weight tiles of a K-step are decoded once into their A fragments, the raw
// registers are refilled with the next K-step's tiles straight away, and the activation
// fragments are read per 16-token tile instead of all at once.
template <int WD, int EPI, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WD == MI_W_BF16 ? 2 : 3, WD == MI_W_BF16 ? 2 : 3))) void gemm_kernel(const uint4* __restrict__ W, int NT, int KT, int T, int K,
                                                   const uint16_t* __restrict__ x, int ldx, EpiArgs e,
                                                   float* __restrict__ slab) {
  __shared__ __attribute__((aligned(16))) uint4 xs[kBM * 8];  // 16 KiB
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int g = lane >> 4, c = lane & 15;
  const int wn = wave >> 1, wm = wave & 1;
  // XCD-aware tile order (see gemm_a8_kernel): XCD = linear id % 8 owns every eighth weight slab
  // and walks all token blocks of a slab back to back
  const int mtiles = ceil_div(T, kBM), ntiles = ceil_div(NT, kBN / 16);
  const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
  const int mblk = seq % mtiles, nblk = (seq / mtiles) * 8 + xcd;
  if (nblk >= ntiles) return;
  const int m0 = mblk * kBM, nt0 = nblk * (kBN / 16) + wn * 4;
  const int nks_all = K / kBK;
  const int ks_per = SPLIT ? ceil_div(nks_all, (int)gridDim.z) : nks_all;
  const int ks_beg = SPLIT ? (int)blockIdx.z * ks_per : 0;
  const int nks = min(ks_beg + ks_per, nks_all);
  constexpr int WPK = (WD == MI_W_BF16) ? 2 : 1;  // weight tiles per K-step

  f32x4_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // x staging: thread -> rows (tid/8 + 32 i), 16-byte chunk tid%8
  const int srow = tid >> 3, sch = tid & 7;
  u32x4_t xr[4], wr[4][WPK];
  auto load_x = [&](int ks) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = min(m0 + srow + 32 * i, T - 1);   // rows past T: a copy of the last row, never stored
      xr[i] = *reinterpret_cast<const u32x4_t*>(x + (size_t)m * ldx + ks * kBK + sch * 8);
    }
  };
  auto load_w = [&](int ks) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int t = 0; t < WPK; ++t)
        wr[i][t] = *reinterpret_cast<const u32x4_t*>(W + ((size_t)min(nt0 + i, NT - 1) * KT + ks * WPK + t) * 64 + lane);
  };

  if (ks_beg < nks) {
    load_x(ks_beg);
    load_w(ks_beg);
  }
  for (int ks = ks_beg; ks < nks; ++ks) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = srow + 32 * i;
      *reinterpret_cast<u32x4_t*>(&xs[r * 8 + (sch ^ xs_swz<WD>(r))]) = xr[i];
    }
    bf16x8_t a0[4], a1[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (WD == MI_W_BF16) {
        a0[i] = __builtin_bit_cast(bf16x8_t, wr[i][0]);
        a1[i] = __builtin_bit_cast(bf16x8_t, wr[i][1]);
      } else {
        const u32x4_t w4 = wr[i][0];
        a0[i] = decode8<WD>(w4[0], w4[1]);
        a1[i] = decode8<WD>(w4[2], w4[3]);
      }
    }
    __syncthreads();
    if (ks + 1 < nks) {      // the raw registers are free again: next K-step's operands
      load_x(ks + 1);
      load_w(ks + 1);
    }
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const int r = wm * 64 + mt * 16 + c;
      const int ch0 = (WD == MI_W_BF16) ? g : 2 * g, ch1 = (WD == MI_W_BF16) ? 4 + g : 2 * g + 1;
      const bf16x8_t b0 = __builtin_bit_cast(bf16x8_t, xs[r * 8 + (ch0 ^ xs_swz<WD>(r))]);
      const bf16x8_t b1 = __builtin_bit_cast(bf16x8_t, xs[r * 8 + (ch1 ^ xs_swz<WD>(r))]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[i][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[i], b0, acc[i][mt], 0, 0, 0);
        acc[i][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[i], b1, acc[i][mt], 0, 0, 0);
      }
    }
    __syncthreads();
  }

#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (nt0 + i >= NT) continue;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const int m = m0 + wm * 64 + mt * 16 + c;
      if (m >= T) continue;
      const int n0 = (nt0 + i) * 16 + g * 4;
      if constexpr (SPLIT) {
        *reinterpret_cast<float4*>(slab + ((size_t)blockIdx.z * T + m) * (NT * 16) + n0) =
            make_float4(acc[i][mt][0], acc[i][mt][1], acc[i][mt][2], acc[i][mt][3]);
      } else {
        epilogue<EPI>(e, m, n0, acc[i][mt]);
      }
    }
  }
}

template <int EPI, bool PARTS>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ slab, int KS, int T, int N, EpiArgs e);

// K-split for grids too small to occupy the chip (768 work-groups are resident at once): below 256
// tiles aim for 512 work-groups, below 384 for 768 (rule measured on the FP8 GEMM).
static int gemm_pick_splitk(int tiles, int nks, int T, int N, size_t ws_bytes) {
  if (!ws_bytes || tiles >= 384) return 1;
  int KS = min(min(8, nks), ceil_div(tiles < 256 ? 512 : 768, tiles));
  while (KS > 1 && (size_t)KS * T * N * sizeof(float) > ws_bytes) --KS;
  return KS;
}

template <int WD>
static int launch_gemm_wd(const LinearW& w, int T, const uint16_t* x, int ldx, int epi, const EpiArgs& e, hipStream_t s,
                          float* splitk_ws, size_t splitk_ws_bytes, SlabSum* defer) {
  const int NT = w.N / 16, KT = w.K / tile_k(WD);
  const int mtiles = ceil_div(T, kBM), ntiles = ceil_div(w.N, kBN);
  const int KS = gemm_pick_splitk(mtiles * ntiles, w.K / kBK, T, w.N, splitk_ws ? splitk_ws_bytes : 0);
  dim3 grid(8 * mtiles * ceil_div(ntiles, 8), 1, KS);
  const uint4* W = reinterpret_cast<const uint4*>(w.w);
#define MI_G(EPI_) \
  do { \
    if (KS == 1) { \
      hipLaunchKernelGGL((gemm_kernel<WD, EPI_, false>), grid, dim3(256), 0, s, W, NT, KT, T, w.K, x, ldx, e, nullptr); \
    } else { \
      hipLaunchKernelGGL((gemm_kernel<WD, EPI_, true>), grid, dim3(256), 0, s, W, NT, KT, T, w.K, x, ldx, e, splitk_ws); \
      if (defer && (EPI_ == EPI_RESID || EPI_ == EPI_F32)) { *defer = SlabSum{splitk_ws, KS, T, w.N, e.scale, e.bias, e.row_scale}; } \
      else hipLaunchKernelGGL((splitk_reduce_kernel<EPI_, false>), dim3(ceil_div(T * (w.N / 4), 256)), dim3(256), 0, s, splitk_ws, KS, T, w.N, e); \
    } \
  } while (0)
  if (epi == EPI_QKV) MI_G(EPI_QKV);
  else if (epi == EPI_SWIGLU) MI_G(EPI_SWIGLU);
  else if (epi == EPI_RESID) MI_G(EPI_RESID);
  else if (epi >= EPI_RELU2) {
    if constexpr (WD == MI_W_BF16) {
      if (epi == EPI_RELU2) MI_G(EPI_RELU2);
      else if (epi == EPI_GLU_CLIP) MI_G(EPI_GLU_CLIP);
      else if (epi == EPI_SOFTCAP) MI_G(EPI_SOFTCAP);
      else MI_G(EPI_HEADS_KV);
    } else { set_error("gemm: this epilogue is built for bf16 weights"); return MI_EINVAL; }
  } else MI_G(EPI_F32);
#undef MI_G
  MI_HIP(hipGetLastError());
  return MI_OK;
}


// instantiated in gemm_wide_bf16.hip / gemm_wide_f8.hip / gemm_wide_i8.hip
extern template int launch_gemm_wide_wd<MI_W_BF16>(const LinearW&, int, const uint16_t*, int, int, const EpiArgs&, hipStream_t, int, int, int, float*, SlabSum*);
extern template int launch_gemm_wide_wd<MI_W_F8E4M3>(const LinearW&, int, const uint16_t*, int, int, const EpiArgs&, hipStream_t, int, int, int, float*, SlabSum*);
extern template int launch_gemm_wide_wd<MI_W_INT8>(const LinearW&, int, const uint16_t*, int, int, const EpiArgs&, hipStream_t, int, int, int, float*, SlabSum*);

// Which tile and K-split: the cheapest of a model of the kernel, us, fitted to 9334 launches: 24 projections of TinyLlama, Llama-8B, Qwen2.5-7B and the layer stacks, 70 ..
// 2000 tokens, the tiles and up to nine slices whose cost came near the least, weights from memory (enough copies in turn to fill the caches).  The choice takes 1.1 % longer than the
// fastest on average with bf16 weights, 0.8 % with fp8, 0.6 % with int8; with the constants before, 2.8, 1.1 and 0.9 %, and without blocks of 96 and 160 tokens 3.9, 2.5 and 3.5.
// Over 50 projections, 30 of them others, 33 .. 2048 tokens: 1.4, 1.0 and 0.7 % where a norm takes the sum, 1.7, 1.6 and 1.5 % where a launch does (before: 3.4, 3.9, 2.0 and 2.5, 2.8, 1.7); fitted to
// all of them it is no better.
// The kernel holds more than half of a CU's LDS, i.e. ONE work-group per CU, so a launch is rounds of 32 work-groups on each of the eight XCDs:
// a round a ramp and epilogue that grow with the tile, beside its K-steps, whose time grows from an almost empty to a full chip; and the weights' stream, where it binds.
// A K-split writes its slabs, and a second launch sums them, or the row norm that follows reads them.
// Unsplit tiles on half of the CUs at most take 12 % more than that, inside a call above all: prompts of 34 .. 300 tokens of ten models in the same process, factor 1, 1.06, 1.12, 1.2:
// -, 0.2, 0.3, 0.2 us a layer less with bf16 weights, -, 0.4, 0.5, 0.3 with fp8, -, 0.04, 0.08, 0.11 with int8; 2560 wide bf16, 40 tokens, 475 -> 453 us a call (gate | up on 112 CUs -> 224).  Where a
// launch sums the slices the choice is 1.7, 1.3 and 1.2 % from the fastest with it.
// What blocks of 96 and 160 tokens are for, us, best of the others -> best: 28672 x 4096 bf16 300 tokens 77.5 -> 67.4, 777 tokens 174 -> 160, fp8 90 tokens 30.6 -> 26.8, 300
// tokens 75.0 -> 66.6; 37888 x 3584 int8 90 tokens 49.2 -> 40.6, 777 tokens 211 -> 190; 12288 x 2048 bf16 777 tokens 47.2 -> 39.4.
// Against the best of 128 x 256 and 256 x 256 alone, us: int8 gate|up of the 7B model at 188 tokens 79 -> 60 (148 tiles of 256 x 256 on 256 CUs, 73 % of
// each filled; 198 of 192 x 192), its down projection 41.6 -> 34.4; bf16 gate|up of TinyLlama 700 tokens 51.6 -> 35.4, 200 tokens 28.4 -> 21.4;
// fp8 QKV of the 8B model 1400 tokens 82.6 -> 63.9; bf16 down projection of 2048 x 14336 at 100 tokens 26.4 -> 17.6.
struct WidePlan { int bm, ntw, ks; double us; };
static WidePlan gemm_wide_plan(int T, int N, int K, size_t ws_bytes, int wd, bool deferred) {
  int cus = 256;
  if (device_num_cu(&cus) != MI_OK || cus < 8) cus = 256;
  struct Model {
    double lo[4], hi[4];           // us per 64-deep K-step on an almost empty chip and on a full one: {1, m ntw, m, ntw}, m = bm / 64
    double deep[2], by_32[4];      // lo and hi: factors of 128-deep K-steps; of 256 x 256 and of the other two tiles with 32-deep K-steps (hi as inside long calls)
    double launch, ramp, area;     // a launch; a round, and what it grows by with m ntw
    double full, full_area;        // factor of a grid without a CU to spare: the slowest decides
    double stream, slab;           // MB of weights a us; us per MB of slabs written
  };
  static const Model kModel[3] = {
      {{0.0018, 0.0429, 0.0171, 0.0848}, {0.0016, 0.0208, 0.0944, 0.1035}, {1, 1}, {0.8862, 1.39, 0.7131, 1.13}, 3.405, 2.328, 0.3204, 1.0014, 0.0029, 6.604, 0.1129},
      {{0.0094, 0.0435, 0.0163, 0.0335}, {0.0129, 0.0545, 0.0524, 0.0468}, {0.8062, 0.9204}, {0, 0, 0, 0}, 4.852, 1.738, 0.4059, 1.0135, 0.0021, 7.348, 0.0531},
      {{0.0182, 0.0154, 0.0396, 0.1147}, {0.0296, 0.0403, 0.0633, 0.1088}, {0.7322, 0.949}, {0, 0, 0, 0}, 5.493, 1.132, 0.488, 1.0151, 0.0012, 7.284, 0.0479}};
  const Model& r = kModel[wd];
  const int nks = K / 64;
  const double mb = (double)T * N * 4e-6, stream = (double)N * K * elem_bytes(wd) * 1e-6 / r.stream;
  WidePlan best{0, 4, 1, 0.};   // (bm 0: none compared yet; one slice is always allowed, so there is one)
  for (const int bm : {32, 64, 96, 128, 160, 192, 256})
    for (int ntw = 2; ntw <= 4; ++ntw) {
      if ((bm == 32) != (T <= 32)) break;        // (32 tokens are the cheapest block that holds them: every term grows with m)
      const double m = bm / 64., area = m * ntw;
      const auto us = [&](const double (&k)[4]) { return k[0] + k[1] * area + k[2] * m + k[3] * ntw; };
      const bool by_32 = wide_tile_by_32(wd, bm, ntw), deep_tile = wide_tile_deep(wd, bm, ntw) && K % 128 == 0;
      const int tiles = ceil_div(T, bm) * ceil_div(N, 64 * ntw);
      for (int ks = 1; ks <= 10; ++ks) {
        const int per = ceil_div(nks, ks);
        if (ks > 1 && (per < 4 || (ks - 1) * per >= nks || (size_t)ks * T * N * sizeof(float) > ws_bytes)) continue;
        double lo = by_32 ? r.by_32[area == 16 ? 0 : 2] : us(r.lo), hi = by_32 ? r.by_32[area == 16 ? 1 : 3] : us(r.hi);
        if (deep_tile && (ks - 1) * ceil_div(K / 128, ks) < K / 128) {   // (as the launch: where 128-deep K-steps leave no slice empty)
          lo *= r.deep[0];
          hi *= r.deep[1];
        }
        const int rounds = ceil_div(ceil_div(tiles, 8) * ks, std::max(1, cus / 8));
        double body = rounds * (r.ramp + r.area * area + per * (lo + (hi - lo) * std::min(1.0, (double)tiles * ks / cus)));
        if (rounds * cus - tiles * ks < 6) body *= r.full + r.full_area * area;
        double cost = r.launch + std::sqrt(body * body + stream * stream);
        if (ks > 1) cost += r.slab * ks * mb + (deferred ? 0.144 * ks * mb : 3.38 + 0.113 * (ks + 1) * mb);
        else if (2 * tiles <= cus) cost *= 1.12;   // (half of the CUs at most: longer inside a call than alone)
        if (best.bm == 0 || cost < best.us) best = WidePlan{bm, ntw, ks, cost};
      }
    }
  return best;
}
static int gemm_wide_ks() {      // MI355X_GEMM_WIDE_KS: 1 = never split K in the wide kernel
  static const int m = [] { const char* v = getenv("MI355X_GEMM_WIDE_KS"); return v ? atoi(v) : 0; }();
  return m;
}
// Rows beside which the register kernel takes in more of the activations than of the weights' share of a CU, in front of the first weights; the wide GEMM brings both side by side,
// but streams long weights no faster and decodes int8 codes once for every two waves that read them.  Which is the faster one: by what the two choices of slices take their
// launches to be, each with the sum of its slices.  Both are models of a kernel alone; a line for each of the three ways a sum goes ties them together, drawn through us a layer of
// 36 models of 1024 .. 8192 wide, feed-forwards of 3584 .. 28672, at 17, 20, 24, 28 and 32 rows, one projection after the other moved to the wide GEMM in the same model (1400 comparisons;
// profiles/few_rows_sweep.txt).  What the choice loses against the faster one of the two, us a layer of 40 .. 330, on the mean, fp8 and int8: slices that a launch adds 0.06 and 0.06 (never
// the wide GEMM 0.54 and 0.11, the rule before 0.33 and 0.11), unsplit 0.04 and 0.06 (0.75 and 0.42; 0.60 and 0.42), sums of 4096 deep and more that the next norm takes 0.23 (0.42; 0.44), int8 see below.  The rule before
// went by the share of a wave's requests that are k-tiles of its own, and tiles that are not a wave's own are no requests any more.
// Not bf16 weights, nor up to 16 rows (28672 x 4096 fp8 23.4 -> 23.8 us); nothing beyond the sizes measured.
bool gemm_wide_few_rows(const LinearW& w, int M, size_t ws_bytes, bool deferred) {
  int cus = 0;
  if (gemm_wide_mode() == 0 || gemm_wide_bm()) return false;      // (128 tokens and more: none of these calls has them)
  if (M < 17 || M > 32 || w.wd == MI_W_BF16 || w.K % 64 != 0 || w.K < 2048 || w.N < 2048 || w.N > 65536 || device_num_cu(&cus) != MI_OK) return false;
  const bool fp8 = w.wd == MI_W_F8E4M3;
  // sums, int8: the register kernel takes 0 .. 9 us less but for the narrowest (2048 .. 3072 square, 24 rows and more: 0.3 .. 1.2 more).  K of 16448 .. 17600 (five k-tiles a wave, the last of them
  // rare) was the wide GEMM's by the rule before, and its tests hold it to that: 1.5 .. 4 more (2048, 3072, 5120 rows).
  if (deferred && !fp8) return w.K > 16384 && w.K <= 17600 && (size_t)w.N * w.K <= 150000000;
  if (deferred && w.K < 4096) return false;                       // (2048 .. 3072 square: 0.3 .. 2 us in favour of the wide GEMM from 20 rows on; held by the same tests)
  const double regs = fp8 ? gemv_regs_us_wd<MI_W_F8E4M3>(M, w.N, w.K, ws_bytes, deferred) : gemv_regs_us_wd<MI_W_INT8>(M, w.N, w.K, ws_bytes, deferred);
  const WidePlan wide = gemm_wide_plan(M, w.N, w.K, gemm_wide_ks() == 1 ? 0 : ws_bytes, w.wd, deferred);
  if (deferred) return 1.6 * wide.us - 10.5 < regs;
  // (three times as wide as deep, 3584 .. 4032 deep, from 25 rows on: level, 0.3 more .. 0.4 less)
  if (wide.ks > 1) return 1.2 * wide.us - 7.5 < regs || (fp8 && M >= 25 && w.K >= 3584 && w.K < 4096 && w.N >= 3 * w.K);
  // fp8 tiles that fill three quarters of the chip to all of it in one round take less than the line says: 24576 .. 32768 rows, 3584 and 4096 deep, at 28 rows 0.1 .. 0.7 less than the registers, at 32 rows
  // 0.2 .. 1.5, at 24 rows 0.5 more to as much
  const int tiles = ceil_div(w.N, 128);
  if (fp8 && M >= 25 && w.K >= 3584 && 4 * tiles >= 3 * cus && tiles <= cus) return true;
  return w.K >= 4096 && 0.85 * wide.us + 4.5 < regs;
}
// The 128 x 128 kernel keeps single 16-row tiles and, where there is no workspace to split K into, grids of less than half the chip.  Everything else is the
// wide kernel's (us at 60 / 100 - 128 tokens, 128 x 128 -> wide: 4096 x 4096 fp8 18.4 / 19.5 -> 9.4 / 11.8, 2560 x 2048 bf16 12.6 / 17.4 -> 11.0 / 11.6).
static bool gemm_wide_wanted(const LinearW& w, int T, size_t ws_bytes) {
  if (w.K % 64 != 0 || (w.N / 16) < 2) return false;
  const int mode = gemm_wide_mode();
  if (mode == 1) return true;
  if (mode == 0) return false;
  return ws_bytes > 0 || ceil_div(T, 128) * ceil_div(w.N, 256) >= 128;
}
int launch_gemm_wide(const LinearW& w, int T, const uint16_t* x, int ldx, int epi, const EpiArgs& e, hipStream_t s,
                     float* splitk_ws, size_t splitk_ws_bytes, SlabSum* defer, bool split_as_deferred, int force_bm, int force_ntw, int force_ks) {
  if (defer) *defer = SlabSum();
  MI_CHECK(!e.next_x, "gemm_wide: hands no norm on");
  MI_CHECK(w.K % 64 == 0 && ldx % 8 == 0, "gemm_wide: K % 64 == 0");
  WidePlan pl = gemm_wide_plan(T, w.N, w.K, gemm_wide_ks() == 1 || !splitk_ws ? 0 : splitk_ws_bytes, w.wd, split_as_deferred || (defer && (epi == EPI_RESID || epi == EPI_F32)));
  const int forced_bm = force_bm ? force_bm : gemm_wide_bm();
  if (forced_bm) pl = WidePlan{forced_bm, force_ntw ? force_ntw : 4, 1, 0.};
  if (force_ks) {
    MI_CHECK(force_ks >= 1 && (force_ks - 1) * ceil_div(w.K / 64, force_ks) < w.K / 64 && (force_ks == 1 || (splitk_ws && (size_t)force_ks * T * w.N * 4 <= splitk_ws_bytes)),
             "gemm_wide: forced K-split must leave no slice empty and fit the workspace");
    pl.ks = force_ks;
  }
  if (w.wd == MI_W_BF16) return launch_gemm_wide_wd<MI_W_BF16>(w, T, x, ldx, epi, e, s, pl.bm, pl.ntw, pl.ks, splitk_ws, defer);
  if (w.wd == MI_W_F8E4M3) return launch_gemm_wide_wd<MI_W_F8E4M3>(w, T, x, ldx, epi, e, s, pl.bm, pl.ntw, pl.ks, splitk_ws, defer);
  return launch_gemm_wide_wd<MI_W_INT8>(w, T, x, ldx, epi, e, s, pl.bm, pl.ntw, pl.ks, splitk_ws, defer);
}

int launch_gemm(const LinearW& w, int T, const uint16_t* x, int ldx, int epi, const EpiArgs& e, hipStream_t s,
                float* splitk_ws, size_t splitk_ws_bytes, SlabSum* defer, bool split_as_deferred) {
  if (defer) *defer = SlabSum();
  MI_CHECK(!e.next_x, "gemm: hands no norm on");
  if (e.far_out) {      // (nothing here stores through L2)
    EpiArgs near = e;
    near.far_out = false;
    return launch_gemm(w, T, x, ldx, epi, near, s, splitk_ws, splitk_ws_bytes, defer, split_as_deferred);
  }
  MI_CHECK(e.rs_n == 0.f, "gemm: no rows with the parts of a norm");
  MI_CHECK(T >= 1, "gemm: T must be >= 1");
  if (gemm_wide_wanted(w, T, splitk_ws ? splitk_ws_bytes : 0) && ldx % 8 == 0)
    return launch_gemm_wide(w, T, x, ldx, epi, e, s, splitk_ws, splitk_ws_bytes, defer, split_as_deferred);
  MI_CHECK(w.N % 16 == 0 && w.K % 64 == 0, "gemm: N % 16 == 0 and K % 64 == 0 required");
  MI_CHECK(ldx % 8 == 0, "gemm: x row stride must be a multiple of 8 elements");
  switch (w.wd) {
    case MI_W_BF16: return launch_gemm_wd<MI_W_BF16>(w, T, x, ldx, epi, e, s, splitk_ws, splitk_ws_bytes, defer);
    case MI_W_F8E4M3: return launch_gemm_wd<MI_W_F8E4M3>(w, T, x, ldx, epi, e, s, splitk_ws, splitk_ws_bytes, defer);
    case MI_W_INT8: return launch_gemm_wd<MI_W_INT8>(w, T, x, ldx, epi, e, s, splitk_ws, splitk_ws_bytes, defer);
  }
  set_error("gemm: bad weight dtype");
  return MI_EINVAL;
}

// =====================================================================================
// GEMM with FP8 activations (context encoding, the MFMA-bound contraction)
// =====================================================================================
// y[m, n] = (sum_k q_x[m, k] * q_w[n, k]) * s_w[n] * s_x[m]   both operands OCP e4m3.
// v_mfma_scale_f32_16x16x128_f8f6f4 with every block scale = 2^0 runs at twice the rate of
// the bf16 (and of the unscaled fp8) MFMA.  Its lane (g = lane >> 4, r = lane & 15) holds 32
// bytes of row r: they are taken as the lane's 16 bytes of weight tile 2s and of tile 2s + 1
// (the contraction order inside an MFMA is free as long as both operands agree), so the
// weight image is the same one the GEMV streams.  Work-group = 4 waves, tile 256 (n) x 128 (m):
// wave w owns n-tiles 4w..4w+3 against all 8 m-tiles (128 fp32 accumulators per lane, one wave
// per SIMD); W fragments come straight from global (every wave reads distinct rows), x8 goes
// through LDS; the next K-step's operands are fetched into registers under the MFMAs.
typedef __attribute__((ext_vector_type(8))) int i32x8_t;
constexpr int kA8BM = 128, kA8BK = 128;   // tile: (64 NTW) weight rows x 128 tokens x 128 K bytes
constexpr int kA8Pitch = kA8BK + 32;   // LDS row pitch in bytes: 160 makes the fragment reads (row c, 16 B at g * 16 / + 64) conflict-free
                                       // over the ds_read_b128 lane groups; 144 left every group two-deep on its banks

// SPLIT: grid.z K-slices each write their raw fp32 accumulators to slab[z][m][n]; splitk_reduce
// sums the slabs in slice order (deterministic) and applies the epilogue.  Used when a short
// prompt leaves the (m-tile x n-tile) grid too small to pull the weights at HBM rate.
template <int EPI, bool SPLIT, int NTW>   // NTW 16-row weight tiles per wave: the tile is (64 NTW) x 128
__global__ __launch_bounds__(256) void gemm_a8_kernel(const uint4* __restrict__ W, int NT, int KT, int T, int K,
                                                      const uint8_t* __restrict__ x8, int ldx, EpiArgs e,
                                                      float* __restrict__ slab) {
  __shared__ __attribute__((aligned(16))) unsigned char xs[kA8BM * kA8Pitch];   // 20 KiB
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int g = lane >> 4, c = lane & 15;
  // XCD-aware tile order.  Work-groups go round-robin over the 8 XCDs (own 4 MiB L2 each), so
  // linear id L runs on XCD L % 8.  An XCD takes every eighth 256-row weight slab and walks ALL
  // token blocks of a slab back to back: the slab (and the K-step the co-resident work-groups
  // are at) is fetched over the fabric once per XCD instead of once per XCD per token block.
  constexpr int BN = 64 * NTW;
  const int mtiles = ceil_div(T, kA8BM), ntiles = ceil_div(NT, BN / 16);
  const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
  const int mblk = seq % mtiles, nblk = (seq / mtiles) * 8 + xcd;
  if (nblk >= ntiles) return;
  const int m0 = mblk * kA8BM, nt0 = nblk * (BN / 16) + wave * NTW;
  const int nks_all = K / kA8BK;
  const int ks_per = SPLIT ? ceil_div(nks_all, (int)gridDim.z) : nks_all;
  const int ks_beg = SPLIT ? (int)blockIdx.z * ks_per : 0;
  const int nks = min(ks_beg + ks_per, nks_all);   // exclusive end of this slice
  constexpr int kUnit = 0x7f7f7f7f;   // E8M0 block scales: 2^0

  f32x4_t acc[NTW][8];
#pragma unroll
  for (int i = 0; i < NTW; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // x staging: 128 rows x 128 B per K-step = 1024 chunks of 16 B, 4 per thread.  The fp8 image
  // is K-step-major, [K / 128][ldx = T rows][128 B]: a work-group's K-step is 16 KiB contiguous.
  u32x4_t xr[4], wr[NTW][2], wn[NTW][2];
  auto load_x = [&](int ks) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = tid + i * 256, row = idx >> 3, ch = idx & 7;
      const int m = min(m0 + row, T - 1);   // rows past T are computed on a copy of the last row, never stored
      xr[i] = *reinterpret_cast<const u32x4_t*>(x8 + ((size_t)ks * ldx + m) * kA8BK + ch * 16);
    }
  };
  auto load_w = [&](u32x4_t (&dst)[NTW][2], int ks) {
#pragma unroll
    for (int i = 0; i < NTW; ++i) {
      const int nt = min(nt0 + i, NT - 1);
#pragma unroll
      for (int t = 0; t < 2; ++t)
        dst[i][t] = *reinterpret_cast<const u32x4_t*>(W + ((size_t)nt * KT + ks * 2 + t) * 64 + lane);
    }
  };
  MI_TRACE_BEGIN();
  MI_STAMP(0);
  if (ks_beg < nks) {
    load_x(ks_beg);
    load_w(wr, ks_beg);
  }
  for (int ks = ks_beg; ks < nks; ++ks) {
    if (ks == ks_beg + 4) MI_STAMP(1);     // tools/trace_gemm.py: phases of the fifth K-step
    if (ks == ks_beg + 5) MI_STAMP(6);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = tid + i * 256, row = idx >> 3, ch = idx & 7;
      *reinterpret_cast<u32x4_t*>(&xs[row * kA8Pitch + ch * 16]) = xr[i];
    }
    __syncthreads();
    if (ks == ks_beg + 4) MI_STAMP(2);
    if (ks + 1 < nks) {
      load_x(ks + 1);
      load_w(wn, ks + 1);
    }
    if (ks == ks_beg + 4) MI_STAMP(3);
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) {
      const unsigned char* xrow = &xs[(mt * 16 + c) * kA8Pitch + g * 16];
      const u32x4_t b0 = *reinterpret_cast<const u32x4_t*>(xrow);        // k-tile 2ks,   chunk g
      const u32x4_t b1 = *reinterpret_cast<const u32x4_t*>(xrow + 64);   // k-tile 2ks+1, chunk g
      const i32x8_t b = {(int)b0[0], (int)b0[1], (int)b0[2], (int)b0[3], (int)b1[0], (int)b1[1], (int)b1[2], (int)b1[3]};
#pragma unroll
      for (int i = 0; i < NTW; ++i) {
        const i32x8_t a = {(int)wr[i][0][0], (int)wr[i][0][1], (int)wr[i][0][2], (int)wr[i][0][3],
                           (int)wr[i][1][0], (int)wr[i][1][1], (int)wr[i][1][2], (int)wr[i][1][3]};
        acc[i][mt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, acc[i][mt], 0, 0, 0, kUnit, 0, kUnit);
      }
    }
    if (ks == ks_beg + 4) MI_STAMP(4);
    __syncthreads();
    if (ks == ks_beg + 4) MI_STAMP(5);
    if (ks + 1 < nks) {
#pragma unroll
      for (int i = 0; i < NTW; ++i) {
        wr[i][0] = wn[i][0];
        wr[i][1] = wn[i][1];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NTW; ++i) {
    if (nt0 + i >= NT) continue;
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) {
      const int m = m0 + mt * 16 + c;
      if (m >= T) continue;
      const int n0 = (nt0 + i) * 16 + g * 4;
      if constexpr (SPLIT) {
        *reinterpret_cast<float4*>(slab + ((size_t)blockIdx.z * T + m) * (NT * 16) + n0) =
            make_float4(acc[i][mt][0], acc[i][mt][1], acc[i][mt][2], acc[i][mt][3]);
      } else {
        epilogue<EPI>(e, m, n0, acc[i][mt]);
      }
    }
  }
  MI_STAMP(7);
  MI_TRACE_END();
}

// ---- FP8 activations on the wide tile ------------------------------------------------------------
// The kernel above keeps three work-groups of 128 x 128 on a CU and takes in 32 KiB per 4.2 MFLOP; this one is
// gemm_wide_kernel's schedule (LDS-DMA ring of three stages, the two wave groups half a K-step apart) on 128 tokens x 256
// weight rows x 128 K bytes: 16 + 32 KiB per 8.4 MFLOP, half the bytes per flop.  (256 x 256 would halve them again but is
// 64 KiB a stage: two stages in 160 KiB, and two stages cannot carry the stagger -- profiles/r03_a8_wide_experiment.txt.)
// A stage: [16 n-tiles][2 k-tiles][64 lanes x 16 B] weight fragments as stored, then 128 activation rows x 128 B with
// 16-byte chunk ch of row r at slot ch ^ (r & 7) (the lane reads chunks g and 4 + g: conflict-free with that key).
constexpr int kA8wStage = 32 * 1024 + 128 * 128, kA8wDma = 6, kA8WideStages = 3;
// (A ninth wave touching the lines of the K-step four ahead, to make the ring's DMAs L2 hits, cost 27 %: 260 -> 330 us on
// gate|up at 2048 tokens -- profiles/r03_a8_wide_experiment.txt.)
template <int EPI, bool SPLIT>
__global__ __launch_bounds__(512) void gemm_a8_wide_kernel(const uint4* __restrict__ W, int NT, int KT, int T, int K,
                                                           const uint8_t* __restrict__ x8, int ldx, EpiArgs e,
                                                           float* __restrict__ slab) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int g = lane >> 4, c = lane & 15;
  const int wm = wave & 1, wn = wave >> 1;      // waves 2 (tokens) x 4 (weight rows), each 64 x 64
  const int mtiles = ceil_div(T, 128), ntiles = ceil_div(NT, 16);
  const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
  const int mblk = seq % mtiles, nblk = (seq / mtiles) * 8 + xcd;
  if (nblk >= ntiles) return;
  const int m0 = mblk * 128, ntb = nblk * 16;
  const int nks = SPLIT ? K / 128 / (int)gridDim.z : K / 128;
  const int ks0 = SPLIT ? (int)blockIdx.z * nks : 0;
  constexpr int kUnit = 0x7f7f7f7f;   // E8M0 block scales: 2^0

  // DMA sources of this lane: weight n-tiles 2w, 2w + 1 (two k-tiles each, adjacent in the image), activation pieces 2w, 2w + 1
  const uint4* wsrc[2];
  const uint8_t* xsrc[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) wsrc[i] = W + ((size_t)min(ntb + 2 * wave + i, NT - 1) * KT + 2 * ks0) * 64 + lane;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = (2 * wave + i) * 8 + (lane >> 3), sl = lane & 7;
    xsrc[i] = x8 + ((size_t)ks0 * ldx + min(m0 + r, T - 1)) * 128 + ((sl ^ (r & 7)) * 16);
  }
  auto issue = [&](int ks) {
    unsigned char* st = smem + (ks % kA8WideStages) * kA8wStage;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int t = 0; t < 2; ++t) glds16(wsrc[i] + ((size_t)ks * 2 + t) * 64, st + ((2 * wave + i) * 2 + t) * 1024);
#pragma unroll
    for (int i = 0; i < 2; ++i) glds16(xsrc[i] + (size_t)ks * ldx * 128, st + 32 * 1024 + (2 * wave + i) * 1024);
  };

  f32x4_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // the schedule of gemm_wide_kernel: READ (fragments to registers) / MULTIPLY (MFMAs only), the groups in opposite phases
  const int grp = __builtin_amdgcn_readfirstlane(wave >> 2);
  issue(0);
  if (nks > 1) issue(1);
  if (grp == 1) {
    if (nks > 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kA8wDma) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
  }
  for (int ks = 0; ks < nks; ++ks) {
    if (grp == 0) {
      if (ks + 1 < nks) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kA8wDma) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __builtin_amdgcn_s_barrier();
    if (ks + 2 < nks) issue(ks + 2);
    const unsigned char* st = smem + (ks % kA8WideStages) * kA8wStage;
    const uint4* xs = reinterpret_cast<const uint4*>(st + 32 * 1024);
    u32x4_t b0[4], b1[4], a0[4], a1[4];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const int r = wm * 64 + mt * 16 + c;
      b0[mt] = *reinterpret_cast<const u32x4_t*>(&xs[r * 8 + (g ^ (r & 7))]);
      b1[mt] = *reinterpret_cast<const u32x4_t*>(&xs[r * 8 + ((4 + g) ^ (r & 7))]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a0[i] = *reinterpret_cast<const u32x4_t*>(st + ((wn * 4 + i) * 2) * 1024 + lane * 16);
      a1[i] = *reinterpret_cast<const u32x4_t*>(st + ((wn * 4 + i) * 2 + 1) * 1024 + lane * 16);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      asm volatile("" : "+v"(b0[j])); asm volatile("" : "+v"(b1[j]));
      asm volatile("" : "+v"(a0[j])); asm volatile("" : "+v"(a1[j]));
    }
    if (grp == 1 && ks + 1 < nks) {
      if (ks + 2 < nks) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kA8wDma) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const i32x8_t b = {(int)b0[mt][0], (int)b0[mt][1], (int)b0[mt][2], (int)b0[mt][3], (int)b1[mt][0], (int)b1[mt][1], (int)b1[mt][2], (int)b1[mt][3]};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const i32x8_t a = {(int)a0[i][0], (int)a0[i][1], (int)a0[i][2], (int)a0[i][3], (int)a1[i][0], (int)a1[i][1], (int)a1[i][2], (int)a1[i][3]};
        acc[i][mt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, acc[i][mt], 0, 0, 0, kUnit, 0, kUnit);
      }
    }
  }
  if (grp == 0) __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int nt = ntb + wn * 4 + i;
    if (nt >= NT) continue;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const int m = m0 + wm * 64 + mt * 16 + c;
      if (m >= T) continue;
      if constexpr (SPLIT) {
        *reinterpret_cast<float4*>(slab + ((size_t)blockIdx.z * T + m) * (NT * 16) + nt * 16 + g * 4) =
            make_float4(acc[i][mt][0], acc[i][mt][1], acc[i][mt][2], acc[i][mt][3]);
      } else {
        epilogue<EPI>(e, m, nt * 16 + g * 4, acc[i][mt]);
      }
    }
  }
}

// PARTS: the row's factor comes as the parts of a norm (EpiArgs::rs_n; calls of up to 32 rows).  Prompts never have them, and four requests, a division and a root for each thread are not for
// nothing: residual sum of 2031 tokens 27.9 us with one kernel for both, 22.2 with two, of 188 6.7 and 6.0.
template <int EPI, bool PARTS>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ slab, int KS, int T, int N, EpiArgs e) {
  const int q = blockIdx.x * 256 + threadIdx.x;      // one (m, 4 consecutive n) per thread
  const int nq = N >> 2;
  if (q >= T * nq) return;
  const int m = q / nq, n0 = (q - m * nq) * 4;
  // what the epilogue needs is requested in front of the slabs, and what hangs off it (the rotary factors) behind their requests
  EpiPre<EPI> pre;
  epi_prefetch<EPI>(e, m, n0, pre);
  const float4 sc = *reinterpret_cast<const float4*>(e.scale + n0), bi = e.bias ? *reinterpret_cast<const float4*>(e.bias + n0) : make_float4(0.f, 0.f, 0.f, 0.f);
  float4 ss = make_float4(0.f, 0.f, 0.f, 0.f);
  float rs = 1.f;
  if constexpr (PARTS) ss = row_parts(e.row_scale, m);
  else rs = e.row_scale ? e.row_scale[m] : 1.f;
  const float4 v = slab_sum4(slab + (size_t)m * N + n0, (size_t)T * N, KS, [&] { epi_prefetch_dependent<EPI>(e, n0, pre); });
  if constexpr (PARTS) rs = row_rinv(ss, e.rs_n, e.rs_eps);
  const float sc4[4] = {sc.x, sc.y, sc.z, sc.w}, b4[4] = {bi.x, bi.y, bi.z, bi.w};
  epilogue_pre<EPI>(e, m, n0, sc4, e.bias ? b4 : nullptr, f32x4_t{v.x, v.y, v.z, v.w}, pre, rs);
}

// (Sums for the host stay in L2: a wave stores 1 KiB of a row with one request, which gains nothing by being stored through and waits.  24 rows of 32000 words, bf16 5120 deep:
//  56.8 us, 60.0 through)
int launch_splitk_reduce(const SlabSum& sl, int epi, const EpiArgs& args, hipStream_t s) {
  MI_CHECK(!args.next_x, "splitk_reduce: hands no norm on");      // (its lanes hold other columns than put_resid adds up)
  EpiArgs e = args;
  e.far_out = false;
  const dim3 grid(ceil_div(sl.T * (sl.N / 4), 256));
#define MI_S(EPI_) case EPI_: \
    if (e.rs_n > 0.f) hipLaunchKernelGGL((splitk_reduce_kernel<EPI_, true>), grid, dim3(256), 0, s, sl.slab, sl.KS, sl.T, sl.N, e); \
    else hipLaunchKernelGGL((splitk_reduce_kernel<EPI_, false>), grid, dim3(256), 0, s, sl.slab, sl.KS, sl.T, sl.N, e); \
    break
  switch (epi) {
    MI_S(EPI_F32); MI_S(EPI_QKV); MI_S(EPI_SWIGLU); MI_S(EPI_RESID); MI_S(EPI_RELU2); MI_S(EPI_GLU_CLIP); MI_S(EPI_SOFTCAP); MI_S(EPI_HEADS_KV);
    default: set_error("splitk_reduce: unknown epilogue"); return MI_EINVAL;
  }
#undef MI_S
  MI_HIP(hipGetLastError());
  return MI_OK;
}

// sum a deferred K-split (SlabSum) the plain way: splitk_reduce + residual epilogue
int launch_splitk_flush(const SlabSum& sl, const float* resid_in, float* out, int ld_out, hipStream_t s) {
  EpiArgs e{};
  e.scale = sl.scale; e.bias = sl.bias; e.row_scale = sl.row_scale; e.rs_n = sl.rs_n; e.rs_eps = sl.rs_eps;
  e.out_f32 = out; e.resid_in = resid_in; e.ld_out = ld_out;
  return launch_splitk_reduce(sl, EPI_RESID, e, s);
}

bool gemm_a8_supported(const LinearW& w) {
  return w.wd == MI_W_F8E4M3 && w.K % kA8BK == 0 && w.N % 16 == 0;
}

int launch_gemm_a8(const LinearW& w, int T, const uint8_t* x8, int ldx, int epi, const EpiArgs& e, hipStream_t s,
                   float* splitk_ws, size_t splitk_ws_bytes, SlabSum* defer) {
  if (defer) *defer = SlabSum();
  MI_CHECK(!e.next_x, "gemm_a8: hands no norm on");
  MI_CHECK(e.rs_n == 0.f, "gemm_a8: no rows with the parts of a norm");
  MI_CHECK(T >= 1, "gemm_a8: T must be >= 1");
  MI_CHECK(gemm_a8_supported(w), "gemm_a8: needs fp8 weights, K % 128 == 0, N % 16 == 0");
  MI_CHECK(ldx >= T && e.row_scale != nullptr, "gemm_a8: x8 is the K-step-major image of >= T rows, with its row scales");
  const int NT = w.N / 16, KT = w.K / 64, nks = w.K / kA8BK;
  {   // The wide tile (MI355X_A8_WIDE: 0 never, 1 always, unset: by plan) where its one-work-group-per-CU grid fills one or two
      // rounds of the chip.  Measured on the Llama-8B shapes against the kernel below (us): 256 tokens gate|up 43.6 vs 45.9,
      // down 24.0 vs 25.6, QKV 17.3 vs 19.4; 512: 76.9 vs 86.0, 34.8 vs 39.6, 23.5 vs 28.0; 1024: down 58.4 vs 68.2, QKV 48.8 vs
      // 51.9 but gate|up (3.5 rounds) 145.0 vs 135.9; 2048: down 121.0 vs 136.1, O 46.2 vs 49.3, gate|up (7 rounds) 260.4 vs
      // 254.2 -- on long grids the three resident work-groups of the 128 x 128 kernel hide more latency than the ring does.
    static const int mode = [] { const char* v = getenv("MI355X_A8_WIDE"); return v ? atoi(v) : -1; }();
    int cus = 256;
    if (device_num_cu(&cus) != MI_OK || cus < 1) cus = 256;
    int best_ks = 0;
    double best_cost = 0.;
    for (int ks = 1; ks <= 8; ks *= 2) {
      if (nks % ks != 0 || nks / ks < 4) continue;
      if (ks > 1 && (!splitk_ws || (size_t)ks * T * w.N * sizeof(float) > splitk_ws_bytes)) continue;
      const int wgs = ceil_div(T, 128) * ceil_div(w.N, 256) * ks, rounds = ceil_div(wgs, cus);
      const bool ok = mode == 1 || (rounds <= 2 && (wgs < cus ? wgs * 10 >= cus * 7 : wgs * 5 >= rounds * cus * 4));
      if (!ok) continue;
      double cost = (double)rounds * (nks / ks) * 1.0;
      if (ks > 1) cost += 4.0 + (double)(ks + 1) * T * w.N * 4.0 / 4.0e6;
      if (best_ks == 0 || cost < best_cost) { best_ks = ks; best_cost = cost; }
    }
    if (mode != 0 && best_ks && T > 128) {
      const int KS = best_ks;
      dim3 grid(8 * ceil_div(T, 128) * ceil_div(ceil_div(w.N, 256), 8), 1, KS);
      const uint4* W = reinterpret_cast<const uint4*>(w.w);
      constexpr int lds = kA8WideStages * kA8wStage;
#define MI_A8W_L(EPI_, SPLIT_, WS_) \
  do { \
    MI_TRY_(ensure_dynamic_lds(reinterpret_cast<const void*>(gemm_a8_wide_kernel<EPI_, SPLIT_>), lds)); \
    hipLaunchKernelGGL((gemm_a8_wide_kernel<EPI_, SPLIT_>), grid, dim3(512), lds, s, W, NT, KT, T, w.K, x8, ldx, e, WS_); \
  } while (0)
#define MI_A8W(EPI_) \
  do { \
    if (KS == 1) { \
      MI_A8W_L(EPI_, false, nullptr); \
    } else { \
      MI_A8W_L(EPI_, true, splitk_ws); \
      if (defer && EPI_ == EPI_RESID) { *defer = SlabSum{splitk_ws, KS, T, w.N, e.scale, e.bias, e.row_scale}; } \
      else hipLaunchKernelGGL((splitk_reduce_kernel<EPI_, false>), dim3(ceil_div(T * (w.N / 4), 256)), dim3(256), 0, s, splitk_ws, KS, T, w.N, e); \
    } \
  } while (0)
      if (epi == EPI_QKV) MI_A8W(EPI_QKV);
      else if (epi == EPI_SWIGLU) MI_A8W(EPI_SWIGLU);
      else if (epi == EPI_RESID) MI_A8W(EPI_RESID);
      else MI_A8W(EPI_F32);
#undef MI_A8W
#undef MI_A8W_L
      MI_HIP(hipGetLastError());
      return MI_OK;
    }
  }
  // 128 x 128 tiles: 64 accumulator registers per lane leave room for three work-groups per CU,
  // which hide each other's load latency (the 256 x 128 tile ran one work-group per CU at 24 % of
  // the matrix-core rate: 29.7 ms for the 2048 bucket against 22.5 ms; forcing a fourth wave per
  // SIMD spills inside the K loop: 122 ms)
  constexpr int ntw = 2;
  const int bn = 64 * ntw;
  const int mtiles = ceil_div(T, kA8BM), ntiles = ceil_div(w.N, bn);
  // K-split only when the tile grid cannot occupy the chip and the slabs stay small
  // (768 work-groups are resident at once.  Measured on the Llama-8B shapes: below 256 tiles aim
  // for 512 work-groups, below 384 for 768; splitting larger grids costs more in slab traffic
  // than it wins -- 6.2 / 8.8 / 13.5 ms for the 256 / 512 / 1024 buckets.)
  const int KS = gemm_pick_splitk(mtiles * ntiles, nks, T, w.N, splitk_ws ? splitk_ws_bytes : 0);
  const uint4* W = reinterpret_cast<const uint4*>(w.w);
  dim3 grid(8 * mtiles * ceil_div(ntiles, 8), 1, KS);   // see the kernel: XCD-aware tile order
#define MI_A8(EPI_) \
  do { \
    if (KS == 1) { \
      hipLaunchKernelGGL((gemm_a8_kernel<EPI_, false, ntw>), grid, dim3(256), 0, s, W, NT, KT, T, w.K, x8, ldx, e, nullptr); \
    } else { \
      hipLaunchKernelGGL((gemm_a8_kernel<EPI_, true, ntw>), grid, dim3(256), 0, s, W, NT, KT, T, w.K, x8, ldx, e, splitk_ws); \
      if (defer && EPI_ == EPI_RESID) { *defer = SlabSum{splitk_ws, KS, T, w.N, e.scale, e.bias, e.row_scale}; } \
      else hipLaunchKernelGGL((splitk_reduce_kernel<EPI_, false>), dim3(ceil_div(T * (w.N / 4), 256)), dim3(256), 0, s, splitk_ws, KS, T, w.N, e); \
    } \
  } while (0)
  if (epi == EPI_QKV) MI_A8(EPI_QKV);
  else if (epi == EPI_SWIGLU) MI_A8(EPI_SWIGLU);
  else if (epi == EPI_RESID) MI_A8(EPI_RESID);
  else MI_A8(EPI_F32);
#undef MI_A8
  MI_HIP(hipGetLastError());
  return MI_OK;
}

// =====================================================================================
// Load-time quantize + tile
// =====================================================================================
__global__ void rowmax_kernel(const float* __restrict__ w, int ld, float* __restrict__ rowmax) {
  const float* r = w + (size_t)blockIdx.x * ld;
  float m = 0.f;
  for (int i = threadIdx.x; i < ld; i += blockDim.x) m = fmaxf(m, fabsf(r[i]));
  __shared__ float sm[256];
  sm[threadIdx.x] = m;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) sm[threadIdx.x] = fmaxf(sm[threadIdx.x], sm[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) rowmax[blockIdx.x] = sm[0];
}
__global__ void allmax_kernel(const float* __restrict__ rowmax, int n, float* __restrict__ out) {
  float m = 0.f;
  for (int i = threadIdx.x; i < n; i += blockDim.x) m = fmaxf(m, rowmax[i]);
  __shared__ float sm[256];
  sm[threadIdx.x] = m;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) sm[threadIdx.x] = fmaxf(sm[threadIdx.x], sm[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = sm[0];
}

// bf16 activations -> e4m3 + per-token scale: s = amax / 448 (all-zero row: 1), q = rne(x / s).
// One work-group per row.
// The row stays in registers between the amax pass and the quantize pass (up to kRqMax 16-byte
// chunks per thread, K <= 16384); longer rows are re-read.
constexpr int kRqMax = 8;
__global__ __launch_bounds__(256) void rowquant_fp8_kernel(const uint16_t* __restrict__ x, int K, int ldx,
                                                           uint8_t* __restrict__ x8, float* __restrict__ row_scale) {
  __shared__ float red[4];
  const int t = blockIdx.x, tid = threadIdx.x;
  const uint16_t* row = x + (size_t)t * ldx;
  const int nchunk = K / 8;
  u32x4_t v[kRqMax];
  float amax = 0.f;
#pragma unroll
  for (int q = 0; q < kRqMax; ++q) {
    const int c8 = tid + q * 256;
    v[q] = c8 < nchunk ? *reinterpret_cast<const u32x4_t*>(row + c8 * 8) : u32x4_t{0, 0, 0, 0};
  }
#pragma unroll
  for (int q = 0; q < kRqMax; ++q)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t w = v[q][k];
      amax = fmaxf(amax, fmaxf(fabsf(bf16lo_to_f32(w)), fabsf(bf16hi_to_f32(w))));
    }
  for (int c8 = tid + kRqMax * 256; c8 < nchunk; c8 += 256) {
    const u32x4_t r = *reinterpret_cast<const u32x4_t*>(row + c8 * 8);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t w = r[k];
      amax = fmaxf(amax, fmaxf(fabsf(bf16lo_to_f32(w)), fabsf(bf16hi_to_f32(w))));
    }
  }
  amax = fmaxf(amax, __shfl_xor(amax, 1));
  amax = fmaxf(amax, __shfl_xor(amax, 2));
  amax = fmaxf(amax, __shfl_xor(amax, 4));
  amax = fmaxf(amax, __shfl_xor(amax, 8));
  amax = fmaxf(amax, __shfl_xor(amax, 16));
  amax = fmaxf(amax, __shfl_xor(amax, 32));
  if ((tid & 63) == 0) red[tid >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float scale = amax > 0.f ? amax / 448.f : 1.f;
  if (tid == 0) row_scale[t] = scale;
  auto emit = [&](const u32x4_t r, int c8) {
    uint32_t o[2] = {0, 0};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t w = r[k];
      const float a = fminf(fmaxf(bf16lo_to_f32(w) / scale, -448.f), 448.f);
      const float b = fminf(fmaxf(bf16hi_to_f32(w) / scale, -448.f), 448.f);
      o[k >> 1] |= (f32_to_e4m3fn(a) | (f32_to_e4m3fn(b) << 8)) << (16 * (k & 1));
    }
    // K-step-major image: [K / 128][T][128 B] (see gemm_a8_kernel: load_x)
    const int k0 = c8 * 8;
    *reinterpret_cast<uint2*>(x8 + ((size_t)(k0 >> 7) * gridDim.x + t) * 128 + (k0 & 127)) = make_uint2(o[0], o[1]);
  };
#pragma unroll
  for (int q = 0; q < kRqMax; ++q) {
    const int c8 = tid + q * 256;
    if (c8 < nchunk) emit(v[q], c8);
  }
  for (int c8 = tid + kRqMax * 256; c8 < nchunk; c8 += 256) emit(*reinterpret_cast<const u32x4_t*>(row + c8 * 8), c8);
}

int launch_rowquant_fp8(const uint16_t* x, int T, int K, int ldx, uint8_t* x8, float* row_scale, hipStream_t s) {
  MI_CHECK(K % 8 == 0 && ldx % 8 == 0, "rowquant: K and the row stride must be multiples of 8");
  hipLaunchKernelGGL(rowquant_fp8_kernel, dim3(T), dim3(256), 0, s, x, K, ldx, x8, row_scale);
  MI_HIP(hipGetLastError());
  return MI_OK;
}

__device__ __forceinline__ int dst_to_src_row(const QuantJob& j, int r) {
  const int rel = r - j.dst_row0;
  if (rel < 0) return -1;
  int i;
  if (j.rowmap == ROWMAP_PLAIN) {
    i = rel;
  } else if (j.rowmap == ROWMAP_ROPE_PAIRS) {
    const int head = rel / j.hd, jj = rel % j.hd;
    i = head * j.hd + ((jj & 1) ? (jj >> 1) + (j.hd >> 1) : (jj >> 1));
  } else {
    if (rel & 1) return -1;
    i = rel >> 1;
  }
  return i < j.n_rows ? i : -1;
}

// one wave per destination tile
template <int WD>
__global__ __launch_bounds__(256) void quant_tile_kernel(QuantJob j, int nt_lo, int nt_cnt, int KT) {
  const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, lane = threadIdx.x & 63;
  if (wave >= nt_cnt * KT) return;
  const int nt = nt_lo + wave / KT, kt = wave % KT;
  const int r = nt * 16 + (lane & 15), gq = lane >> 4;
  const int i = dst_to_src_row(j, r);
  if (i < 0) return;
  constexpr int EPL = (WD == MI_W_BF16) ? 8 : 16;  // elements per lane
  const int col0 = kt * (EPL * 4) + gq * EPL;      // first of the lane's columns, relative to src_col0
  const bool pad_row = i >= j.n_rows - j.pad_rows;
  const int k_src = j.K - j.pad_cols;
  if (pad_row || col0 >= k_src) {                  // EPL divides every head size: a lane is all padding or none
    if (pad_row && kt == 0 && gq == 0) j.dst_scale[r] = 1.f;
    if (!pad_row && kt == 0 && gq == 0) {
      float sc = 1.f;
      if constexpr (WD != MI_W_BF16) {
        const float qm = (WD == MI_W_INT8) ? 127.f : 448.f;
        const float am = (j.quant_type == MI_Q_PER_TENSOR_SYMMETRIC) ? j.tmp_rowmax[j.src_rows_total] : j.tmp_rowmax[j.src_row0 + i];
        sc = am > 0.f ? am / qm : 1.f;
      }
      j.dst_scale[r] = sc;
    }
    reinterpret_cast<uint4*>(j.dst)[((size_t)nt * KT + kt) * 64 + lane] = make_uint4(0, 0, 0, 0);
    return;
  }
  const int srow = j.src_row0 + i;
  const float* src = j.src + (size_t)srow * j.ld + j.src_col0 + col0;
  float scale = 1.f;
  if constexpr (WD != MI_W_BF16) {
    const float qmax = (WD == MI_W_INT8) ? 127.f : 448.f;
    const float amax = (j.quant_type == MI_Q_PER_TENSOR_SYMMETRIC) ? j.tmp_rowmax[j.src_rows_total] : j.tmp_rowmax[srow];
    scale = amax > 0.f ? amax / qmax : 1.f;
  }
  if (kt == 0 && gq == 0) j.dst_scale[r] = scale;
  uint4 out;
  if constexpr (WD == MI_W_BF16) {
    uint32_t o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) o[k] = pack_bf16x2(src[2 * k], src[2 * k + 1]);
    out = make_uint4(o[0], o[1], o[2], o[3]);
  } else {
    const float qmax = (WD == MI_W_INT8) ? 127.f : 448.f;
    uint32_t o[4] = {0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      float t = src[k] / scale;
      t = fminf(fmaxf(t, -qmax), qmax);
      uint32_t b;
      if constexpr (WD == MI_W_INT8) b = (uint32_t)(int)rintf(t) & 0xffu;
      else b = f32_to_e4m3fn(t);
      o[k >> 2] |= b << (8 * (k & 3));
    }
    out = make_uint4(o[0], o[1], o[2], o[3]);
  }
  reinterpret_cast<uint4*>(j.dst)[((size_t)nt * KT + kt) * 64 + lane] = out;
}

int run_quant_job(const QuantJob& j, hipStream_t s) {
  MI_CHECK(j.K % 64 == 0, "quantize: K % 64 == 0 required");
  if (j.wd != MI_W_BF16) {
    hipLaunchKernelGGL(rowmax_kernel, dim3(j.src_rows_total), dim3(256), 0, s, j.src, j.ld, j.tmp_rowmax);
    hipLaunchKernelGGL(allmax_kernel, dim3(1), dim3(256), 0, s, j.tmp_rowmax, j.src_rows_total, j.tmp_rowmax + j.src_rows_total);
  }
  // destination rows touched: [dst_row0, dst_row0 + span)
  const int span = (j.rowmap == ROWMAP_EVERY_OTHER) ? 2 * j.n_rows : j.n_rows;
  const int nt_lo = j.dst_row0 / 16, nt_hi = ceil_div(j.dst_row0 + span, 16);
  const int KT = j.K / tile_k(j.wd);
  const int waves = (nt_hi - nt_lo) * KT;
  const dim3 grid(ceil_div(waves, 4)), block(256);
  if (j.wd == MI_W_BF16) hipLaunchKernelGGL((quant_tile_kernel<MI_W_BF16>), grid, block, 0, s, j, nt_lo, nt_hi - nt_lo, KT);
  else if (j.wd == MI_W_F8E4M3) hipLaunchKernelGGL((quant_tile_kernel<MI_W_F8E4M3>), grid, block, 0, s, j, nt_lo, nt_hi - nt_lo, KT);
  else hipLaunchKernelGGL((quant_tile_kernel<MI_W_INT8>), grid, block, 0, s, j, nt_lo, nt_hi - nt_lo, KT);
  MI_HIP(hipGetLastError());
  return MI_OK;
}

// tiled -> row-major (inspection / tests)
__global__ void untile_kernel(const uint4* __restrict__ tiled, int NT, int KT, int K, int eb, unsigned char* __restrict__ out) {
  const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, lane = threadIdx.x & 63;
  if (wave >= NT * KT) return;
  const int nt = wave / KT, kt = wave % KT;
  const uint4 v = tiled[(size_t)wave * 64 + lane];
  const int r = nt * 16 + (lane & 15);
  // 16 bytes = 16 elements (1-byte types) or 8 elements (bf16)
  const size_t byte_col = (size_t)kt * 64 + (lane >> 4) * 16;
  *reinterpret_cast<uint4*>(out + (size_t)r * K * eb + byte_col) = v;
}

int launch_untile(const void* tiled, int N, int K, int wd, void* out, hipStream_t s) {
  MI_CHECK(N % 16 == 0 && K % 64 == 0, "untile: N % 16 == 0 and K % 64 == 0 required");
  const int NT = N / 16, KT = K / tile_k(wd);
  hipLaunchKernelGGL(untile_kernel, dim3(ceil_div(NT * KT, 4)), dim3(256), 0, s,
                     reinterpret_cast<const uint4*>(tiled), NT, KT, K, elem_bytes(wd), reinterpret_cast<unsigned char*>(out));
  MI_HIP(hipGetLastError());
  return MI_OK;
}

__global__ void bf16_to_f32_kernel(const uint16_t* __restrict__ in, float* __restrict__ out, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    out[i] = bf16_to_f32(in[i]);
}
int launch_bf16_to_f32(const uint16_t* in, float* out, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(bf16_to_f32_kernel, dim3(2048), dim3(256), 0, s, in, out, n);
  MI_HIP(hipGetLastError());
  return MI_OK;
}

}  // namespace mi
