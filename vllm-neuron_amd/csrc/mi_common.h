// Shared device/host helpers for libmi355x_vllm (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>

#include "../../include/mi355x_vllm.h"

namespace mi {

typedef __attribute__((ext_vector_type(8))) short bf16x8_t;   // 8 bf16 = one MFMA 16x16x32 operand
typedef __attribute__((ext_vector_type(4))) float f32x4_t;    // MFMA 16x16 accumulator
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
typedef __attribute__((ext_vector_type(2))) float f32x2_t;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;

constexpr int kWave = 64;

// ---- error plumbing -------------------------------------------------------------------
void set_error(const std::string& msg);
#define MI_HIP(expr)                                                                  \
  do {                                                                                \
    hipError_t _e = (expr);                                                           \
    if (_e != hipSuccess) {                                                           \
      mi::set_error(std::string(#expr) + ": " + hipGetErrorString(_e));               \
      return MI_EHIP;                                                                 \
    }                                                                                 \
  } while (0)
#define MI_CHECK(cond, msg)                                                           \
  do {                                                                                \
    if (!(cond)) {                                                                    \
      mi::set_error(std::string(msg) + " [" #cond "]");                               \
      return MI_EINVAL;                                                               \
    }                                                                                 \
  } while (0)

// ---- scalar conversions ---------------------------------------------------------------
__device__ __forceinline__ float bf16_to_f32(uint16_t h) {
  return __builtin_bit_cast(float, (uint32_t)h << 16);
}
__device__ __forceinline__ float bf16lo_to_f32(uint32_t packed) {
  return __builtin_bit_cast(float, packed << 16);
}
__device__ __forceinline__ float bf16hi_to_f32(uint32_t packed) {
  return __builtin_bit_cast(float, packed & 0xffff0000u);
}
// round-to-nearest-even; plain cast lowers to v_cvt_pk_bf16_f32 on gfx950 and keeps NaN a NaN
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  return __builtin_bit_cast(uint16_t, (__bf16)f);
}
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  bf16x2_t v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}

// ---- weight-fragment decode: 8 stored weights -> 8 bf16 (one MFMA operand) --------------
// fp8 e4m3fn and int8 values are exactly representable in bf16.
template <int WD>
__device__ __forceinline__ bf16x8_t decode8(uint32_t lo, uint32_t hi);

template <>
__device__ __forceinline__ bf16x8_t decode8<MI_W_F8E4M3>(uint32_t lo, uint32_t hi) {
  union { bf16x2_t p[4]; bf16x8_t v; } u;
  u.p[0] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, false);
  u.p[1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, true);
  u.p[2] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, false);
  u.p[3] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, true);
  return u.v;
}

__device__ __forceinline__ uint32_t i8x2_to_bf16x2(uint32_t w, int byte0, int byte1) {
  float a = (float)(int)(int8_t)(w >> (8 * byte0));
  float b = (float)(int)(int8_t)(w >> (8 * byte1));
  return pack_bf16x2(a, b);
}
template <>
__device__ __forceinline__ bf16x8_t decode8<MI_W_INT8>(uint32_t lo, uint32_t hi) {
  union { uint32_t p[4]; bf16x8_t v; } u;
  u.p[0] = i8x2_to_bf16x2(lo, 0, 1);
  u.p[1] = i8x2_to_bf16x2(lo, 2, 3);
  u.p[2] = i8x2_to_bf16x2(hi, 0, 1);
  u.p[3] = i8x2_to_bf16x2(hi, 2, 3);
  return u.v;
}

// two neighbouring codes of a word: its low half or its high half
template <int WD>
__device__ __forceinline__ uint32_t decode2(uint32_t w, int half) {
  if constexpr (WD == MI_W_F8E4M3)
    return __builtin_bit_cast(uint32_t, half ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, true) : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, false));
  else return i8x2_to_bf16x2(w, 2 * half, 2 * half + 1);
}

// ---- cross-lane sums inside an aligned group of 4, 8 or 16 lanes (DPP, no LDS) ------------
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  float t = __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
  return v + t;
}
// after the call every lane of the group holds the group's sum
template <int LANES>
__device__ __forceinline__ float group_sum(float v) {
  static_assert(LANES == 4 || LANES == 8 || LANES == 16, "group of 4, 8 or 16 lanes");
  if (LANES == 16) v = dpp_add<0x140>(v);  // row_mirror       i <-> 15-i
  if (LANES >= 8) v = dpp_add<0x141>(v);   // row_half_mirror  i <-> 7-i (within 8)
  v = dpp_add<0xB1>(v);                    // quad_perm [1,0,3,2]
  v = dpp_add<0x4E>(v);                    // quad_perm [2,3,0,1]
  return v;
}

__device__ __forceinline__ float wave_sum(float v) {
  v = group_sum<16>(v);
  v += __shfl_xor(v, 16);
  v += __shfl_xor(v, 32);
  return v;
}

// streamed-once 16-byte load (global_load_dwordx4 ... nt): keeps weight bytes out of the way
// of the L2 lines that ARE reused (activations, scales)
__device__ __forceinline__ uint4 nt_load16(const uint4* p) {
  const u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
  return make_uint4(v[0], v[1], v[2], v[3]);
}

// A 16-byte store to `at` bytes behind `base` (the same for the whole wave) that does not stay in this XCD's L2 (sc1).  What a kernel leaves dirty there is written out when
// the kernel ends, in front of the next one's start; written through it leaves while the kernel still works.  (A builtin: the results of MFMAs that are still
// on their way are waited for in front of an instruction the compiler knows, and not in front of inline asm.)
__device__ __forceinline__ void store_through(void* base, uint32_t at, f32x4_t v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), __builtin_amdgcn_make_buffer_rsrc(base, 0, 0xffffffffu, 0x00020000), at, 0, 16);
}

// fp32 -> OCP e4m3fn, round-nearest-even, saturating at +-448: the hardware convert of gfx950 (v_cvt_pk_fp8_f32; OCP
// formats on this chip).  The clamp in front makes the result independent of the instruction's own out-of-range rule; a NaN
// input becomes +-448 like any other out-of-range value.  (Written out it is ~20 integer / select instructions per value,
// on which the per-token quantization passes of the FP8-activation path were VALU-bound.)
__device__ __forceinline__ uint32_t f32_to_e4m3fn(float f) {
  const float c = __builtin_fminf(__builtin_fmaxf(f, -448.f), 448.f);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(c, 0.f, 0, false) & 0xffu;
}


// ---- weight stream primitives -----------------------------------------------------------
// MI_STREAM_ASM = 0 (default): plain non-temporal loads; hipcc owns the s_waitcnt placement.
//   It drains to vmcnt(0) once per pair of batches, so latency is hidden by wave-level
//   parallelism (16 waves per CU), not by depth per wave.
// MI_STREAM_ASM = 1: loads issued from inline asm and retired by hand-counted waits
//   (cdna_hip_programming.md 5.7).  Measured hazard on hipcc 7.2: whenever an in-flight buffer is
//   live across a control-flow merge the register allocator resolves the phi with v_mov copies
//   of registers whose loads have not landed.  csrc/audit_stream.py detects exactly that in the
//   emitted ISA; the build refuses such a library.  Kept for experiments only.
#ifndef MI_STREAM_ASM
#define MI_STREAM_ASM 0
#endif
#if MI_STREAM_ASM
__device__ __forceinline__ void stream_load16(u32x4_t& dst, const uint4* p) {
  asm volatile("global_load_dwordx4 %0, %1, off nt ; stream_load" : "=v"(dst) : "v"(p) : "memory");
}
template <int N>
__device__ __forceinline__ void stream_wait(u32x4_t& r) {
  asm volatile("s_waitcnt vmcnt(%1) ; stream_release %0" : "+v"(r) : "n"(N) : "memory");
}
#else
__device__ __forceinline__ void stream_load16(u32x4_t& dst, const uint4* p) {
#ifdef MI_STREAM_PLAIN   // probe builds: default cache policy instead of the streaming hint
  dst = *reinterpret_cast<const u32x4_t*>(p);
#else
  dst = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
#endif
}
template <int N>
__device__ __forceinline__ void stream_wait(u32x4_t&) {}
#endif

// A batch of 1 KiB weight tiles from the `first` of W on, of which there are `n` (both the same for the whole wave): what lies beyond is zeros and no request to
// memory.  TWO: two descriptors, 4 KiB apart, where a second offset register is one too many (an instruction's own offset ends at 4095).
template <bool TWO = false, int U>
__device__ __forceinline__ void stream_batch(u32x4_t (&buf)[U], const uint4* W, int first, int n, int lane) {
  int bytes = min(max(n, 0), U) * 1024;
  asm("" : "+v"(first), "+v"(bytes));   // (else hipcc folds the two below away, keeps some in vector registers and loops over the lanes for the descriptor)
  const uint4* at = W + (size_t)(unsigned)__builtin_amdgcn_readfirstlane(first) * 64;
  const int size = __builtin_amdgcn_readfirstlane(bytes);
  constexpr int S = TWO ? 4 : U;
  const auto r = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint4*>(at), 0, size, 0x00020000);
  const auto r4 = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint4*>(at + 256), 0, max(size - 4096, 0), 0x00020000);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    buf[u] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(u < S ? r : r4, lane * 16 + u % S * 1024, 0, 2));   // (2: streaming, nt)
    __builtin_amdgcn_sched_barrier(0x3cf);   // in the order they are multiplied: a wait for one is a wait for all requested before it
  }
}

__host__ __device__ __forceinline__ int ceil_div(int a, int b) { return (a + b - 1) / b; }

// ---- per-device launch state ------------------------------------------------------------
// One process may drive several GPUs (the in-process tensor-parallel group): kernel attributes
// and the CU count belong to the CURRENT device, never to the process.
// A K-split GEMM whose slabs have not been summed yet: y[m, n] = (sum_z slab[z][m][n]) * scale[n] (* row_scale[m]) + bias[n]
// (the arithmetic of splitk_reduce_kernel + epilogue, in that order).  Consumed by the row-norm kernel that reads the
// residual stream next (one launch and one round trip of the residual less), or flushed by launch_splitk_flush.
struct SlabSum {
  const float* slab = nullptr;      // [KS][T][N] raw fp32 accumulators
  int KS = 0, T = 0, N = 0;
  const float* scale = nullptr;     // [N]
  const float* bias = nullptr;      // [N] or null
  const float* row_scale = nullptr; // [T] or null (FP8 activations)
  float rs_n = 0.f, rs_eps = 0.f;   // as EpiArgs
};
constexpr int kNormParts = 4;       // work-groups of a row in norm_parts_kernel, each with a sum of squares of its own
#ifdef __HIPCC__
// A row's factor: p[m], or (n > 0) 1 / rms of a row of n numbers from its parts' sums of squares p[kNormParts m ..].  Requests without a branch: what they stand
// behind stays in flight.
struct RowFactor {
  float a, b, c, d;
  __device__ __forceinline__ void request(const float* p, int m, float n) {
    const bool parts = n > 0.f;
    const float* q = p + (parts ? kNormParts * m : m);
    const int step = parts ? 1 : 0;
    a = q[0]; b = q[step]; c = q[2 * step]; d = q[3 * step];
  }
  __device__ __forceinline__ float value(float n, float eps) const { return n > 0.f ? rsqrtf(((a + b) + (c + d)) / n + eps) : a; }
};
// the same in two steps where the parts are known to be there
__device__ __forceinline__ float4 row_parts(const float* p, int m) { return *reinterpret_cast<const float4*>(p + kNormParts * m); }
__device__ __forceinline__ float row_rinv(float4 ss, float n, float eps) { return rsqrtf(((ss.x + ss.y) + (ss.z + ss.w)) / n + eps); }
// The sum of KS slabs' four numbers at p, `stride` numbers apart, in slice order.  Five requests leave before the first is waited for: one after the
// other they cost a trip to memory each (the row norm over 8 slabs of 242 x 4096: 13.9 us that way, 9.3 now, of which the bytes take 6.3).
struct Nothing { __device__ __forceinline__ void operator()() const {} };
template <typename F = Nothing>      // between(): other requests, behind the first slabs' ones
__device__ __forceinline__ float4 slab_sum4(const float* __restrict__ p, size_t stride, int KS, F&& between = F()) {
  constexpr int U = 5;
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int z = 0; z < KS; z += U) {
    float4 q[U];
#pragma unroll
    for (int u = 0; u < U; ++u) q[u] = *reinterpret_cast<const float4*>(p + (size_t)min(z + u, KS - 1) * stride);
    if (z == 0) between();
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (z + u < KS) { v.x += q[u].x; v.y += q[u].y; v.z += q[u].z; v.w += q[u].w; }
  }
  return v;
}
#endif
int device_num_cu(int* out);                                  // CUs of the current device
int ensure_dynamic_lds(const void* kernel, int bytes);        // hipFuncSetAttribute where (device, kernel) has fewer so far

// weight tile geometry: a tile is 16 rows x TILE_K(wd) columns = 1 KiB, lane l owns
// row (l & 15), k-chunk (l >> 4) of 16 bytes.
__host__ __device__ __forceinline__ int tile_k(int wd) { return wd == MI_W_BF16 ? 32 : 64; }
__host__ __device__ __forceinline__ int elem_bytes(int wd) { return wd == MI_W_BF16 ? 2 : 1; }

}  // namespace mi
