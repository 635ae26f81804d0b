// Paged-KV attention kernels for gfx950.  See attn_kernels.h for the contract.
//
// Token generation (attn_decode_kernel): HBM-bound.  One work-group per
// (context split, kv head, sequence); its waves walk 32-token tiles of the sequence's blocks,
// two tiles in flight per wave.  The query heads of the kv group are the columns of MFMA tiles
// (S^T = K.Q^T from K fragments loaded straight from the pool; O^T += V^T.P^T with V parked in a
// wave-private LDS tile and read transposed), so the arithmetic per byte is a few hundred
// cycles per 16 KiB tile -- the VALU dot-product form this replaced cost ~3000.  With fewer
// (sequence, kv head) pairs than CUs the context is split over work-groups and the splits are
// merged by attn_combine_kernel in a fixed order (deterministic); otherwise one work-group
// covers the whole sequence.
//
// Context encoding (attn_prefill_kernel): MFMA flash attention over the same pool.  Scores
// are computed transposed (S^T = K.Q^T) so the accumulator registers ARE the B operand of
// the P.V product (no LDS round trip for P); V is staged transposed in LDS.

#include "attn_kernels.h"

namespace mi {

#define MI_TRY_A(expr)             \
  do {                             \
    int _rc = (expr);              \
    if (_rc != MI_OK) return _rc;  \
  } while (0)

// LDS-DMA: 64 lanes x 16 bytes from per-lane global addresses into 1 KiB of LDS starting at `l` (wave-uniform)
__device__ __forceinline__ void glds16(const void* g, unsigned char* l) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                   (__attribute__((address_space(3))) void*)l, 16, 0, 0);
}

__device__ __forceinline__ float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }
// exp2(x - m) with the -inf conventions of online softmax (m finite or -inf)
__device__ __forceinline__ float sexp2(float x, float m) {
  return (x == -INFINITY) ? 0.f : fexp2(x - m);
}

// =====================================================================================
// token generation
// =====================================================================================
typedef __attribute__((ext_vector_type(4))) short s16x4_t;
constexpr int kNt = 2;   // a buffer load's `nt`: lines nobody reads again

// NW waves per work-group.  FINAL: the work-group covers the whole context of its (sequence, kv
// head) and writes the bf16 output itself (grid (1, nkv, B)); otherwise it covers context split
// blockIdx.x of NS and leaves (o, m, l) partials for attn_combine_kernel.
//
// A wave walks 32-token tiles.  The G <= 16 query heads of the kv group are the 16 columns of the
// MFMA tiles (the idle columns cost nothing: the kernel is bound by bytes, not by the matrix core):
//     S^T[token][head]  = K_tile . Q^T             2 x HD/32 MFMA 16x16x32 (two 16-token halves)
//     O^T[d][head]     += V_tile^T . P^T           HD/16 MFMA 16x16x32, k = the tile's 32 tokens
// K goes from the pool straight into A fragments (lane (g, c): token c, 16 B of the row).  V is
// read as whole rows, parked row-major in a wave-private LDS tile and picked up transposed by
// ds_read_b64_tr_b16.  The P.V k-slot (g, j) is bound to token (j < 4 ? 4g + j : 16 + 4g + j - 4),
// which is where the two S^T accumulators already hold that token's score, so the exponentiated
// scores are the B operand as they stand.
// Every wave keeps TWO tiles in flight (the next tile is requested before the current one is
// consumed); halves of a tile beyond the context lie outside of their buffer and read as zeros, so
// the loop has no predicated loads.  Rows of the last tile beyond the context are masked by score;
// the pool must not hold NaN/Inf there (the library zero-fills it and only ever writes finite values).
//
// MERGE (with !FINAL): the context splits of one (sequence, kv head) are merged by whichever of
// their NS work-groups finishes LAST, inside this launch -- no combine launch.  No work-group ever
// waits for another (nothing can hang): each publishes its partial with write-through (sc1) stores,
// every storing wave drains them, one lane takes a ticket from an agent-scope counter, and the
// work-group whose ticket is NS - 1 reads all NS partials back with sc1 loads (past its L1; no
// other reader of these lines exists in the launch, so no L2 holds a stale copy) and writes the
// bf16 output.  No fence is needed: the work-group whose add came last is told so by
// the value its add returned, and there is one work-group per CU (the launches that merge ask for
// kMergeLds of LDS to keep it so).  The merge itself runs in split order, so the
// result does not depend on which work-group performs it.  The counter is left at 0 for the next launch.
template <int HD, int NW, bool FINAL, bool MERGE = false>
__device__ __forceinline__ void attn_decode_body(
    unsigned char* dsm, int split, int kvh, int seq, const uint16_t* __restrict__ q, const uint16_t* __restrict__ kpool, const uint16_t* __restrict__ vpool,
    int bs, const int32_t* __restrict__ block_table, int MB, const int32_t* __restrict__ ctx_lens,
    int nh, int nkv, int G, int NS, float* __restrict__ o_part, float* __restrict__ ml_part,
    uint16_t* __restrict__ out, float scale_log2e, unsigned int* __restrict__ tickets, int R,
    int num_blocks) {
  // R > 1 (the target's pass of a speculation step): batch rows b R .. b R + R - 1 are the SAME sequence
  // at consecutive positions (one block-table row, context lengths growing by one).  Their query heads
  // sit side by side in the 16 MFMA columns (column = row-in-sequence * G + head, G R <= 16) and each
  // column masks by its own row's context length: the K/V of the sequence is read once, not R times.
  constexpr int KP = HD + 8;        // LDS row pitch (elements)
  constexpr int CPR = HD / 8;       // 16-byte chunks per row
  constexpr int KS = HD / 32, DN = HD / 16;
  constexpr int NV = 32 * CPR / 64; // 16-byte V loads per lane per tile
  constexpr int VT = 32 * KP;       // elements of one wave's V tile
  uint16_t* Vs = reinterpret_cast<uint16_t*>(dsm);                       // [NW][32][KP] bf16
  float* sm_ml = reinterpret_cast<float*>(dsm + (size_t)NW * VT * 2);    // [NW][16][2]

  const int b = seq * R;                        // first batch row of the sequence
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int g = lane >> 4, c = lane & 15;
  const int Gc = G * R;                         // live MFMA columns
  const int cr = c / G, ch = c - cr * G;        // column c = (row of the sequence, head of the kv group)
  // Tiles are dealt round-robin: wave w of split s takes tiles s NW + w, + NS NW, ...  Which tile a wave STARTS
  // with therefore does not depend on the context length, so (num_blocks > 0) its first K/V request goes out
  // beside the load of the context length instead of behind it (one L2 round trip less on the way to the first
  // MFMA); what it fetched is masked by score, or never consumed when the tile lies beyond the context.
  const int stride = NS * NW, t_first = split * NW + wave;
  uint16_t* Vw = Vs + wave * VT;

  // A 32-token tile is two 16-token halves; with block_size 16 (vLLM's default) they sit in two different blocks.  Lane 2 i + u holds the pool
  // row of half u of the wave's tile i_base + i: the block table is read once for 32 tiles, not in front of every request, where the wait for the block's
  // number was one for all requests before it (vector memory retires in order), so that two tiles never were in flight together.  us a launch, 8 kv heads of 128:
  // 32 sequences of 37 - 1000 tokens 23.3 -> 20.2, of 500 each 15.7 -> 14.6, 16 of 30 - 1000 14.6 -> 12.1; 5 of 4 kv heads, 300 - 1900 tokens 10.0 -> 8.4.
  constexpr int kIds = 32;
  auto rows_at = [&](int i0) {
    const int tok = (t_first + (i0 + (lane >> 1)) * stride) * 32 + (lane & 1) * 16, bi = tok / bs;
    int blk = block_table[(size_t)b * MB + min(bi, MB - 1)];
    if (num_blocks > 0) blk = min(max(blk, 0), num_blocks - 1);        // (asked for ahead of the context length: any row of the pool)
    return ((uint32_t)blk * nkv + kvh) * bs + (tok - bi * bs);
  };
  int i_base = 0;
  uint32_t rows = rows_at(0);
  // the wave's tile i; halves beyond the context read as zeros, without a request
  const int koff = (c * HD + g * 8) * 2, voff = lane * 16;
  u32x4_t kA[2 * KS], vA[NV], kB[2 * KS], vB[NV];
  auto issue = [&](u32x4_t (&kr)[2 * KS], u32x4_t (&vr)[NV], int i, int limit) {
    const int tok0 = (t_first + i * stride) * 32;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const size_t at = (size_t)(uint32_t)__builtin_amdgcn_readlane((int)rows, 2 * (i - i_base) + u) * HD;
      const int bytes = tok0 + 16 * u < limit ? 16 * HD * 2 : 0;
      const auto kb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(kpool) + at, 0, bytes, 0x00020000);
      // K fragment (u, ks): token 16u + c, dims 32 ks + 8 g ..
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        kr[u * KS + ks] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(kb, koff + ks * 64, 0, kNt));
    }
    // V rows: lane-linear 16-byte chunks (whole rows per instruction)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const size_t at = (size_t)(uint32_t)__builtin_amdgcn_readlane((int)rows, 2 * (i - i_base) + u) * HD;
      const auto vb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(vpool) + at, 0, tok0 + 16 * u < limit ? 16 * HD * 2 : 0, 0x00020000);
#pragma unroll
      for (int j = 0; j < NV / 2; ++j)
        vr[u * (NV / 2) + j] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(vb, voff + j * 1024, 0, kNt));
    }
  };
  if (num_blocks > 0) issue(kA, vA, 0, 0x7fffffff);
  int ctx = 0;                                  // the longest context of the sequence's rows bounds the tiles walked
  for (int r = 0; r < R; ++r) ctx = max(ctx, ctx_lens[b + r]);
  const int ctx_c = c < Gc ? ctx_lens[b + cr] : 0;   // what this lane's column may attend to
  if (num_blocks <= 0) issue(kA, vA, 0, ctx);
  const int nt = ceil_div(ctx, 32), mine = t_first < nt ? ceil_div(nt - t_first, stride) : 0;       // this wave's tiles

  u32x4_t qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
    qf[ks] = (c < Gc) ? *reinterpret_cast<const u32x4_t*>(q + ((size_t)(b + cr) * nh + kvh * G + ch) * HD + ks * 32 + g * 8)
                      : u32x4_t{0, 0, 0, 0};
  f32x4_t acc[DN];
#pragma unroll
  for (int dn = 0; dn < DN; ++dn) acc[dn] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float mrow = -INFINITY, lrow = 0.f;   // head c: running max (same on its 4 lanes), this lane's share of the sum
  const int tr_row = (lane & 15) >> 2, tr_col = (lane & 3) * 4;

  auto update = [&](const u32x4_t (&kr)[2 * KS], const u32x4_t (&vr)[NV], int tt) {
    // park V (the previous tile's transposed reads are complete: their values fed MFMAs already)
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = lane + 64 * i;
      *reinterpret_cast<u32x4_t*>(&Vw[(idx / CPR) * KP + (idx % CPR) * 8]) = vr[i];
    }
    asm volatile("" ::: "memory");   // LDS ops of one wave execute in order; keep the compiler from reordering them
    f32x4_t st[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      st[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const u32x4_t kw = kr[u * KS + ks], qw = qf[ks];
        st[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kw), __builtin_bit_cast(bf16x8_t, qw), st[u], 0, 0, 0);
      }
    }
    s16x4_t vlo[DN], vhi[DN];
#pragma unroll
    for (int dn = 0; dn < DN; ++dn) {
      const uint16_t* r0 = &Vw[(4 * g + tr_row) * KP + 16 * dn + tr_col];
      vlo[dn] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4_t __attribute__((address_space(3)))*)r0);
      vhi[dn] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4_t __attribute__((address_space(3)))*)(r0 + 16 * KP));
    }
    const int tok0 = tt * 32;
    float pv[8];
    float mx = -INFINITY;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float sv = st[u][i] * scale_log2e;
        if (tok0 + 16 * u + 4 * g + i >= ctx_c) sv = -INFINITY;
        pv[4 * u + i] = sv;
        mx = fmaxf(mx, sv);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));       // -inf where the column has no live token in this tile (sexp2 conventions)
    const float mn = fmaxf(mrow, mx);
    const float alpha = sexp2(mrow, mn);
    float ps = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      pv[k] = sexp2(pv[k], mn);
      ps += pv[k];
    }
    const bool moved = mn != mrow;
    mrow = mn;
    lrow = lrow * alpha + ps;
    union { uint32_t w[4]; bf16x8_t v; } pk;
#pragma unroll
    for (int k = 0; k < 4; ++k) pk.w[k] = pack_bf16x2(pv[2 * k], pv[2 * k + 1]);
    if (__any(moved)) {
#pragma unroll
      for (int dn = 0; dn < DN; ++dn) {
        acc[dn][0] *= alpha; acc[dn][1] *= alpha; acc[dn][2] *= alpha; acc[dn][3] *= alpha;
      }
    }
#pragma unroll
    for (int dn = 0; dn < DN; ++dn) {
      const s16x4_t lo = vlo[dn], hi = vhi[dn];
      const bf16x8_t a = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      acc[dn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pk.v, acc[dn], 0, 0, 0);
    }
  };

  for (int i = 0; i < mine; i += 2) {
    if (i + 3 > i_base + kIds) {
      i_base = i;
      rows = rows_at(i);
      asm volatile("" : "+v"(rows));            // (waited for here, not where every pass comes by)
    }
    issue(kB, vB, i + 1, ctx);
    update(kA, vA, t_first + i * stride);
    issue(kA, vA, i + 2, ctx);
    if (i + 1 < mine) update(kB, vB, t_first + (i + 1) * stride);
  }

  // ---- merge the waves: O^T / m / l of wave w go to its own (now idle) LDS tile --------------
  lrow += __shfl_xor(lrow, 16);
  lrow += __shfl_xor(lrow, 32);
  asm volatile("" ::: "memory");
  float* so = reinterpret_cast<float*>(Vw);            // [16 heads][HD] f32 = 8 KiB at HD 128 <= the tile
#pragma unroll
  for (int dn = 0; dn < DN; ++dn) *reinterpret_cast<f32x4_t*>(&so[c * HD + 16 * dn + 4 * g]) = acc[dn];
  if (g == 0) {
    sm_ml[(wave * 16 + c) * 2] = mrow;
    sm_ml[(wave * 16 + c) * 2 + 1] = lrow;
  }
  __syncthreads();
  for (int idx = tid; idx < Gc * HD; idx += NW * 64) {
    const int h = idx / HD, d = idx % HD;       // h: MFMA column
    const int hr = h / G, hh = h - hr * G;      // -> (row of the sequence, head)
    float M = sm_ml[h * 2];
#pragma unroll
    for (int w = 1; w < NW; ++w) M = fmaxf(M, sm_ml[(w * 16 + h) * 2]);
    float o = 0.f, L = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {  // wave order: deterministic
      const float f = sexp2(sm_ml[(w * 16 + h) * 2], M);
      o += f * reinterpret_cast<const float*>(Vs + w * VT)[h * HD + d];
      L += f * sm_ml[(w * 16 + h) * 2 + 1];
    }
    if constexpr (FINAL) {
      out[((size_t)(b + hr) * nh + kvh * G + hh) * HD + d] = f32_to_bf16(L > 0.f ? o / L : 0.f);   // empty context -> zeros
    } else if constexpr (MERGE) {
      const size_t row = ((size_t)(b + hr) * nh + kvh * G + hh) * kAttnMaxSplits + split;   // fixed stride: a head's m/l block is one 128-byte line
      __hip_atomic_store(&o_part[row * HD + d], o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // global_store ... sc1
      if (d == 0) {
        __hip_atomic_store(&ml_part[row * 2], M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&ml_part[row * 2 + 1], L, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    } else {
      const size_t row = ((size_t)(b + hr) * nh + kvh * G + hh) * kAttnMaxSplits + split;   // fixed stride: a head's m/l block is one 128-byte line
      o_part[row * HD + d] = o;
      if (d == 0) {
        ml_part[row * 2] = M;
        ml_part[row * 2 + 1] = L;
      }
    }
  }
  if constexpr (MERGE && !FINAL) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // EVERY storing wave drains its write-through stores
    __syncthreads();
    int* s_last = reinterpret_cast<int*>(sm_ml);        // the m/l staging is dead behind the barrier
    if (tid == 0) {
      unsigned int* tk = tickets + (size_t)b * nkv + kvh;
      const unsigned int t = __hip_atomic_fetch_add(tk, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const bool last = t == (unsigned int)(NS - 1);
      if (last) __hip_atomic_store(tk, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // ready for the next launch
      *s_last = last ? 1 : 0;
    }
    __syncthreads();
    if (*s_last) {
      for (int idx = tid; idx < G * HD; idx += NW * 64) {
        const int h = idx / HD, d = idx % HD;
        const size_t row0 = ((size_t)b * nh + kvh * G + h) * kAttnMaxSplits;
        float mv[kAttnMaxSplits], lv[kAttnMaxSplits], ov[kAttnMaxSplits];
#pragma unroll
        for (int sp = 0; sp < kAttnMaxSplits; ++sp) {
          const bool ok = sp < NS;
          mv[sp] = ok ? __hip_atomic_load(&ml_part[(row0 + sp) * 2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : -INFINITY;
          lv[sp] = ok ? __hip_atomic_load(&ml_part[(row0 + sp) * 2 + 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.f;
          ov[sp] = ok ? __hip_atomic_load(&o_part[(row0 + sp) * HD + d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.f;
        }
        float M = -INFINITY;
#pragma unroll
        for (int sp = 0; sp < kAttnMaxSplits; ++sp) M = fmaxf(M, mv[sp]);
        float acc_o = 0.f, L = 0.f;
#pragma unroll
        for (int sp = 0; sp < kAttnMaxSplits; ++sp) {   // split order: the same sums as attn_combine_kernel
          const float f = sexp2(mv[sp], M);
          acc_o += f * ov[sp];
          L += f * lv[sp];
        }
        out[((size_t)b * nh + kvh * G + h) * HD + d] = f32_to_bf16(L > 0.f ? acc_o / L : 0.f);
      }
    }
  }
}
template <int HD, int NW, bool FINAL, bool MERGE = false>
__global__ __launch_bounds__(NW * 64) void attn_decode_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ kpool, const uint16_t* __restrict__ vpool,
    int bs, const int32_t* __restrict__ block_table, int MB, const int32_t* __restrict__ ctx_lens,
    int nh, int nkv, int G, int NS, float* __restrict__ o_part, float* __restrict__ ml_part,
    uint16_t* __restrict__ out, float scale_log2e, unsigned int* __restrict__ tickets = nullptr, int R = 1,
    int num_blocks = 0) {
  extern __shared__ __attribute__((aligned(16))) unsigned char dsm[];
  attn_decode_body<HD, NW, FINAL, MERGE>(dsm, blockIdx.x, blockIdx.y, blockIdx.z, q, kpool, vpool, bs, block_table, MB, ctx_lens, nh, nkv, G, NS, o_part, ml_part, out,
                                         scale_log2e, tickets, R, num_blocks);
}
template <int HD, int NW>
constexpr size_t attn_decode_lds() { return (size_t)NW * 32 * (HD + 8) * 2 + (size_t)NW * 16 * 2 * sizeof(float); }
constexpr size_t kMergeLds = 96 * 1024;   // of a launch that merges: more than half a CU's LDS, so that no two of its work-groups share a CU

// Merge the context splits of one (sequence, head) in split order.  All partials are
// fetched before the first use (kAttnMaxSplits is a compile-time bound), so the kernel is
// one L2 round trip deep.
template <int HD>
__global__ __launch_bounds__(HD) void attn_combine_kernel(const float* __restrict__ o_part, const float* __restrict__ ml_part,
                                                          int NS, int nh, uint16_t* __restrict__ out) {
  const int head = blockIdx.x, b = blockIdx.y, d = threadIdx.x;
  const size_t row0 = ((size_t)b * nh + head) * kAttnMaxSplits;
  float mv[kAttnMaxSplits], lv[kAttnMaxSplits], ov[kAttnMaxSplits];
#pragma unroll
  for (int s = 0; s < kAttnMaxSplits; ++s) {
    const bool ok = s < NS;
    const float2 ml = ok ? *reinterpret_cast<const float2*>(ml_part + (row0 + s) * 2) : make_float2(-INFINITY, 0.f);
    mv[s] = ml.x;
    lv[s] = ml.y;
    ov[s] = ok ? o_part[(row0 + s) * HD + d] : 0.f;
  }
  float M = -INFINITY;
#pragma unroll
  for (int s = 0; s < kAttnMaxSplits; ++s) M = fmaxf(M, mv[s]);
  float acc = 0.f, L = 0.f;
#pragma unroll
  for (int s = 0; s < kAttnMaxSplits; ++s) {
    const float f = sexp2(mv[s], M);
    acc += f * ov[s];
    L += f * lv[s];
  }
  out[((size_t)b * nh + head) * HD + d] = f32_to_bf16(L > 0.f ? acc / L : 0.f);   // empty context -> zeros
}

// Up to 128 tokens of 128-wide heads (256 of 64-wide ones) four waves of one work-group take at most one tile (two) each, and the combine launch costs more
// than the split gains.  us per step, split + combine -> one launch: TinyLlama 1 row of 40 tokens 880 -> 822, of 250 892 -> 860; 8B fp8 4 rows
// of 64 / 125 tokens 1160 -> 1115 / 1128, at 250 / 450 tokens 1166 -> 1164 / 1217; 7B int8 6 rows of 200 1300 -> 1293.
bool attn_decode_short(int B, int nkv, int hd, int max_ctx) {
  return max_ctx > 0 && max_ctx * hd <= 128 * 128 && attn_decode_splits(B, nkv) > 1;
}
int attn_decode_splits(int B, int nkv) {
  int ns = 256 / (B * nkv);  // ~one work-group per CU; >= 4 tiles (one per wave) each at 1k context
  return ns < 1 ? 1 : (ns > kAttnMaxSplits ? kAttnMaxSplits : ns);
}
// [tickets: kAttnTickets counters, one per (sequence, kv head), zero between launches]
// [m/l partials: B x nh rows of one 128-byte line][o partials]  -- the ticket block and the m/l
// rows sit at offsets that do not depend on the batch size of the call
constexpr int kAttnTickets = 1024;
size_t attn_scratch_bytes(int B, int nh, int hd) {
  return kAttnTickets * sizeof(unsigned int) + (size_t)B * nh * kAttnMaxSplits * (hd + 2) * sizeof(float);
}
// In launches of decode rows alone off by default: measured on Llama-3.1-8B decode (B 4, ctx 1024) the in-launch merge costs the
// last work-group ~5.4 us (write-through drain + returning atomic + sc1 read-back are three
// dependent trips to memory) against 4.8 us for the separate combine launch: 2.157 vs 2.138 ms per
// step.  MI355X_ATTN_MERGE=1 selects it (same results: tests/test_model_gpu.py runs both).
static bool attn_merge_enabled() {
  static const bool on = [] { const char* v = getenv("MI355X_ATTN_MERGE"); return v && v[0] == '1'; }();
  return on;
}

template <int HD>
static int launch_decode_t(const uint16_t* q, const uint16_t* kpool, const uint16_t* vpool, int bs,
                           const int32_t* bt, int MB, const int32_t* ctx, int B, int nh, int nkv,
                           uint16_t* out, void* scratch, hipStream_t s, bool tickets_zeroed, int R, int num_blocks, int max_ctx) {
  const int G = nh / nkv, Bs = B / R, NS = attn_decode_splits(Bs, nkv);   // Bs sequences of R batch rows each
  // in-launch merge: needs every split's work-group resident on a CU of its own (grid <= CUs) and
  // the ticket counters at zero (the model keeps them so; the per-op entry cannot know)
  int num_cu = 0;
  if (device_num_cu(&num_cu) != MI_OK) return MI_EHIP;
  const bool merge = attn_merge_enabled() && R == 1 && NS > 1 && tickets_zeroed && NS * nkv * B <= num_cu && nkv * B <= kAttnTickets;
  unsigned int* tickets = reinterpret_cast<unsigned int*>(scratch);
  float* ml_part = reinterpret_cast<float*>(tickets + kAttnTickets);
  float* o_part = ml_part + (size_t)B * nh * kAttnMaxSplits * 2;
  const float scale_log2e = 1.4426950408889634f / sqrtf((float)HD);
  constexpr size_t lds8 = attn_decode_lds<HD, 8>(), lds4 = attn_decode_lds<HD, 4>();
  {
    int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(attn_decode_kernel<HD, 8, true>), (int)lds8);
    if (rc == MI_OK) rc = ensure_dynamic_lds(reinterpret_cast<const void*>(attn_decode_kernel<HD, 4, true>), (int)lds4);
    if (rc == MI_OK) rc = ensure_dynamic_lds(reinterpret_cast<const void*>(attn_decode_kernel<HD, 4, false>), (int)lds4);
    if (rc == MI_OK) rc = ensure_dynamic_lds(reinterpret_cast<const void*>(attn_decode_kernel<HD, 4, false, true>), (int)kMergeLds);
    if (rc != MI_OK) return rc;
  }
  if (attn_decode_short(Bs, nkv, HD, max_ctx)) {
    hipLaunchKernelGGL((attn_decode_kernel<HD, 4, true>), dim3(1, nkv, Bs), dim3(256), lds4, s, q,
                       kpool, vpool, bs, bt, MB, ctx, nh, nkv, G, 1, nullptr, nullptr, out, scale_log2e, nullptr, R, num_blocks);
  } else if (NS == 1) {
    // Enough (sequence, kv head) pairs to fill the chip: one launch, no partials.  (Measured: a
    // single CU sustains only ~32 GB/s from HBM however many loads its waves keep in flight, so
    // a short grid must split the context over CUs -- the one-launch form at B x nkv = 32 took
    // 16 us per 1k tokens of context against 8 + 5 us for split + combine.)
    hipLaunchKernelGGL((attn_decode_kernel<HD, 8, true>), dim3(1, nkv, Bs), dim3(512), lds8, s, q,
                       kpool, vpool, bs, bt, MB, ctx, nh, nkv, G, 1, nullptr, nullptr, out, scale_log2e, nullptr, R, num_blocks);
  } else if (merge) {
    hipLaunchKernelGGL((attn_decode_kernel<HD, 4, false, true>), dim3(NS, nkv, B), dim3(256), kMergeLds, s, q,
                       kpool, vpool, bs, bt, MB, ctx, nh, nkv, G, NS, o_part, ml_part, out, scale_log2e, tickets);
  } else {
    hipLaunchKernelGGL((attn_decode_kernel<HD, 4, false>), dim3(NS, nkv, Bs), dim3(256), lds4, s, q,
                       kpool, vpool, bs, bt, MB, ctx, nh, nkv, G, NS, o_part, ml_part, nullptr, scale_log2e, nullptr, R, num_blocks);
    hipLaunchKernelGGL((attn_combine_kernel<HD>), dim3(nh, B), dim3(HD), 0, s, o_part, ml_part, NS, nh, out);
  }
  MI_HIP(hipGetLastError());
  return MI_OK;
}

int launch_attn_decode(const uint16_t* q, const uint16_t* kpool, const uint16_t* vpool, int block_size,
                       const int32_t* block_table, int MB, const int32_t* ctx_lens, int B, int nh,
                       int nkv, int hd, uint16_t* out, void* scratch, hipStream_t s, bool tickets_zeroed, int rows_per_seq,
                       int num_blocks, int max_ctx) {
  MI_CHECK(hd == 64 || hd == 128, "attention: head_dim must be 64 or 128");
  MI_CHECK(rows_per_seq >= 1 && B % rows_per_seq == 0 && (nh / nkv) * rows_per_seq <= 16,
           "attention: rows_per_seq must divide the batch and q heads per kv head x rows_per_seq must be <= 16");
  MI_CHECK(nh % nkv == 0 && nh / nkv <= 16, "attention: q heads per kv head must be 1..16");
  MI_CHECK(block_size % 16 == 0, "attention: block_size must be a multiple of 16");
  if (hd == 128) return launch_decode_t<128>(q, kpool, vpool, block_size, block_table, MB, ctx_lens, B, nh, nkv, out, scratch, s, tickets_zeroed, rows_per_seq, num_blocks, max_ctx);
  return launch_decode_t<64>(q, kpool, vpool, block_size, block_table, MB, ctx_lens, B, nh, nkv, out, scratch, s, tickets_zeroed, rows_per_seq, num_blocks, max_ctx);
}

// =====================================================================================
// context encoding
// =====================================================================================
// One work-group per (32*QB queries, kv head): wave w owns q head (w % Gp) of the kv group and
// query block (w / Gp), i.e. 32 queries = two 16-query MFMA tiles that share every K / V
// fragment; the G heads of the group share the K/V tiles staged in LDS (one HBM read per group).
// Per 64-key tile:  S^T_u[key][q] = K_u . Q^T        (u = 0..3: four 16-key MFMA tiles)
//                   O^T[d][q]    += V^T[d][key] . P^T[key][q]   (two k-steps of 32 keys)
// The MFMA k-slot (g, j) of P.V k-step kk is bound to key 32 kk + (j < 4 ? 4g + j : 16 + 4g + j - 4),
// which is where S^T_{2kk} / S^T_{2kk+1} already hold that key's score for lane (g, q): the
// exponentiated accumulators are the B operand as they stand (no LDS round trip for P).  V stays
// row-major in LDS; its transposed A fragments come from ds_read_b64_tr_b16 (4 keys x 16 dims
// per 16-lane group).  Next tile's K/V are prefetched into registers under the MFMAs.

template <int HD, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void attn_prefill_kernel(
    const uint16_t* __restrict__ q, int T, int q_pos0, const uint16_t* __restrict__ kpool,
    const uint16_t* __restrict__ vpool, int bs, const int32_t* __restrict__ block_table, int nh, int nkv, int G,
    int Gp, int paired, uint16_t* __restrict__ out, float scale_log2e) {
  // row pitch (elements): head_dim + 16, i.e. 288 B = 72 banks (head_dim 128) or 160 B = 40 banks (64).  Either way the 16 rows
  // of a ds_read_b128 lane group start on 16 different 4-bank windows (its lanes of the next 16-byte column take the windows in
  // between) and the 8 rows of a ds_read_b64_tr_b16 group own 8 banks each: no conflicts.  (At head_dim + 8 one pair of lanes
  // per group met on a bank: 37 % of the LDS cycles, SQ_LDS_BANK_CONFLICT.)
  constexpr int KP = HD + 16;
  constexpr int CPR = HD / 8;   // 16-byte chunks per row
  constexpr int DN = HD / 16, KS = HD / 32;
  constexpr int TK = 64;        // keys per tile
  constexpr int LD = (TK * CPR) / (WAVES * 64);  // 16-byte loads per thread per K (or V) tile
  __shared__ __attribute__((aligned(16))) uint16_t Ks[TK * KP];
  __shared__ __attribute__((aligned(16))) uint16_t Vs[TK * KP];
  __shared__ int32_t bt_lds[kPrefillMaxBlocks];   // this sequence's block table: one L2 trip, not one per tile

  constexpr int nthr = WAVES * 64, waves = WAVES;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int g = lane >> 4, c = lane & 15;
  const int kvh = blockIdx.y, QB = waves / Gp;
  const int hl = wave % Gp, qb = wave / Gp;
  const bool head_ok = hl < G;
  const int head = kvh * G + min(hl, G - 1);
  const int kv_len = q_pos0 + T;
  for (int i = threadIdx.x; i < ceil_div(kv_len, bs); i += nthr) bt_lds[i] = block_table[i];

  // Causal work grows linearly with the query block index.  paired (long prompts): a work-group
  // takes block x and then its complement (nblk - 1 - x), every work-group the same number of key
  // tiles, one work-group per CU.  Otherwise one block per work-group, heaviest first: two
  // work-groups share a CU (a wave's softmax arithmetic runs under the other's MFMAs) and the
  // dispatcher hands out the light blocks as the heavy ones finish.  (Measured on Llama-8B shapes:
  // unpaired wins 1-3 % of the whole prefill up to the 1024 bucket, pairing wins 9 % at 2048.)
  const int nblk = ceil_div(T, 32 * QB);
  for (int pass = 0; pass < (paired ? 2 : 1); ++pass) {
  const int xb = !paired ? nblk - 1 - (int)blockIdx.x : (pass == 0 ? (int)blockIdx.x : nblk - 1 - (int)blockIdx.x);
  if (pass == 1 && xb <= (int)blockIdx.x) break;   // odd count: the middle block is done once
  const int wg_q0 = xb * 32 * QB;
  const int q0 = wg_q0 + 32 * qb;            // this wave's 32 queries

  u32x4_t qf[2][KS];
  int qpos[2];
  bool qok[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int qi = q0 + 16 * t + c;
    qok[t] = head_ok && qi < T;
    qpos[t] = q_pos0 + min(qi, T - 1);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[t][ks] = qok[t] ? *reinterpret_cast<const u32x4_t*>(q + ((size_t)qi * nh + head) * HD + ks * 32 + g * 8)
                         : u32x4_t{0, 0, 0, 0};
  }
  f32x4_t acc[2][DN];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int dn = 0; dn < DN; ++dn) acc[t][dn] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float mrow[2] = {-INFINITY, -INFINITY}, lrow[2] = {0.f, 0.f};

  const int wg_last_pos = q_pos0 + min(wg_q0 + 32 * QB - 1, T - 1);
  const int ntiles = wg_last_pos / TK + 1;
  const int w_first_pos = q_pos0 + min(q0, T - 1), w_last_pos = q_pos0 + min(q0 + 31, T - 1);

  __syncthreads();   // block table staged (pass 0) / previous pass done with the K/V tiles
  // register prefetch of one K/V tile (each thread: LD chunks of K and of V)
  // Two register sets, two tiles ahead: with one wave per SIMD a tile's arithmetic (~1 us) is
  // shorter than an HBM round trip, so the tile after next is requested before this one is used.
  // (ext vectors: hipcc keeps arrays of them in VGPRs; HIP's uint4 struct goes to scratch)
  u32x4_t kregA[LD], vregA[LD], kregB[LD], vregB[LD];
  auto prefetch = [&](u32x4_t (&kreg)[LD], u32x4_t (&vreg)[LD], int tile) {
    tile = min(tile, ntiles - 1);
#pragma unroll
    for (int i = 0; i < LD; ++i) {
      const int idx = tid + i * nthr;
      const int key = idx / CPR, ch = idx % CPR;
      const int ta = min(tile * TK + key, kv_len - 1);   // clamp: rows past the context are masked anyway
      const int blk = bt_lds[ta / bs];
      const size_t src = (((size_t)blk * nkv + kvh) * bs + (ta % bs)) * HD + ch * 8;
      kreg[i] = *reinterpret_cast<const u32x4_t*>(kpool + src);
      vreg[i] = *reinterpret_cast<const u32x4_t*>(vpool + src);
    }
  };
  prefetch(kregA, vregA, 0);
  prefetch(kregB, vregB, 1);

  auto do_tile = [&](u32x4_t (&kreg)[LD], u32x4_t (&vreg)[LD], int tile) {
    __syncthreads();  // every wave is done reading the previous tile
#pragma unroll
    for (int i = 0; i < LD; ++i) {
      const int idx = tid + i * nthr;
      const int key = idx / CPR, ch = idx % CPR;
      *reinterpret_cast<u32x4_t*>(&Ks[key * KP + ch * 8]) = kreg[i];
      *reinterpret_cast<u32x4_t*>(&Vs[key * KP + ch * 8]) = vreg[i];
    }
    __syncthreads();
    prefetch(kreg, vreg, tile + 2);
    if (tile * TK > w_last_pos) return;   // wave-uniform: every key of this tile is in this wave's future

    // ---- S^T = K . Q^T ------------------------------------------------------------------
    // One wave per SIMD: latency is hidden by issue order, not by other waves.  All 16 K
    // fragments are requested first, then the 32 MFMAs run back to back.
    bf16x8_t kf[4][KS];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        kf[u][ks] = *reinterpret_cast<const bf16x8_t*>(&Ks[(16 * u + c) * KP + ks * 32 + g * 8]);
    f32x4_t st[4][2];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      st[u][0] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      st[u][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        st[u][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[u][ks], __builtin_bit_cast(bf16x8_t, qf[0][ks]), st[u][0], 0, 0, 0);
        st[u][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[u][ks], __builtin_bit_cast(bf16x8_t, qf[1][ks]), st[u][1], 0, 0, 0);
      }
    }
    // V^T fragments for the P.V product: requested now, so their LDS latency runs under the
    // softmax arithmetic.  tr read: lane 4q' + p of a 16-lane group addresses row q' (a key),
    // columns 4p..4p+3 (dims); lane i receives column i (dim 16 dn + i) of the 4 rows = 4
    // consecutive k-slots of the A fragment.
    const int tr_row = (lane & 15) >> 2, tr_col = (lane & 3) * 4;
    s16x4_t vlo[2][DN], vhi[2][DN];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int dn = 0; dn < DN; ++dn) {
        const uint16_t* r0 = &Vs[(32 * kk + 4 * g + tr_row) * KP + 16 * dn + tr_col];
        vlo[kk][dn] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4_t __attribute__((address_space(3)))*)r0);
        vhi[kk][dn] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4_t __attribute__((address_space(3)))*)(r0 + 16 * KP));
      }
    // ---- causal mask + online softmax (query c of q-tile t; its keys sit on the 4 lanes g) --
    // Only the tiles that straddle the diagonal need the mask; every other tile takes the lean
    // path: max on the raw scores, then one fma + one exp2 per score.  The O^T rescale is skipped
    // (exactly: alpha == 1) when no lane's running maximum moved.
    const bool need_mask = tile * TK + TK - 1 > w_first_pos;
    bf16x8_t pb[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float pv[16];
      float mn, alpha, ps = 0.f;
      if (need_mask) {
        float mx = -INFINITY;
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float sv = st[u][t][i] * scale_log2e;
            if (tile * TK + 16 * u + 4 * g + i > qpos[t]) sv = -INFINITY;
            st[u][t][i] = sv;
            mx = fmaxf(mx, sv);
          }
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        mn = fmaxf(mrow[t], mx);
        alpha = sexp2(mrow[t], mn);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            pv[4 * u + i] = sexp2(st[u][t][i], mn);
            ps += pv[4 * u + i];
          }
      } else {
        float mx = st[0][t][0];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) mx = fmaxf(mx, st[u][t][i]);
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        mn = fmaxf(mrow[t], mx * scale_log2e);      // finite: every key of the tile is visible
        alpha = fexp2(mrow[t] - mn);                // exp2(-inf) = 0 on the first tile
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            pv[4 * u + i] = fexp2(fmaf(st[u][t][i], scale_log2e, -mn));
            ps += pv[4 * u + i];
          }
      }
      const bool moved = mn != mrow[t];
      mrow[t] = mn;
      lrow[t] = lrow[t] * alpha + ps;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        union { uint32_t w[4]; bf16x8_t v; } pk;
#pragma unroll
        for (int k = 0; k < 4; ++k) pk.w[k] = pack_bf16x2(pv[8 * kk + 2 * k], pv[8 * kk + 2 * k + 1]);
        pb[t][kk] = pk.v;
      }
      if (__any(moved)) {
#pragma unroll
        for (int dn = 0; dn < DN; ++dn) {
          acc[t][dn][0] *= alpha; acc[t][dn][1] *= alpha; acc[t][dn][2] *= alpha; acc[t][dn][3] *= alpha;
        }
      }
    }
    // ---- O^T += V^T . P^T ----------------------------------------------------------------
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
      for (int dn = 0; dn < DN; ++dn) {
        const s16x4_t lo = vlo[kk][dn], hi = vhi[kk][dn];
        const bf16x8_t a = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        acc[0][dn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb[0][kk], acc[0][dn], 0, 0, 0);
        acc[1][dn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb[1][kk], acc[1][dn], 0, 0, 0);
      }
    }
  };
  for (int tile = 0; tile < ntiles; tile += 2) {
    do_tile(kregA, vregA, tile);
    if (tile + 1 < ntiles) do_tile(kregB, vregB, tile + 1);
  }
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    float lsum = lrow[t];
    lsum += __shfl_xor(lsum, 16);
    lsum += __shfl_xor(lsum, 32);
    if (qok[t]) {
      const float inv = 1.f / lsum;
      uint16_t* orow = out + ((size_t)(q0 + 16 * t + c) * nh + head) * HD;
#pragma unroll
      for (int dn = 0; dn < DN; ++dn) {
        const uint2 pk = make_uint2(pack_bf16x2(acc[t][dn][0] * inv, acc[t][dn][1] * inv),
                                    pack_bf16x2(acc[t][dn][2] * inv, acc[t][dn][3] * inv));
        *reinterpret_cast<uint2*>(orow + 16 * dn + 4 * g) = pk;
      }
    }
  }
  }  // pass
}


// =====================================================================================
// context encoding, second generation: 32x32x16 MFMAs, K/V tiles by LDS-DMA, two waves per SIMD
// =====================================================================================
// What the counters of the kernel above asked for (17 % MFMA-busy at one wave per
// SIMD, 408 registers, 144 accumulator moves and a ds_write staging pass per 64-key tile):
//   * a wave owns ONE 32-query block of one q head: S^T[key][q] = K . Q^T on v_mfma_f32_32x32x16_bf16
//     puts a query on a lane (its 32 scores of a 64-key tile in 32 registers of lanes l and l + 32), so
//     the row maximum / sum is 31 VALU ops and ONE v_permlane32_swap, and the exponentiated
//     accumulators, packed pairwise to bf16, ARE the B operand of O^T[d][q] += V^T . P^T (k-slot j of
//     lane half h <-> key 16 s + 8 (j >> 2) + 4 h + (j & 3): the transposed V reads are bound to that order);
//   * K and V tiles (64 keys) arrive by LDS-DMA (global_load_lds, 1 KiB per wave-instruction) into a
//     ring of three 32 KiB stages: no staging registers, no ds_write, two tiles in flight while one is
//     multiplied, retired by a counted vmcnt in front of ONE raw barrier per tile.  The paged pool is
//     addressed per piece (4 keys x 256 B at head_dim 128): the block id is a scalar load, the per-lane
//     part of the source address is constant for the whole kernel;
//   * the LDS image is rows of head_dim bf16 whose 16-byte chunks are XOR-swizzled by the key (applied
//     to the per-lane SOURCE address of the DMA and to the reads): conflict-free for the ds_read_b128
//     row reads of K (16 lanes = 16 keys = 16 different slots) and for the ds_read_b64_tr_b16
//     transposed reads of V (a half-wave's 4 keys land on 4 different 64-byte windows);
//   * ~170 registers: two waves per SIMD.  A work-group is NW waves = QB query blocks x Gp q heads of
//     one kv group, all sharing the K/V ring.  Causal work grows with the block index, so the QB blocks
//     of a work-group are complementary pairs (j, nblk - 1 - j): every SIMD of the chip gets the same
//     number of key tiles, and the light block's waves keep issuing DMAs for the heavy one's tail.
// Softmax: the running maximum used in the exponent is only moved when the tile's maximum exceeds it
// by more than kDeferLog2 (deferred rescale): p <= 2^kDeferLog2 instead of <= 1, O and l carry the
// same factor, the quotient O / l is unchanged up to rounding; the 64-register rescale of O^T becomes rare.
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
constexpr float kDeferLog2 = 6.f;

// {v of this lane, v of lane ^ 32} in some order (max / sum do not care): one v_permlane32_swap.  The elements of the
// builtin's result are copied out before the bit cast: hipcc 7.2 reads element 0 for __builtin_bit_cast(float, r[1]),
// which made a row's sum 2 x (its lower half's sum).
__device__ __forceinline__ f32x2_t swap32_pair(float v) {
  const unsigned a = __builtin_bit_cast(unsigned, v);
  const auto r = __builtin_amdgcn_permlane32_swap(a, a, false, false);
  const unsigned r0 = r[0], r1 = r[1];
  return f32x2_t{__builtin_bit_cast(float, r0), __builtin_bit_cast(float, r1)};
}

template <int HD>
__device__ __forceinline__ int kv_swz(int key) {   // XOR key of the 16-byte chunk index of a K/V row in LDS
  if constexpr (HD == 128) return ((key & 3) << 2) | ((key >> 2) & 3);          // 256-byte rows, 16 chunks
  else return (((key >> 1) & 1) << 2) | ((key >> 2) & 3);                        // 128-byte rows,  8 chunks
}

constexpr int kPrefillSlices = 6;   // of the keys, at most

// A work-group has the heads of one kv head, or the sub-th of `subs` equal parts of them.
// KH 2: the waves of a head are two, which take a step's two tiles of keys, one each, and put their sums together at the end: a work-group then has one query
// block at a time (NW = 2 Gp).  KH 1: a wave takes every tile of its block, and a work-group has NW / Gp blocks.
// A tile is a chain of LDS reads, products and exponentials, 1.6 us for a wave that has its SIMD to itself and 1.3 where two share it.  With 4 heads on a kv head two
// blocks used to share a work-group: the wave of the light one left the other alone for most of the way, and up to 1000 tokens half of the CUs had none.
// Alone, us, 32 heads of 128 on 8: 500 tokens 16.0 -> 13.6, 1000 26.8 -> 22.2, 900 behind 900 47.1 -> 33.9, 2031 49.3 -> 45.9 (60 tokens, whose one tile leaves the second wave idle, 7.1 -> 7.6: those keep KH 1).
// Without the loads from memory 2031 tokens take 40.0, without the exponentials 44.5; half a step between the two parts (as in the wide GEMM): 53.4.
// 16 waves for 8 heads do not fit the registers: 5 .. 8 heads on a kv head go to two work-groups, which both read its keys.  28 heads of 128 on 4, us: 500 tokens
// 18.8 -> 14.0, 1000 32.0 -> 22.3, 188 behind 512 23.0 -> 16.5, 900 behind 900 51.7 -> 33.2, 2031 58.1 -> 44.0; 32 heads of 64 on 4: 239 8.6 -> 6.9, 1000 23.2 -> 15.1, 2031 42.6 -> 30.0.
template <int HD, int NW, int KH>
__device__ __forceinline__ void attn_prefill2_body(
    unsigned char* smem, int bx, int kvh, int sub, int subs, int bz, int nz, const uint16_t* __restrict__ q, int T, int q_pos0, const uint16_t* __restrict__ kpool,
    const uint16_t* __restrict__ vpool, int bs, int bs_shift, const int32_t* __restrict__ block_table, int nh, int nkv,
    int G, int Gp, int nblk, int paired, float* __restrict__ o_part, float* __restrict__ ml_part, uint16_t* __restrict__ out, float scale_log2e) {
  constexpr int TK = 64;                       // keys per tile
  constexpr int ROWB = HD * 2;                 // bytes per K/V row
  constexpr int CPR = HD / 8;                  // 16-byte chunks per row
  constexpr int KPP = 1024 / ROWB;             // keys per 1 KiB DMA piece (4 / 8)
  constexpr int NP = TK / KPP;                 // pieces per K (or V) tile (16 / 8)
  constexpr int KBYTES = TK * ROWB;            // 16 / 8 KiB
  constexpr int VAT = KH * KBYTES;             // a stage: the K of a step's KH tiles, then their V
  constexpr int STAGE = 2 * VAT;
  constexpr int NSTAGE = KH == 1 ? 3 : 2;
  constexpr int PPW = KH * NP / NW;            // K pieces per wave and step (V the same)
  static_assert(KH * NP % NW == 0, "pieces must divide over the waves");
  constexpr int CNT = 2 * PPW;                 // DMA instructions per wave and step
  constexpr int KSTEPS = HD / 16, DB = HD / 32, DW = DB / KH;   // (DW: 32-dim blocks of the output that a wave stores)

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int QB = KH == 1 ? NW / Gp : 1;
  const int hl = wave % Gp, slot = KH == 1 ? wave / Gp : 0, part = KH == 1 ? 0 : wave / Gp;
  const int per = ceil_div(G, subs), h0 = min(sub * per, G - 1), hn = min(per, G - sub * per);      // this work-group's heads of the kv head's (hn <= 0: none)
  const int head = kvh * G + h0 + max(min(hl, hn - 1), 0);
  const bool head_ok = hl < hn;
  const int kv_len = q_pos0 + T;
  const int last_piece_key = ((kv_len - 1) / KPP) * KPP;
  const int qq = lane & 31, h = lane >> 5;
  const int npair = (nblk + 1) >> 1;

  // ---- per-lane constants of the LDS image -------------------------------------------------------
  // DMA: lane i of a piece fills slot (i % CPR) of key (i / CPR) of the piece: it fetches the chunk the swizzle puts there
  const int kip = lane / CPR, dslot = lane % CPR;
  int dma_sw;
  if constexpr (HD == 128) dma_sw = (kip << 2) | (wave & 3);                 // kv_swz(4 piece + kip), piece = wave (mod 4)
  else dma_sw = (((kip >> 1) & 1) << 2) | ((2 * (wave & 1) + (kip >> 2)) & 3);   // kv_swz(8 piece + kip), piece = wave (mod 2)
  const int dma_lane_off = kip * HD + ((dslot ^ dma_sw) * 8);                // elements, relative to the piece's first row
  // K row reads (A operand of S^T): key qq of a 32-key block, chunk 2 ks + h
  int kaddr[KSTEPS];
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) kaddr[ks] = qq * ROWB + (((2 * ks + h) ^ kv_swz<HD>(qq)) * 16);
  // V transposed reads (A operand of O^T): group gi = lane >> 4 covers dims 16 (gi & 1) .. + 15 of a 32-dim block for lane half
  // h = gi >> 1; lane 4 qr + pc of the group addresses key row (4 h + qr [+ 8]) at dims 4 pc .. 4 pc + 3
  const int gi = lane >> 4, qr = (lane & 15) >> 2, pc = lane & 3;
  int vaddr[DB][2];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int key = 4 * h + qr + 8 * u;                                     // (+ 32 b + 16 s: no effect on the swizzle key)
      const int chunk = 4 * db + 2 * (gi & 1) + (pc >> 1);
      vaddr[db][u] = key * ROWB + ((chunk ^ kv_swz<HD>(key)) * 16) + 8 * (pc & 1);
    }

  const int passes = QB == 1 && paired ? 2 : 1;
  for (int pass = 0; pass < passes; ++pass) {
    // ---- which query block this wave owns --------------------------------------------------------
    int blk_q, pair;
    bool blk_ok;
    if (QB == 1 && !paired) {            // a work-group per block, the heavy ones first
      pair = bx;
      blk_q = nblk - 1 - pair;
      blk_ok = pair < nblk;
    } else if (QB == 1) {                // one block at a time: the heavy one of pair bx, then the light one
      pair = bx;
      blk_q = pass == 0 ? nblk - 1 - pair : pair;
      blk_ok = pair < npair && !(pass == 1 && pair == nblk - 1 - pair);
    } else {
      pair = bx * (QB >> 1) + (slot >> 1);
      blk_q = (slot & 1) ? nblk - 1 - pair : pair;
      blk_ok = pair < npair && !((slot & 1) && pair == nblk - 1 - pair);
    }
    const int q0 = blk_q * 32;
    const bool active = blk_ok && head_ok;
    // tiles: this wave's, and the work-group's (the heaviest block any of its waves owns)
    const int p_first = q_pos0 + min(q0, T - 1), p_last = q_pos0 + min(q0 + 31, T - 1);
    const int nt_wave = active ? p_last / TK + 1 : 0;
    int wg_pair0 = QB == 1 ? bx : bx * (QB >> 1);
    int wg_blk = QB == 1 ? (pass == 0 ? nblk - 1 - wg_pair0 : wg_pair0) : nblk - 1 - wg_pair0;   // heaviest block of the work-group
    wg_blk = max(min(wg_blk, nblk - 1), 0);
    const int nt_all = (q_pos0 + min(wg_blk * 32 + 31, T - 1)) / TK + 1;
    // steps of this slice of them: all, or the bz-th of nz slices of the keys
    const int steps = ceil_div(nt_all, KH), s_per = ceil_div(steps, nz), s0 = bz * s_per, s1 = min(steps, s0 + s_per);

    // ---- Q fragments (B operand of S^T): Q[q0 + qq][16 ks + 8 h ..] ---------------------------------
    const int qi = min(q0 + qq, T - 1);
    const int qpos = q_pos0 + qi;
    u32x4_t qf[KSTEPS];
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks)
      qf[ks] = active ? *reinterpret_cast<const u32x4_t*>(q + ((size_t)qi * nh + head) * HD + ks * 16 + h * 8) : u32x4_t{0, 0, 0, 0};

    f32x16_t o[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[db][r] = 0.f;
    float m_used = -INFINITY, lsum = 0.f;

    // Block ids are fetched (scalar loads) one step ahead of the DMAs that use them: the round trip to the scalar cache / L2
    // runs under a tile's arithmetic instead of in front of the global_load_lds it feeds.
    int pf_blk[PPW], pf_off[PPW];
    auto fetch_ids = [&](int t) {
#pragma unroll
      for (int i = 0; i < PPW; ++i) {
        const int k0 = min(t * KH * TK + (wave + NW * i) * KPP, last_piece_key);   // rows past the context: the last piece again (masked by position)
        int bi;
        if (bs_shift >= 0) { bi = k0 >> bs_shift; pf_off[i] = k0 & (bs - 1); }
        else { bi = k0 / bs; pf_off[i] = k0 - bi * bs; }
        pf_blk[i] = block_table[bi];
      }
    };
    auto issue = [&](int st) {                  // the step whose ids fetch_ids loaded last
      unsigned char* base = smem + st * STAGE;
#pragma unroll
      for (int i = 0; i < PPW; ++i) {
        const int piece = wave + NW * i;
        const size_t row = ((size_t)pf_blk[i] * nkv + kvh) * bs + pf_off[i];
        glds16(kpool + row * HD + dma_lane_off, base + piece * 1024);
        glds16(vpool + row * HD + dma_lane_off, base + VAT + piece * 1024);
      }
    };

    constexpr int kAhead = NSTAGE - 1;          // steps in flight in front of the one that is read
    int st_issue = kAhead, st_read = 0;
    if (s0 < s1) { fetch_ids(s0); issue(0); }
    if (kAhead > 1 && s0 + 1 < s1) { fetch_ids(s0 + 1); issue(1); }
    fetch_ids(s0 + kAhead);
    // hipcc waits for a plain load at its first use -- inside the tile loop, as vmcnt(0) on every iteration, which would drain
    // the two tiles in flight each time.  Taking the Q fragments through an empty asm here puts that wait in front of the loop.
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) asm volatile("" : "+v"(qf[ks]));
    for (int step = s0; step < s1; ++step) {
      if (kAhead > 1 && step + 1 < s1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(CNT) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();            // every wave's pieces of this step are in; everyone is done reading the one before
      if (step + kAhead < s1) {
        issue(st_issue);
        st_issue = st_issue == NSTAGE - 1 ? 0 : st_issue + 1;
        fetch_ids(step + kAhead + 1);
      }
      const int t = step * KH + part;
      const unsigned char* Kst = smem + st_read * STAGE + part * KBYTES;
      const unsigned char* Vst = Kst + VAT;
      st_read = st_read == NSTAGE - 1 ? 0 : st_read + 1;
      if (t >= nt_wave) continue;                // wave-uniform: the tile lies in this block's future (or the slot is idle)

      // ---- S^T = K . Q^T : two 32-key blocks.  The K fragments of a block are requested one block ahead of the MFMAs
      // that take them (8 reads in flight; hipcc left to itself issues read -> wait -> MFMA one at a time) ----
      f32x16_t sc[2];
      {
        bf16x8_t kf[KSTEPS];
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) kf[ks] = *reinterpret_cast<const bf16x8_t*>(Kst + kaddr[ks]);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
#pragma unroll
          for (int r = 0; r < 16; ++r) sc[b][r] = 0.f;
#pragma unroll
          for (int ks = 0; ks < KSTEPS; ++ks) {
            sc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[ks], __builtin_bit_cast(bf16x8_t, qf[ks]), sc[b], 0, 0, 0);
            if (b == 0) kf[ks] = *reinterpret_cast<const bf16x8_t*>(Kst + 32 * ROWB + kaddr[ks]);
          }
        }
        __builtin_amdgcn_sched_group_barrier(0x100, KSTEPS, 0);
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      }
      // ---- online softmax: this lane holds 32 scores of query qq (keys (r & 3) + 8 (r >> 2) + 4 h of each block) ----
      const bool need_mask = t * TK + TK - 1 > p_first;
      if (need_mask) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (t * TK + 32 * b + (r & 3) + 8 * (r >> 2) + 4 * h > qpos) sc[b][r] = -INFINITY;
      }
      float mx = sc[0][0];
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[b][r]);
      {
        const f32x2_t sw = swap32_pair(mx);
        mx = fmaxf(sw[0], sw[1]);
      }
      const float ms = mx * scale_log2e;         // key 0 is visible to every query: finite from the first tile on, but for a later slice of the keys
      const bool moved = ms > m_used + kDeferLog2;
      if (__any(moved)) {
        const float mn = moved ? ms : m_used;
        const float alpha = moved ? fexp2(m_used - mn) : 1.f;   // exp2(-inf) = 0 on the first tile
        m_used = mn;
        lsum *= alpha;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
      }
      // ---- p = exp2(s - m), packed to bf16 = the B operands of O^T += V^T . P^T.  The transposed V fragments of the first
      // kVAhead MFMAs are requested in front of the exponentials (no dependence), the rest kVAhead MFMAs ahead of their use ----
      // The transposed reads are inline asm: behind the builtin hipcc assumes the read may alias the LDS-DMAs in flight and
      // drains them (s_waitcnt vmcnt(0) per tile).  Their completion is counted by hand: LDS reads return in order, and between
      // the first V read of a tile and its last MFMA the wave issues no other LDS or scalar-memory instruction.
      constexpr int NPV = 4 * DB;               // MFMAs: (b, s2) outer, d-block inner
      constexpr int kVAhead = 4;
      s16x4_t vlo[NPV], vhi[NPV];
      unsigned vbase[DB][2];
      const unsigned vst_lds = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)Vst;
#pragma unroll
      for (int db = 0; db < DB; ++db) { vbase[db][0] = vst_lds + vaddr[db][0]; vbase[db][1] = vst_lds + vaddr[db][1]; }
#define MI_VREAD(i_)                                                                                                         \
      do {                                                                                                                   \
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(vlo[i_]) : "v"(vbase[(i_) % DB][0]), "n"(16 * ((i_) / DB) * ROWB)); \
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(vhi[i_]) : "v"(vbase[(i_) % DB][1]), "n"(16 * ((i_) / DB) * ROWB)); \
      } while (0)
      MI_VREAD(0); MI_VREAD(1); MI_VREAD(2); MI_VREAD(3);
      static_assert(kVAhead == 4, "the prefetch above is written out for 4");
      bf16x8_t pb[4];
      const float m_exp = (KH > 1 || nz > 1) && m_used == -INFINITY ? 0.f : m_used;   // (a slice or part whose keys so far all lie ahead of this query)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        float pv[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          pv[r] = fexp2(fmaf(sc[b][r], scale_log2e, -m_exp));    // masked: exp2(-inf) = 0
          lsum += pv[r];
        }
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          union { uint32_t w[4]; bf16x8_t v; } pk;
#pragma unroll
          for (int k = 0; k < 4; ++k) pk.w[k] = pack_bf16x2(pv[8 * s2 + 2 * k], pv[8 * s2 + 2 * k + 1]);
          pb[2 * b + s2] = pk.v;
        }
      }
      // ---- O^T += V^T . P^T --------------------------------------------------------------------------
      // before MFMA i: reads issued = 2 min(i + 1 + kVAhead - 1, NPV) ... all but the ones behind fragment i may be outstanding
#define MI_PV(i_)                                                                                                            \
      do {                                                                                                                   \
        constexpr int issued = 2 * ((i_) + kVAhead < NPV ? (i_) + kVAhead : NPV);                                            \
        asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(vlo[i_]), "+v"(vhi[i_]) : "n"(issued - 2 * ((i_) + 1)));               \
        const s16x4_t lo = vlo[i_], hi = vhi[i_];                                                                            \
        const bf16x8_t a = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};                                         \
        o[(i_) % DB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, pb[(i_) / DB], o[(i_) % DB], 0, 0, 0);                     \
        if constexpr ((i_) + kVAhead < NPV) MI_VREAD((i_) + kVAhead);                                                        \
      } while (0)
      MI_PV(0); MI_PV(1); MI_PV(2); MI_PV(3); MI_PV(4); MI_PV(5); MI_PV(6); MI_PV(7);
      if constexpr (NPV == 16) { MI_PV(8); MI_PV(9); MI_PV(10); MI_PV(11); MI_PV(12); MI_PV(13); MI_PV(14); MI_PV(15); }
#undef MI_PV
#undef MI_VREAD
    }
    // ---- epilogue: O^T[d][q] / l -> out[q][head][d]; lanes l and l + 32 hold neighbouring 4-dim groups of one query:
    // one v_permlane32_swap per pair of groups makes 16-byte stores of them
    {
      const f32x2_t sw = swap32_pair(lsum);
      lsum = sw[0] + sw[1];
    }
    const bool st_ok = active && q0 + qq < T;
    // the wave's blocks of dims, from d0 on; KH 2: behind the other part's sums for them, which come through the ring's LDS
    auto finish = [&](auto d0c) {
      constexpr int d0 = decltype(d0c)::value;
      if constexpr (KH > 1) {
        constexpr int other = DB - DW - d0, kPiece = DW * 4096 + 512;         // DW x 4 x [lane] f32x4, [lane] (m, l)
        unsigned char* mine = smem + wave * kPiece;
        const unsigned char* theirs = smem + (part == 0 ? wave + Gp : wave - Gp) * kPiece;
        __syncthreads();                       // everyone is done reading the ring
#pragma unroll
        for (int i = 0; i < DW * 4; ++i) {
          const int db = other + i / 4, r = 4 * (i % 4);
          *reinterpret_cast<f32x4_t*>(mine + i * 1024 + lane * 16) = f32x4_t{o[db][r], o[db][r + 1], o[db][r + 2], o[db][r + 3]};
        }
        *reinterpret_cast<f32x2_t*>(mine + DW * 4096 + lane * 8) = f32x2_t{m_used, lsum};
        __syncthreads();
        const f32x2_t ml = *reinterpret_cast<const f32x2_t*>(theirs + DW * 4096 + lane * 8);
        // (a part without a key for this query counts nothing; a NaN score moves no maximum: the sum carries it)
        const float M = fmaxf(m_used, ml[0]);
        const float wa = m_used == -INFINITY && lsum == 0.f ? 0.f : fexp2(m_used - M), wb = ml[0] == -INFINITY && ml[1] == 0.f ? 0.f : fexp2(ml[0] - M);
        lsum = lsum * wa + ml[1] * wb;
        m_used = M;
#pragma unroll
        for (int i = 0; i < DW * 4; ++i) {
          const f32x4_t v = *reinterpret_cast<const f32x4_t*>(theirs + i * 1024 + lane * 16);
#pragma unroll
          for (int k = 0; k < 4; ++k) o[d0 + i / 4][4 * (i % 4) + k] = o[d0 + i / 4][4 * (i % 4) + k] * wa + v[k] * wb;
        }
      }
      if (nz > 1) {   // unnormalised, with its maximum and sum: attn_prefill_combine_kernel puts the slices together
        const size_t row = ((size_t)bz * T + q0 + qq) * nh + head;
        if (st_ok && h == 0 && part == 0) *reinterpret_cast<float2*>(ml_part + 2 * row) = make_float2(m_used, lsum);
        if (st_ok && (m_used != -INFINITY || lsum != 0.f)) {
#pragma unroll
          for (int db = d0; db < d0 + DW; ++db)
#pragma unroll
            for (int k = 0; k < 4; ++k)
              *reinterpret_cast<float4*>(o_part + row * HD + 32 * db + 8 * k + 4 * h) =
                  make_float4(o[db][4 * k], o[db][4 * k + 1], o[db][4 * k + 2], o[db][4 * k + 3]);
        }
        return;
      }
      // (KH 2: a sum of 0 is one behind scores that are all -inf, whose row is 0 x inf, the NaN it is where one wave takes all tiles)
      const float inv = KH > 1 || lsum > 0.f ? 1.f / lsum : 0.f;
      uint16_t* orow = out + ((size_t)(q0 + qq) * nh + head) * HD;
#pragma unroll
      for (int db = d0; db < d0 + DW; ++db)
#pragma unroll
        for (int k2 = 0; k2 < 4; k2 += 2) {      // dim groups k2, k2 + 1: dims 32 db + 8 k + 4 h + (0..3)
          uint32_t a0 = pack_bf16x2(o[db][4 * k2 + 0] * inv, o[db][4 * k2 + 1] * inv);
          uint32_t a1 = pack_bf16x2(o[db][4 * k2 + 2] * inv, o[db][4 * k2 + 3] * inv);
          uint32_t b0 = pack_bf16x2(o[db][4 * k2 + 4] * inv, o[db][4 * k2 + 5] * inv);
          uint32_t b1 = pack_bf16x2(o[db][4 * k2 + 6] * inv, o[db][4 * k2 + 7] * inv);
          const auto x = __builtin_amdgcn_permlane32_swap(a0, b0, false, false);
          const auto y = __builtin_amdgcn_permlane32_swap(a1, b1, false, false);
          // lower half: [own group k2 | upper's group k2] = dims 8 k2 .. 8 k2 + 7; upper half: [lower's k2 + 1 | own k2 + 1]
          const u32x4_t v = {x[0], y[0], x[1], y[1]};
          if (st_ok) *reinterpret_cast<u32x4_t*>(orow + 32 * db + 8 * (k2 + h)) = v;
        }
    };
    if (KH == 1 || part == 0) finish(std::integral_constant<int, 0>());
    else finish(std::integral_constant<int, DB - DW>());
    __syncthreads();   // the ring is reused by the next pass
  }
}
template <int HD, int NW, int KH>
constexpr int attn_prefill2_lds() { return std::max((KH == 1 ? 3 : 2) * KH * 2 * 64 * 2 * HD, KH == 1 ? 0 : NW * (HD / 64 * 4096 + 512)); }
// The kv heads are the fastest of the grid: with 8 (4) of them an XCD's work-groups read the keys of one, and the heavy blocks of all start first.
template <int HD, int NW, int KH>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_prefill2_kernel(
    const uint16_t* __restrict__ q, int T, int q_pos0, const uint16_t* __restrict__ kpool,
    const uint16_t* __restrict__ vpool, int bs, int bs_shift, const int32_t* __restrict__ block_table, int nh, int nkv,
    int G, int Gp, int subs, int nblk, int paired, float* __restrict__ o_part, float* __restrict__ ml_part, uint16_t* __restrict__ out, float scale_log2e) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int parts = KH > 1 ? subs : 1, kvh = (int)blockIdx.x / parts;
  attn_prefill2_body<HD, NW, KH>(smem, blockIdx.y, kvh, (int)blockIdx.x - kvh * parts, parts, blockIdx.z, gridDim.z, q, T, q_pos0, kpool, vpool, bs, bs_shift, block_table, nh, nkv, G, Gp, nblk, paired, o_part,
                             ml_part, out, scale_log2e);
}

// A prompt's chunk and the requests that generate beside it, in one launch: neither fills the chip, and one after the other they cost 11.1 + 8.0 us at 239 tokens
// beside 3 contexts of up to 900 (8B model).  Work-groups x from `nd` on are the prompt's, gx of every slice of the keys; those before them one
// (split, sequence) each of the others.
struct DecodeSide { const uint16_t* q; const int32_t* block_table; const int32_t* ctx_lens; int MB, NS, nd, num_blocks; float *o_part, *ml_part; uint16_t* out; unsigned int* tickets; };
template <int HD, int KH, bool FINAL>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_mixed_kernel(
    const uint16_t* __restrict__ q, int T, int q_pos0, const uint16_t* __restrict__ kpool,
    const uint16_t* __restrict__ vpool, int bs, int bs_shift, const int32_t* __restrict__ block_table, int nh, int nkv,
    int G, int Gp, int subs, int nblk, int paired, int gx, int ns, float* __restrict__ o_part, float* __restrict__ ml_part, uint16_t* __restrict__ out, float scale_log2e, DecodeSide d) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  if ((int)blockIdx.x >= d.nd) {
    const int x = (int)blockIdx.x - d.nd;
    const int two = KH > 1 && subs == 2, y = two ? x >> 1 : x;      // (four sub-groups: not here)
    attn_prefill2_body<HD, 8, KH>(smem, y % gx, blockIdx.y, two ? x & 1 : 0, two ? 2 : 1, y / gx, ns, q, T, q_pos0, kpool, vpool, bs, bs_shift, block_table, nh, nkv, G, Gp, nblk,
                              paired, o_part, ml_part, out, scale_log2e);
  } else {
    attn_decode_body<HD, 8, FINAL, !FINAL>(smem, (int)blockIdx.x % d.NS, blockIdx.y, (int)blockIdx.x / d.NS, d.q, kpool, vpool, bs, d.block_table, d.MB, d.ctx_lens, nh, nkv, G, d.NS,
                                   d.o_part, d.ml_part, d.out, scale_log2e, d.tickets, 1, d.num_blocks);
  }
}

// the slices of the keys put together: out = sum_z 2^(m_z - M) O_z / sum_z 2^(m_z - M) l_z; four elements of a head per thread
template <int HD>
__global__ __launch_bounds__(256) void attn_prefill_combine_kernel(const float* __restrict__ o_part, const float* __restrict__ ml_part, int ns, int rows,
                                                                   uint16_t* __restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x, row = i / (HD / 4), d = i % (HD / 4) * 4;
  if (row >= rows) return;                     // rows = tokens x heads
  float2 ml[kPrefillSlices];
  float4 o[kPrefillSlices];
  float M = -INFINITY;
#pragma unroll
  for (int z = 0; z < kPrefillSlices; ++z) {   // requests of every slice leave together; those behind the last are copies of it and count nothing
    const size_t r = (size_t)min(z, ns - 1) * rows + row;
    ml[z] = *reinterpret_cast<const float2*>(ml_part + 2 * r);
    o[z] = *reinterpret_cast<const float4*>(o_part + r * HD + d);
  }
#pragma unroll
  for (int z = 0; z < kPrefillSlices; ++z) M = fmaxf(M, ml[z].x);
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  float l = 0.f;
#pragma unroll
  for (int z = 0; z < kPrefillSlices; ++z) {
    if (z >= ns || (ml[z].x == -INFINITY && ml[z].y == 0.f)) continue;   // (a slice without a key for this query wrote no O)
    const float w = fexp2(ml[z].x - M);
    l = fmaf(w, ml[z].y, l);
    v.x = fmaf(w, o[z].x, v.x); v.y = fmaf(w, o[z].y, v.y); v.z = fmaf(w, o[z].z, v.z); v.w = fmaf(w, o[z].w, v.w);
  }
  const float inv = 1.f / l;   // every query sees key 0: l is 0 only behind scores that are all -inf, whose row is 0 x inf, the NaN it is without slices
  *reinterpret_cast<uint2*>(out + (size_t)row * HD + d) = make_uint2(pack_bf16x2(v.x * inv, v.y * inv), pack_bf16x2(v.z * inv, v.w * inv));
}

static bool attn_prefill_v1() {   // MI355X_ATTN_PREFILL_V1=1: the first-generation kernel (A/B)
  static const bool on = [] { const char* v = getenv("MI355X_ATTN_PREFILL_V1"); return v && v[0] == '1'; }();
  return on;
}

static int prefill_heads(int G) { return G <= 1 ? 1 : (G <= 2 ? 2 : (G <= 4 ? 4 : 8)); }
struct PrefillPlan { int Gp, kh, nw, subs, nblk, bs_shift, paired, gx, ns; float *o_part = nullptr, *ml_part = nullptr; };
// Where one wave a head takes less time, from 3 heads on a kv head on.  By two waves each, 5 to 8 heads are two work-groups, and 3 and 4 leave the second block of a pair to a second pass:
// behind a long prefix, or in another round of work-groups, that can cost more than the waves save.  Tiles that a work-group walks, of its block or of a pair of blocks one after the other,
// times the rounds (single waves of 3 and 4 heads: pairs side by side, the heavy ones first, so a later round is half as long); a step of two tiles by two waves takes 1.1 of a tile by one, where
// that one shares its SIMD 1.4 (64-wide heads: never).  Of 400 shapes (4 to 16 kv heads, 100 .. 2048 tokens behind 0 .. 6000) the choice is 0.1 % from the faster on the average, 9 % at worst.
// us, two waves -> one: 64 heads of 128 on 8, 1500 tokens 72 -> 57, 2048 92 -> 79; 64 of 64 on 8, 1500 43 -> 37; 32 of 128 on 8, 1500 behind 2000 98 -> 92; but 28 on 4, 1500 behind 2000 87 (97).
static bool prefill_one_wave(int heads, int T, int q_pos0, int nkv, int hd, int num_cu) {
  const int nblk = ceil_div(T, 32), npair = (nblk + 1) / 2, kv = q_pos0 + T;
  const auto walk = [&](int kh) {
    const int groups = nkv * (heads == 8 ? kh : 1), paired = nblk * groups > num_cu;
    return (ceil_div(kv, 64 * kh) + (paired ? ceil_div(q_pos0 + 32, 64 * kh) : 0)) * ceil_div((paired ? npair : nblk) * groups, num_cu);
  };
  if (heads == 8) return walk(1) < 1.1 * walk(2);
  return hd == 128 && ceil_div(kv, 64) + (ceil_div(npair * nkv, num_cu) - 1) * ceil_div(q_pos0 + T / 2, 64) < 1.4 * walk(2);
}
static PrefillPlan prefill_plan(int T, int q_pos0, int block_size, int nh, int nkv, int hd, float* ws, size_t ws_bytes, int num_cu, bool mixed = false) {
  // second generation: 8 waves = (8 / Gp) query blocks x Gp heads, blocks in complementary pairs; or, from 3 heads on a kv head on, a block of up to 4 heads, two waves each
  PrefillPlan p;
  p.Gp = prefill_heads(nh / nkv);
  // two waves a head from half a second tile on (81 keys, 17 tokens: 6.6 -> 7.2 us; 97: as fast)
  p.kh = p.Gp >= 4 && q_pos0 + T > 96 && !prefill_one_wave(p.Gp, T, q_pos0, nkv, hd, num_cu) ? 2 : 1;
  p.subs = p.kh == 2 && p.Gp == 8 ? 2 : 1;
  if (p.subs == 2) p.Gp = 4;
  p.nw = 8;
  const int groups = nkv * p.subs;             // of heads: work-groups that read the same queries' keys
  const int nblk = ceil_div(T, 32), npair = (nblk + 1) / 2, qb = p.kh == 2 ? 1 : 8 / p.Gp;
  int bs_shift = -1;
  for (int sh = 4; sh < 20; ++sh) if ((1 << sh) == block_size) bs_shift = sh;
  // One block per work-group (two waves a head, or 5 .. 8 heads): pairs only where single blocks would not all run at once.
  const int paired = qb > 1 || nblk * groups > num_cu;
  const int gx = paired ? ceil_div(npair, qb >= 2 ? qb / 2 : 1) : nblk;
  // A short prompt, or the rest of one behind cached keys, leaves most of the chip idle while each work-group walks its tiles, 1.75 us each (two of them by pairs of waves 2.4, 1.4 of 64-wide heads):
  // slices of the keys then, at least two tiles each, the cheapest by that and the second launch, which moves every slice's O out and in.
  // 188 tokens behind 512 cached ones, 28 heads on 4: 40.8 us in 12 work-groups of two passes, 16.7 + 4.8 in four slices, 13.8 + 4.8 in three by pairs of waves, 16.5 by
  // pairs without: what slices cost whatever their number is more there.  (Not with 64-wide heads: 100 tokens behind 800, 32 heads on 4, 1439 us a call with slices, 1497 without.)
  int ns = 1;
  const int steps = ceil_div(q_pos0 + T, 64 * p.kh);
  const double per_step = p.kh == 1 ? 1.75 : hd == 128 ? 2.4 : 1.4;
  double best = per_step * steps * ceil_div(gx * groups, num_cu);
  for (int z = 2; ws && z <= kPrefillSlices; ++z) {
    const size_t part = (size_t)z * T * nh;
    if (ceil_div(steps, z) * p.kh < 2 || part * (hd + 2) * sizeof(float) > ws_bytes) break;
    const double cost = per_step * ceil_div(steps, z) * ceil_div(gx * groups * z, num_cu) + (p.kh == 2 && hd == 128 ? 6.0 : 4.5) + (double)part * hd * 8.0 / 4e6;
    if (cost < best) { best = cost; ns = z; }
  }
  // Where twice the work-groups find a CU each: two heads to a work-group of four waves.  A wave then has its SIMD to itself, and a work-group half the results to put together: some 1 us less and 0.2 a
  // step.  us a call: 7B int8 188 behind 512 tokens 2276 -> 2253, 300 tokens 3301 -> 3272, 8B fp8 100 1938 -> 1911, 400 3717 -> 3679, TinyLlama 300 1711 -> 1686, bf16 100 behind 800 1653 -> 1629.  Not in
  // place of slices: 8B 136 tokens behind 864 2287 in slices, 2325 in fewer slices of these; 236 behind 1664 2758 and 2800.
  if (!mixed && p.kh == 2 && nblk * groups * 2 <= num_cu && (per_step - 0.2) * steps - 1.0 < best) {
    p.nw = 4;
    p.Gp = 2;
    p.subs *= 2;
    ns = 1;
  }
  p.nblk = nblk; p.bs_shift = bs_shift; p.paired = paired; p.gx = gx; p.ns = ns;
  if (ns > 1) { p.o_part = ws; p.ml_part = ws + (size_t)ns * T * nh * hd; }
  return p;
}
static void launch_prefill_combine(const PrefillPlan& p, int T, int nh, int hd, uint16_t* out, hipStream_t s) {
  if (p.ns <= 1) return;
  const dim3 grid(ceil_div(T * nh * (hd / 4), 256));
  if (hd == 128) hipLaunchKernelGGL((attn_prefill_combine_kernel<128>), grid, dim3(256), 0, s, p.o_part, p.ml_part, p.ns, T * nh, out);
  else hipLaunchKernelGGL((attn_prefill_combine_kernel<64>), grid, dim3(256), 0, s, p.o_part, p.ml_part, p.ns, T * nh, out);
}

int launch_attn_prefill(const uint16_t* q, int T, int q_pos0, const uint16_t* kpool, const uint16_t* vpool,
                        int block_size, const int32_t* block_table, int nh, int nkv, int hd, uint16_t* out,
                        hipStream_t s, float* ws, size_t ws_bytes) {
  MI_CHECK(hd == 64 || hd == 128, "attention: head_dim must be 64 or 128");
  MI_CHECK(T >= 1 && q_pos0 >= 0, "attention: bad T / q_pos0");
  MI_CHECK(nh % nkv == 0 && nh / nkv <= 8, "attention: q heads per kv head must be 1..8");
  MI_CHECK(ceil_div(q_pos0 + T, block_size) <= kPrefillMaxBlocks, "attention: context spans more than 4096 blocks");
  const int G = nh / nkv;
  const float scale_log2e = 1.4426950408889634f / sqrtf((float)hd);
  const int Gp = prefill_heads(G);
  if (!attn_prefill_v1()) {
    int num_cu = 0;
    MI_TRY_A(device_num_cu(&num_cu));
    const PrefillPlan p = prefill_plan(T, q_pos0, block_size, nh, nkv, hd, ws, ws_bytes, num_cu);
#define MI_P2(HD_, NW_, KH_) do { \
      constexpr int lds = attn_prefill2_lds<HD_, NW_, KH_>(); \
      MI_TRY_A(ensure_dynamic_lds(reinterpret_cast<const void*>(attn_prefill2_kernel<HD_, NW_, KH_>), lds)); \
      hipLaunchKernelGGL((attn_prefill2_kernel<HD_, NW_, KH_>), dim3(nkv * p.subs, p.gx, p.ns), dim3(NW_ * 64), lds, s, q, T, q_pos0, kpool, vpool, block_size, p.bs_shift, \
                         block_table, nh, nkv, G, p.Gp, p.subs, p.nblk, p.paired, p.o_part, p.ml_part, out, scale_log2e); \
    } while (0)
    if (p.kh == 1) { if (hd == 128) MI_P2(128, 8, 1); else MI_P2(64, 8, 1); }
    else if (p.nw == 4) { if (hd == 128) MI_P2(128, 4, 2); else MI_P2(64, 4, 2); }
    else { if (hd == 128) MI_P2(128, 8, 2); else MI_P2(64, 8, 2); }
#undef MI_P2
    launch_prefill_combine(p, T, nh, hd, out, s);
    MI_HIP(hipGetLastError());
    return MI_OK;
  }
  const int waves = Gp < 4 ? 4 : Gp, QB = waves / Gp;
  const int nqb = ceil_div(T, 32 * QB);
  const int paired = nqb * nkv > 384 ? 1 : 0;   // more blocks than 1.5 per CU: pair complementary ones
  const dim3 grid(paired ? ceil_div(nqb, 2) : nqb, nkv);
#define MI_PF(HD_, W_) hipLaunchKernelGGL((attn_prefill_kernel<HD_, W_>), grid, dim3(W_ * 64), 0, s, q, T, q_pos0, kpool, vpool, block_size, block_table, nh, nkv, G, Gp, paired, out, scale_log2e)
  if (hd == 128) { if (waves == 4) MI_PF(128, 4); else MI_PF(128, 8); }
  else { if (waves == 4) MI_PF(64, 4); else MI_PF(64, 8); }
#undef MI_PF
  MI_HIP(hipGetLastError());
  return MI_OK;
}

// Eight waves a work-group here, four in the launch of its own: half the splits, and none (so no combine launch) up to 256 tokens of 128-wide heads, 512 of 64-wide
// ones, twice the other's limit.  us per call, splits -> none: 8B fp8 239 + 3 of 250 tokens 2977 -> 2940, of 500 2974 -> 2988, of 1000 2979 -> 3114; 64 + 6 of 300
// 2177 -> 2145, of 600 2197 -> 2215; TinyLlama 300 + 4 of 500 2234 -> 2178, of 1000 2228 -> 2296.
// Splits are merged in this launch by whichever ends last (MERGE): what that takes is hidden by the prompt's work-groups, where a launch of one's own behind both was in line.  A work-group has its CU
// to itself (kMergeLds; two waves a SIMD).  us a call, combine launch -> merged: 8B fp8 239 + 3 2649 -> 2617 (a layer 10.6 + 4.7 -> 12.2), 64 + 6 1939 -> 1922, 500 + 1 3971 -> 3916, TinyLlama 300 + 4 1991 -> 1960,
// 7B int8 200 + 3 2515 -> 2506.
static int mixed_splits(const AttnMixed& m, int nkv, int hd) { return m.max_ctx > 0 && m.max_ctx * hd <= 256 * 128 ? 1 : ceil_div(attn_decode_splits(m.B, nkv), 2); }
template <int HD>
static int mixed_lds(int kh, int splits) {
  const int need = std::max<int>(kh == 2 ? attn_prefill2_lds<HD, 8, 2>() : attn_prefill2_lds<HD, 8, 1>(), (int)attn_decode_lds<HD, 8>());
  return splits > 1 ? std::max<int>(need, kMergeLds) : need;
}
int attn_mixed_lds(int hd, int kh, int splits) { return hd == 128 ? mixed_lds<128>(kh, splits) : mixed_lds<64>(kh, splits); }
template <int HD>
static int launch_mixed_t(const AttnMixed& m, const PrefillPlan& p, int T, int q_pos0, const uint16_t* q, const int32_t* bt, uint16_t* out, const uint16_t* kpool,
                          const uint16_t* vpool, int bs, int nh, int nkv, hipStream_t s) {
  const float scale_log2e = 1.4426950408889634f / sqrtf((float)HD);
  float* ml_part = reinterpret_cast<float*>(reinterpret_cast<unsigned int*>(m.scratch) + kAttnTickets);
  float* o_part = ml_part + (size_t)m.B * nh * kAttnMaxSplits * 2;
  const int NS = mixed_splits(m, nkv, HD);
  const DecodeSide d{m.q, m.block_table, m.ctx_lens, m.MB, NS, NS * m.B, m.num_blocks, o_part, ml_part, m.out, reinterpret_cast<unsigned int*>(m.scratch)};
  const int lds = attn_mixed_lds(HD, p.kh, NS);
  const auto fn = p.kh == 2 ? (NS == 1 ? attn_mixed_kernel<HD, 2, true> : attn_mixed_kernel<HD, 2, false>)
                            : (NS == 1 ? attn_mixed_kernel<HD, 1, true> : attn_mixed_kernel<HD, 1, false>);
  MI_TRY_A(ensure_dynamic_lds(reinterpret_cast<const void*>(fn), lds));
  hipLaunchKernelGGL(fn, dim3(d.nd + p.gx * p.ns * p.subs, nkv), dim3(512), lds, s, q, T, q_pos0, kpool, vpool, bs, p.bs_shift, bt, nh, nkv, nh / nkv, p.Gp, p.subs, p.nblk, p.paired,
                     p.gx, p.ns, p.o_part, p.ml_part, out, scale_log2e, d);
  launch_prefill_combine(p, T, nh, HD, out, s);
  MI_HIP(hipGetLastError());
  return MI_OK;
}
int launch_attn_mixed(const AttnMixed& m, int T, int q_pos0, const uint16_t* q, const int32_t* block_table, uint16_t* out, const uint16_t* kpool, const uint16_t* vpool,
                      int block_size, int nh, int nkv, int hd, hipStream_t s, float* ws, size_t ws_bytes) {
  MI_CHECK(hd == 64 || hd == 128, "attention: head_dim must be 64 or 128");
  MI_CHECK(block_size % 16 == 0, "attention: block_size must be a multiple of 16");
  MI_CHECK(T >= 1 && q_pos0 >= 0 && m.B >= 1, "attention: bad T / q_pos0");
  MI_CHECK(nh % nkv == 0 && nh / nkv <= 8, "attention: q heads per kv head must be 1..8");
  MI_CHECK(ceil_div(q_pos0 + T, block_size) <= kPrefillMaxBlocks, "attention: context spans more than 4096 blocks");
  // One launch where both sides find a CU for every work-group; beyond that the prompt's wait behind the others' (us per call, two launches -> one: 8B model
  // 239 + 3 tokens 3105 -> 2980, 64 + 6 2205 -> 2108, TinyLlama 300 + 4 2385 -> 2245, 8B bf16 500 + 6 4862 -> 4724; 1900 + 3 13035 -> 13097).
  int num_cu = 0;
  MI_TRY_A(device_num_cu(&num_cu));
  const PrefillPlan p = prefill_plan(T, q_pos0, block_size, nh, nkv, hd, ws, ws_bytes, num_cu, true);
  if (attn_prefill_v1() || (p.gx * p.ns * p.subs + mixed_splits(m, nkv, hd) * m.B) * nkv > num_cu) {
    int rc = launch_attn_decode(m.q, kpool, vpool, block_size, m.block_table, m.MB, m.ctx_lens, m.B, nh, nkv, hd, m.out, m.scratch, s, false, 1, m.num_blocks, m.max_ctx);
    return rc != MI_OK ? rc : launch_attn_prefill(q, T, q_pos0, kpool, vpool, block_size, block_table, nh, nkv, hd, out, s, ws, ws_bytes);
  }
  return hd == 128 ? launch_mixed_t<128>(m, p, T, q_pos0, q, block_table, out, kpool, vpool, block_size, nh, nkv, s)
                   : launch_mixed_t<64>(m, p, T, q_pos0, q, block_table, out, kpool, vpool, block_size, nh, nkv, s);
}

// =====================================================================================
// standalone KV write (the model path writes K/V from the QKV epilogue instead)
// =====================================================================================
__global__ void kv_write_kernel(const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
                                const int64_t* __restrict__ slots, int nkv, int hd, uint16_t* __restrict__ kpool,
                                uint16_t* __restrict__ vpool, int bs) {
  const int t = blockIdx.x;
  const long slot = slots[t];
  if (slot < 0) return;
  const int blk = (int)(slot / bs), off = (int)(slot % bs);
  const int chunks = nkv * hd / 8;
  for (int i = threadIdx.x; i < chunks; i += blockDim.x) {
    const int head = (i * 8) / hd, d = (i * 8) % hd;
    const size_t dst = (((size_t)blk * nkv + head) * bs + off) * hd + d;
    *reinterpret_cast<uint4*>(kpool + dst) = *reinterpret_cast<const uint4*>(k + (size_t)t * nkv * hd + i * 8);
    *reinterpret_cast<uint4*>(vpool + dst) = *reinterpret_cast<const uint4*>(v + (size_t)t * nkv * hd + i * 8);
  }
}

int launch_kv_write(const uint16_t* k, const uint16_t* v, const int64_t* slots, int T, int nkv, int hd,
                    uint16_t* kpool, uint16_t* vpool, int block_size, hipStream_t s) {
  MI_CHECK(hd % 8 == 0, "kv_write: head_dim % 8 == 0 required");
  if (T == 0) return MI_OK;
  hipLaunchKernelGGL(kv_write_kernel, dim3(T), dim3(128), 0, s, k, v, slots, nkv, hd, kpool, vpool, block_size);
  MI_HIP(hipGetLastError());
  return MI_OK;
}

}  // namespace mi
