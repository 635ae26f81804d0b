// Gated delta rule.  See delta_rule.h.
#include "delta_rule.h"

#include <algorithm>

namespace mi {

namespace {

constexpr int kC = kDeltaChunk;

__device__ __forceinline__ float silu(float v) { return v * __builtin_amdgcn_rcpf(1.f + __expf(-v)); }
__device__ __forceinline__ float gate(float v) { return __builtin_amdgcn_rcpf(1.f + __expf(-v)); }
__device__ __forceinline__ float sigmoid(float v) { return 1.f / (1.f + expf(-v)); }
// max(v, 0) + log(1 + w), w = exp(-|v|): the series where w is small (its first left-out term is w^5 / 5)
__device__ __forceinline__ float softplus(float v) {
  const float w = __expf(-fabsf(v)), series = w * (1.f - w * (0.5f - w * (1.f / 3.f - 0.25f * w)));
  return fmaxf(v, 0.f) + (w < 0.02f ? series : __logf(1.f + w));
}
__device__ __forceinline__ float log_decay(float z, float dt, float a_log) { return -expf(a_log) * softplus(z + dt); }
__device__ __forceinline__ void put1(uint16_t* p, float v) { *p = f32_to_bf16(v); }
__device__ __forceinline__ void put1(float* p, float v) { *p = v; }
__device__ __forceinline__ void put4(uint16_t* p, const float (&v)[4]) { *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])); }
__device__ __forceinline__ void put4(float* p, const float (&v)[4]) { *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]); }

// ---- token generation ---------------------------------------------------------------------------------------------------------
// One work-group per (head, row): the whole state of the head in registers, requested first; thread (vq, dg) owns columns
// 4 vq .. + 3 of rows dg RPT .. + RPT - 1.  Both products with the decayed state are taken in one pass (o = S^T q + (k.q) u).
constexpr int kTokenThreads = 512;
template <typename T, int VQ, int RPT>
__global__ __launch_bounds__(kTokenThreads) void delta_token_kernel(DeltaGeom g, DeltaIn in, const AttnSeg* __restrict__ segs, T* __restrict__ y, int ldy) {
  constexpr int NW = kTokenThreads / 64;
  __shared__ float qs[256], ks[256], gs[256], vs[256];
  __shared__ float norms[3];
  __shared__ __attribute__((aligned(16))) float red[2][NW][VQ * 4];
  const int h = blockIdx.x, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  int row = blockIdx.y, seq = blockIdx.y;
  if (segs) {
    const AttnSeg sg = segs[blockIdx.y];
    if (sg.n != 1) return;
    row = sg.row0; seq = sg.seq;
  }
  const int slot = in.slots[seq], p = in.pos[row], vq = tid % VQ, dg = tid / VQ;
  const bool vin = vq * 4 < g.dvp;
  float* S0 = in.state + ((size_t)slot * g.H + h) * g.dkp * g.dvp + vq * 4;
  float4 S[RPT];
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int d = dg * RPT + i;
    S[i] = p > 0 && vin && d < g.dkp ? *reinterpret_cast<const float4*>(S0 + (size_t)d * g.dvp) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  // convolutions of the head's channels; position p goes to a row of the ring that nobody reads in this launch
  const int C = g.channels(), r = g.H / g.G, kvh = h / r;
  const float* x = in.proj + (size_t)row * in.ldp;
  float* ring = in.ring + (size_t)slot * g.taps * C;
  for (int i = tid; i < 2 * g.dk + g.dv; i += kTokenThreads) {
    const int part = i < g.dk ? 0 : i < 2 * g.dk ? 1 : 2, d = i - part * g.dk;
    const int ch = part == 2 ? 2 * g.G * g.dk + h * g.dv + d : (part * g.G + kvh) * g.dk + d;
    const float now = x[ch];
    float a = 0.f;
    for (int j = 0; j + 1 < g.taps; ++j) {
      const int q = p - (g.taps - 1 - j);
      if (q >= 0) a = __builtin_fmaf(in.conv[(size_t)j * C + ch], ring[(size_t)(q % g.taps) * C + ch], a);
    }
    a = silu(__builtin_fmaf(in.conv[(size_t)(g.taps - 1) * C + ch], now, a));
    if (part == 2 || h % r == 0) ring[(size_t)(p % g.taps) * C + ch] = now;
    (part == 0 ? qs : part == 1 ? ks : vs)[d] = a;
  }
  for (int d = tid; d < g.dkp; d += kTokenThreads) {
    if (d >= g.dk) { qs[d] = ks[d] = 0.f; gs[d] = 1.f; continue; }
    gs[d] = expf(log_decay(in.z[(size_t)row * in.ldz + h * g.dk + d], in.dt[h * g.dk + d], in.a_log[h]));
  }
  for (int d = g.dv + tid; d < g.dvp; d += kTokenThreads) vs[d] = 0.f;
  const float beta = sigmoid(x[in.beta + h]);
  __syncthreads();
  if (wave < 3) {
    float s = 0.f;
    for (int d = lane; d < g.dk; d += 64) s = __builtin_fmaf(wave == 1 ? ks[d] : qs[d], wave == 0 ? qs[d] : ks[d], s);
    s = wave_sum(s);
    if (lane == 0) norms[wave] = s;
  }
  __syncthreads();
  const float fq = 1.f / sqrtf(norms[0] + 1e-6f) * (1.f / sqrtf((float)g.dk)), fk = 1.f / sqrtf(norms[1] + 1e-6f), qk = norms[2] * fq * fk;
  float4 r1 = make_float4(0.f, 0.f, 0.f, 0.f), r2 = r1;
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int d = dg * RPT + i;
    if (d >= g.dkp) continue;
    const float gd = gs[d], kd = ks[d] * fk, qd = qs[d] * fq;
    S[i].x *= gd; S[i].y *= gd; S[i].z *= gd; S[i].w *= gd;
    r1.x = __builtin_fmaf(S[i].x, kd, r1.x); r1.y = __builtin_fmaf(S[i].y, kd, r1.y); r1.z = __builtin_fmaf(S[i].z, kd, r1.z); r1.w = __builtin_fmaf(S[i].w, kd, r1.w);
    r2.x = __builtin_fmaf(S[i].x, qd, r2.x); r2.y = __builtin_fmaf(S[i].y, qd, r2.y); r2.z = __builtin_fmaf(S[i].z, qd, r2.z); r2.w = __builtin_fmaf(S[i].w, qd, r2.w);
  }
#pragma unroll
  for (int m = VQ; m < 64; m *= 2) {
    r1.x += __shfl_xor(r1.x, m); r1.y += __shfl_xor(r1.y, m); r1.z += __shfl_xor(r1.z, m); r1.w += __shfl_xor(r1.w, m);
    r2.x += __shfl_xor(r2.x, m); r2.y += __shfl_xor(r2.y, m); r2.z += __shfl_xor(r2.z, m); r2.w += __shfl_xor(r2.w, m);
  }
  if (lane < VQ) {
    *reinterpret_cast<float4*>(&red[0][wave][vq * 4]) = r1;
    *reinterpret_cast<float4*>(&red[1][wave][vq * 4]) = r2;
  }
  __syncthreads();
  r1 = make_float4(0.f, 0.f, 0.f, 0.f);
  r2 = r1;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const float4 a = *reinterpret_cast<const float4*>(&red[0][w][vq * 4]), b = *reinterpret_cast<const float4*>(&red[1][w][vq * 4]);
    r1.x += a.x; r1.y += a.y; r1.z += a.z; r1.w += a.w;
    r2.x += b.x; r2.y += b.y; r2.z += b.z; r2.w += b.w;
  }
  if (!vin) r1 = r2 = make_float4(0.f, 0.f, 0.f, 0.f);
  float4 u = make_float4(0.f, 0.f, 0.f, 0.f);
  if (vin) u = make_float4(beta * (vs[vq * 4] - r1.x), beta * (vs[vq * 4 + 1] - r1.y), beta * (vs[vq * 4 + 2] - r1.z), beta * (vs[vq * 4 + 3] - r1.w));
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int d = dg * RPT + i;
    if (!vin || d >= g.dkp) continue;
    const float kd = ks[d] * fk;
    S[i].x = __builtin_fmaf(kd, u.x, S[i].x); S[i].y = __builtin_fmaf(kd, u.y, S[i].y); S[i].z = __builtin_fmaf(kd, u.z, S[i].z); S[i].w = __builtin_fmaf(kd, u.w, S[i].w);
    *reinterpret_cast<float4*>(S0 + (size_t)d * g.dvp) = S[i];
  }
  if (wave) return;                                  // (VQ <= 64 lanes of the first wave hold every column)
  float o[4] = {__builtin_fmaf(qk, u.x, r2.x), __builtin_fmaf(qk, u.y, r2.y), __builtin_fmaf(qk, u.z, r2.z), __builtin_fmaf(qk, u.w, r2.w)};
  float ss = lane < VQ ? (o[0] * o[0] + o[1] * o[1]) + (o[2] * o[2] + o[3] * o[3]) : 0.f;     // (padding columns are zero)
  ss = wave_sum(ss);
  const float f = 1.f / sqrtf(ss / (float)g.dv + in.eps);
  if (lane >= VQ) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int v = vq * 4 + i;
    if (v < g.dv) put1(y + (size_t)row * ldy + h * g.dv + v, o[i] * f * in.norm[v] * gate(in.z[(size_t)row * in.ldz + in.gate + h * g.dv + v]));
  }
}

// ---- prompts: the chunks of a ragged batch ------------------------------------------------------------------------------------
struct ChunkAt { AttnSeg sg; int t0, n; bool ok, last; };     // rows t0 .. + n of the segment
__device__ __forceinline__ ChunkAt chunk_at(const AttnSeg* segs, int nseg, int c) {
  for (int i = 0; i < nseg; ++i) {
    const AttnSeg sg = segs[i];
    if (sg.n < 2) continue;
    const int k = ceil_div(sg.n, kC);
    if (c < k) return ChunkAt{sg, c * kC, min(kC, sg.n - c * kC), true, c == k - 1};
    c -= k;
  }
  return ChunkAt{AttnSeg{0, 0, 0, 0}, 0, 0, false, false};
}

// The record of a chunk and head, in floats: -W, Q', K' as [dkp / 16] tiles of 16 x 16 (W, Q': token x channel; K': channel x token),
// exp L_end [dkp], T and P T [16][16], and [dvp / 16] tiles (token x column) of values that the scan replaces by outputs.  A head's
// records follow each other: the scan reads on without a gap.
struct Factors { float *w, *q, *k, *e, *t, *m, *v; };
__host__ __device__ __forceinline__ size_t record_floats(int dkp, int dvp) { return (size_t)49 * dkp + 512 + 16 * dvp; }
__device__ __forceinline__ Factors factors_at(float* base, size_t index, int dkp, int dvp) {
  float* p = base + index * record_floats(dkp, dvp);
  return Factors{p, p + 16 * dkp, p + 32 * dkp, p + 48 * dkp, p + 49 * dkp, p + 49 * dkp + 256, p + 49 * dkp + 512};
}

// where the input of a convolution `i` rows behind the segment's start lies (negative: ahead of it; ahead of the sequence: anywhere
// valid, conv_known is false).  Addresses are selected, not branched over: loads stay in flight together.
__device__ __forceinline__ const float* conv_at(const DeltaIn& in, const AttnSeg& sg, const float* ring, int taps, int C, int ch, int i) {
  const int p = max(sg.pos0 + i, 0) % taps;
  const float *a = in.proj + (size_t)(sg.row0 + max(i, 0)) * in.ldp + ch, *b = ring + (size_t)p * C + ch;
  return i >= 0 ? a : b;
}
__device__ __forceinline__ bool conv_known(const AttnSeg& sg, int i) { return sg.pos0 + i >= 0; }
__device__ __forceinline__ float conv_in(const DeltaIn& in, const AttnSeg& sg, const float* ring, int taps, int C, int ch, int i) {
  const float v = *conv_at(in, sg, ring, taps, C, ch, i);
  return conv_known(sg, i) ? v : 0.f;
}

// LDS written by some lanes of a wave, read by others of it
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
constexpr int kPairTiles = 36, kPairParts = 7;

// Bound by vector instructions (79 % of the time at 2600 a wave, 16 heads of 128, 2048 tokens) until phases were given shapes that need few of them: a thread
// takes whole columns of the convolution straight to LDS or memory, the decays' sums run over eight tokens a lane and its neighbour, eight lanes share a row's norm, and
// exponents are kept in powers of two: 1860 instructions, 53.1 -> 45.6 us, 151 MB at 3.3 TB/s.
template <int TAPS>
__global__ __launch_bounds__(256) void delta_factors_kernel(DeltaGeom g, DeltaIn in, const AttnSeg* __restrict__ segs, int nseg, int c0, float* __restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int pitch = g.dkp + 4;
  float *qs = sm, *ks = qs + kC * pitch, *Ls = ks + kC * pitch, *gs = Ls + kC * pitch, *red = gs;   // (red: in place of gs once that is used up)
  __shared__ float As[kC][kC + 1], Ps[kC][kC + 1], Ts[kC][kC + 1], Ms[kC][kC + 1], bs[kC];
  const ChunkAt at = chunk_at(segs, nseg, c0 + blockIdx.x);
  if (!at.ok) return;
  const int h = blockIdx.y, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = at.n, C = g.channels(), kvh = h / (g.H / g.G);
  const Factors F = factors_at(out, (size_t)h * gridDim.x + blockIdx.x, g.dkp, g.dvp);
  const float* ring = in.ring + (size_t)in.slots[at.sg.seq] * g.taps * C;
  const float* rows = in.proj + (size_t)(at.sg.row0 + at.t0) * in.ldp;
  const bool inside = at.t0 >= TAPS - 1 && n == kC;      // every input is a row of the batch: no clamps, no ring
  constexpr int kHalf = kC / 2, NA = TAPS > 0 ? kC + TAPS - 1 : 1, NB = TAPS > 0 ? kHalf + TAPS - 1 : 1, NW = TAPS > 0 ? TAPS : 1;
  // inputs of channel ch from TAPS - 1 rows ahead of the chunk's token t0 on
  auto request = [&](auto& x, float (&w)[NW], int ch, int t0) {
    constexpr int N = sizeof(x) / sizeof(float);
    if constexpr (TAPS > 0) {
      if (inside) {
        const unsigned char* from = reinterpret_cast<const unsigned char*>(rows - (size_t)(TAPS - 1) * in.ldp);
        uint32_t off = ((uint32_t)t0 * in.ldp + ch) * 4;
#pragma unroll
        for (int k = 0; k < N; ++k, off += (uint32_t)in.ldp * 4) x[k] = *reinterpret_cast<const float*>(from + off);
      } else {
#pragma unroll
        for (int k = 0; k < N; ++k) x[k] = conv_in(in, at.sg, ring, TAPS, C, ch, at.t0 + min(t0 + k - (TAPS - 1), n - 1));
      }
#pragma unroll
      for (int j = 0; j < TAPS; ++j) w[j] = in.conv[(uint32_t)j * C + ch];
    }
  };
  // the convolution of token t0 + t (0 behind the chunk's end and in padding channels)
  auto convolved = [&](const auto& x, const float (&w)[NW], int ch, int t0, int t, bool ok) {
    float a = 0.f;
    if constexpr (TAPS > 0) {
#pragma unroll
      for (int j = 0; j < TAPS; ++j) a = __builtin_fmaf(w[j], x[t + j], a);
    } else {
      for (int j = 0; j < g.taps; ++j)
        a = __builtin_fmaf(in.conv[(size_t)j * C + ch], conv_in(in, at.sg, ring, g.taps, C, ch, at.t0 + min(t0 + t, n - 1) - (g.taps - 1 - j)), a);
    }
    float r = silu(a);
    asm("" : "+v"(r));                                    // (a select, not a branch around every one)
    return ok && t0 + t < n ? r : 0.f;
  };
  // decays: a lane takes eight tokens of a channel, its neighbour the other eight
  constexpr float kLog2e = 1.4426950408889634f;
  const float decay = expf(in.a_log[h]) * kLog2e;
  const int zh = (tid & 1) * kHalf;
  const float* zr = in.z + (size_t)(at.sg.row0 + at.t0) * in.ldz + h * g.dk;
  float z0[kHalf];
  auto request_z = [&](int d) {
#pragma unroll
    for (int u = 0; u < kHalf; ++u) z0[u] = zr[(uint32_t)min(zh + u, n - 1) * in.ldz + min(d, g.dk - 1)];
  };
  request_z(tid >> 1);
  // convolutions: a thread takes a channel of q or k down the chunk and one of v down half of it, requested together
  for (int base = 0; base < 2 * max(g.dkp, g.dvp); base += 256) {
    const int i = base + tid;
    const int part = i >= g.dkp, d = min(i - part * g.dkp, g.dkp - 1), cha = (part * g.G + kvh) * g.dk + min(d, g.dk - 1);
    const int vh = i >= g.dvp ? kHalf : 0, vd = min(i - (vh ? g.dvp : 0), g.dvp - 1), chb = 2 * g.G * g.dk + h * g.dv + min(vd, g.dv - 1);
    float xa[NA], xb[NB], wa[NW], wb[NW];
    request(xa, wa, cha, 0);
    request(xb, wb, chb, vh);
    if (i < 2 * g.dkp) {
      float* dst = (part ? ks : qs) + d;
#pragma unroll
      for (int t = 0; t < kC; ++t) dst[t * pitch] = convolved(xa, wa, cha, 0, t, d < g.dk);
    }
    if (i < 2 * g.dvp) {
      float* dst = F.v + (vd >> 4) * 256 + vh * 16 + (vd & 15);
#pragma unroll
      for (int t = 0; t < kHalf; ++t) dst[t * 16] = convolved(xb, wb, chb, vh, t, vd < g.dv);
    }
  }
  // running sums of the decays' logarithms, the decays beside them
  for (int d = tid >> 1; d < g.dkp; d += 128) {
    if (d >= 128) request_z(d);
    const float zdt = in.dt[h * g.dk + min(d, g.dk - 1)];
    float lg[kHalf], sum = 0.f;
#pragma unroll
    for (int u = 0; u < kHalf; ++u) {
      lg[u] = d < g.dk && zh + u < n ? -decay * softplus(z0[u] + zdt) : 0.f;
      sum += lg[u];
    }
    const float other = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, sum), 0xB1, 0xf, 0xf, true));   // the neighbour's
    float L = zh ? other : 0.f;
#pragma unroll
    for (int u = 0; u < kHalf; ++u) {
      L += lg[u];
      Ls[(zh + u) * pitch + d] = L;
      gs[(zh + u) * pitch + d] = __builtin_amdgcn_exp2f(lg[u]);
    }
  }
  if (tid < kC) bs[tid] = tid < n ? sigmoid(rows[(size_t)tid * in.ldp + in.beta + h]) : 0.f;
  __syncthreads();
  {   // unit rows: eight lanes a row
    const int v = tid >> 3;
    float* r = (v < kC ? qs : ks) + (v & (kC - 1)) * pitch;
    float s = 0.f;
    for (int d = (tid & 7) * 4; d < g.dkp; d += 32) {
      const float4 x = *reinterpret_cast<const float4*>(r + d);
      s = __builtin_fmaf(x.x, x.x, s); s = __builtin_fmaf(x.y, x.y, s); s = __builtin_fmaf(x.z, x.z, s); s = __builtin_fmaf(x.w, x.w, s);
    }
    s = group_sum<8>(s);
    const float f = 1.f / sqrtf(s + 1e-6f) * (v < kC ? 1.f / sqrtf((float)g.dk) : 1.f);
    for (int d = (tid & 7) * 4; d < g.dkp; d += 32) {
      float4* p = reinterpret_cast<float4*>(r + d);
      const float4 x = *p;
      *p = make_float4(x.x * f, x.y * f, x.z * f, x.w * f);
    }
  }
  __syncthreads();
  // pairs: a thread takes one of the 36 tiles of tokens (2 I, 2 I + 1) x (2 J, 2 J + 1), J <= I, and every seventh group of four channels
  float a[4] = {0.f, 0.f, 0.f, 0.f}, p[4] = {0.f, 0.f, 0.f, 0.f};        // (i0,j0) (i0,j1) (i1,j0) (i1,j1)
  const int part = tid / kPairTiles, tl = tid - part * kPairTiles;
  if (part < kPairParts) {
    int I = 0;
#pragma unroll
    for (int k = 1; k < 8; ++k) I += tl >= k * (k + 1) / 2 ? 1 : 0;
    const int J = tl - I * (I + 1) / 2, i0 = 2 * I, j0 = 2 * J;
    const bool diag = I == J;
    for (int d = part * 4; d < g.dkp; d += 4 * kPairParts) {
      const float4 ki0 = *reinterpret_cast<const float4*>(ks + i0 * pitch + d), ki1 = *reinterpret_cast<const float4*>(ks + (i0 + 1) * pitch + d);
      const float4 qi0 = *reinterpret_cast<const float4*>(qs + i0 * pitch + d), qi1 = *reinterpret_cast<const float4*>(qs + (i0 + 1) * pitch + d);
      const float4 kj0 = *reinterpret_cast<const float4*>(ks + j0 * pitch + d), kj1 = *reinterpret_cast<const float4*>(ks + (j0 + 1) * pitch + d);
      const float4 Li = *reinterpret_cast<const float4*>(Ls + i0 * pitch + d), Lj = *reinterpret_cast<const float4*>(Ls + (j0 + 1) * pitch + d);
      const float4 gi = *reinterpret_cast<const float4*>(gs + (i0 + 1) * pitch + d), gj = *reinterpret_cast<const float4*>(gs + (j0 + 1) * pitch + d);
      auto one = [&](float k0, float k1, float q0, float q1, float c0, float c1, float li, float lj, float g1, float h1) {
        const float e = __builtin_amdgcn_exp2f(li - lj);   // (diagonal tiles: the entry above the diagonal, left out below)
        const float e11 = diag ? 1.f : e * g1, e00 = diag ? 1.f : e * h1;
        const float x00 = c0 * e00, x01 = c1 * e, x10 = x00 * g1, x11 = c1 * e11;
        a[0] = __builtin_fmaf(k0, x00, a[0]); a[1] = __builtin_fmaf(k0, x01, a[1]); a[2] = __builtin_fmaf(k1, x10, a[2]); a[3] = __builtin_fmaf(k1, x11, a[3]);
        p[0] = __builtin_fmaf(q0, x00, p[0]); p[1] = __builtin_fmaf(q0, x01, p[1]); p[2] = __builtin_fmaf(q1, x10, p[2]); p[3] = __builtin_fmaf(q1, x11, p[3]);
      };
      one(ki0.x, ki1.x, qi0.x, qi1.x, kj0.x, kj1.x, Li.x, Lj.x, gi.x, gj.x);
      one(ki0.y, ki1.y, qi0.y, qi1.y, kj0.y, kj1.y, Li.y, Lj.y, gi.y, gj.y);
      one(ki0.z, ki1.z, qi0.z, qi1.z, kj0.z, kj1.z, Li.z, Lj.z, gi.z, gj.z);
      one(ki0.w, ki1.w, qi0.w, qi1.w, kj0.w, kj1.w, Li.w, Lj.w, gi.w, gj.w);
    }
  }
  __syncthreads();
  if (part < kPairParts) {
    float4* r = reinterpret_cast<float4*>(red + tid * 8);
    r[0] = make_float4(a[0], a[1], a[2], a[3]);
    r[1] = make_float4(p[0], p[1], p[2], p[3]);
  }
  // k exp L and q exp L in place of k and q, K' out: a thread takes eight tokens of a channel
  for (int u = tid; u < 2 * g.dkp; u += 256) {
    const int d = u < g.dkp ? u : u - g.dkp, t0 = u < g.dkp ? 0 : 8;
    const float end = Ls[(kC - 1) * pitch + d];
    float o[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int r = (t0 + t) * pitch + d;
      const float L = Ls[r], e = __builtin_amdgcn_exp2f(L), k = ks[r];
      o[t] = k * __builtin_amdgcn_exp2f(end - L);
      ks[r] = k * e;
      qs[r] *= e;
    }
    float* kt = F.k + (d >> 4) * 256 + (d & 15) * 16 + t0;
    *reinterpret_cast<float4*>(kt) = make_float4(o[0], o[1], o[2], o[3]);
    *reinterpret_cast<float4*>(kt + 4) = make_float4(o[4], o[5], o[6], o[7]);
    if (t0 == 0) F.e[d] = __builtin_amdgcn_exp2f(end);
  }
  __syncthreads();
  {
    const int i = tid >> 4, j = tid & 15, I = i >> 1, J = j >> 1, at8 = (I * (I + 1) / 2 + J) * 8 + (i & 1) * 2 + (j & 1);
    float av = 0.f, pv = 0.f;
    if (j <= i) {
#pragma unroll
      for (int w = 0; w < kPairParts; ++w) { av += red[w * kPairTiles * 8 + at8]; pv += red[w * kPairTiles * 8 + at8 + 4]; }
    }
    As[i][j] = j < i ? av * bs[i] : 0.f;
    Ps[i][j] = j <= i ? pv : 0.f;
    Ts[i][j] = 0.f;
  }
  __syncthreads();
  if (wave == 0) {   // X = (I + A)^-1: the two diagonal blocks by forward substitution, a lane per column; X21 = -X22 A21 X11
    if (lane < kC) {
      const int b8 = lane & 8, j = lane & 7;
      float x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float v = i == j ? 1.f : 0.f;
#pragma unroll
        for (int m = 0; m < i; ++m) v = __builtin_fmaf(-As[b8 + i][b8 + m], x[m], v);
        x[i] = v;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) Ts[b8 + i][b8 + j] = x[i];
    }
    wave_order();
    const int i = lane >> 3, j = lane & 7;
    float y = 0.f;
#pragma unroll
    for (int m = 0; m < 8; ++m) y = __builtin_fmaf(As[8 + i][m], Ts[m][j], y);
    Ms[i][j] = y;
    wave_order();
    y = 0.f;
#pragma unroll
    for (int m = 0; m < 8; ++m) y = __builtin_fmaf(-Ts[8 + i][8 + m], Ms[m][j], y);
    wave_order();
    Ts[8 + i][j] = y;
  }
  __syncthreads();
  if (tid < kC * kC) Ts[tid >> 4][tid & 15] *= bs[tid & 15];
  __syncthreads();
  {
    const int i = tid >> 4, j = tid & 15;
    float m = 0.f;
#pragma unroll
    for (int k = 0; k < kC; ++k) m = __builtin_fmaf(Ps[i][k], Ts[k][j], m);
    Ms[i][j] = m;
    F.t[tid] = Ts[i][j];
    F.m[tid] = m;
  }
  __syncthreads();
  const int g4 = lane >> 4, c = lane & 15;
  for (int t = wave; t < g.dkp / 16; t += 4) {
    f32x4_t w = {0.f, 0.f, 0.f, 0.f}, q = w;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float b = ks[(4 * s + g4) * pitch + 16 * t + c];
      w = __builtin_amdgcn_mfma_f32_16x16x4f32(Ts[c][4 * s + g4], b, w, 0, 0, 0);
      q = __builtin_amdgcn_mfma_f32_16x16x4f32(Ms[c][4 * s + g4], b, q, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 4 * g4 + r;
      F.w[t * 256 + i * 16 + c] = -w[r];
      F.q[t * 256 + i * 16 + c] = qs[i * pitch + 16 * t + c] - q[r];
    }
  }
}

// Keys of more than 128 numbers.  One work-group per (head, 16 value columns, segment): the chunks of the segment in order.  A wave holds NT 16-channel tiles of the
// state as MFMA accumulators, which are the B operands of the next chunk's products as they stand; the partial sums of u and
// o over the channels meet in LDS, once per chunk.
template <int NT>
__global__ __launch_bounds__(256) void delta_scan_kernel(DeltaGeom g, float* __restrict__ state, const int32_t* __restrict__ slots,
                                                         const AttnSeg* __restrict__ segs, int c0, int nchunks, int nvt, float* __restrict__ records) {
  __shared__ f32x4_t ps[2][2][4][64];
  int id = blockIdx.x, h, vt;
  if (g.H % 8 == 0) {        // the column blocks of a head on one XCD: they read the same factors
    const int k = id >> 3;
    h = (id & 7) + 8 * (k / nvt);
    vt = k % nvt;
  } else {
    h = id / nvt;
    vt = id % nvt;
  }
  const int si = blockIdx.y;
  const AttnSeg sg = segs[si];
  if (sg.n < 2) return;
  int first = 0;             // the segment's first chunk among all
  for (int i = 0; i < si; ++i) first += segs[i].n < 2 ? 0 : ceil_div(segs[i].n, kC);
  const int k0 = max(c0 - first, 0), k1 = min(c0 + nchunks - first, ceil_div(sg.n, kC));
  if (k0 >= k1) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, g4 = lane >> 4, c = lane & 15, tiles = g.dkp / 16;
  float* S0 = state + ((size_t)slots[sg.seq] * g.H + h) * g.dkp * g.dvp + vt * 16 + c;
  f32x4_t S[NT];
  // Factors and values of the next kAhead chunks are in flight.  Addresses: a uniform part that moves from chunk to chunk and lane
  // offsets (bytes) that do not.
  constexpr int kAhead = 2;
  struct Frag { f32x4_t w[NT], q[NT], k[NT], e[NT]; float t, m, x; };
  uint32_t off[NT], eoff[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int tile = wave * NT + t, tl = min(tile, tiles - 1);            // (past the last tile: S stays zero)
    off[t] = (tl * 256 + c * 16 + 4 * g4) * 4;
    eoff[t] = (tl * 16 + 4 * g4) * 4;
#pragma unroll
    for (int r = 0; r < 4; ++r) S[t][r] = sg.pos0 + k0 > 0 && tile < tiles ? S0[(size_t)(tile * 16 + 4 * g4 + r) * g.dvp] : 0.f;
  }
  const uint32_t toff = (c * 16 + 4 * wave + g4) * 4, xoff = ((4 * wave + g4) * 16 + c) * 4, ooff = ((4 * g4 + wave) * 16 + c) * 4;
  auto at = [](float* base, uint32_t bytes) { return reinterpret_cast<unsigned char*>(base) + bytes; };
  auto record = [&](int k) { return factors_at(records, (size_t)h * nchunks + (first + k - c0), g.dkp, g.dvp); };
  auto load_w = [&](const Factors& F, Frag& f, int t) { f.w[t] = *reinterpret_cast<const f32x4_t*>(at(F.w, off[t])); };
  auto load_q = [&](const Factors& F, Frag& f, int t) { f.q[t] = *reinterpret_cast<const f32x4_t*>(at(F.q, off[t])); };
  auto load_k = [&](const Factors& F, Frag& f, int t) { f.k[t] = *reinterpret_cast<const f32x4_t*>(at(F.k, off[t])); };
  auto load_e = [&](const Factors& F, Frag& f, int t) { f.e[t] = *reinterpret_cast<const f32x4_t*>(at(F.e, eoff[t])); };
  auto load_rest = [&](const Factors& F, Frag& f, int i) {
    if (i == 0) f.t = *reinterpret_cast<const float*>(at(F.t, toff));
    if (i == 1) f.m = *reinterpret_cast<const float*>(at(F.m, toff));
    if (i == 2) f.x = *reinterpret_cast<const float*>(at(F.v + vt * 256, xoff));
  };
  auto load = [&](int k, Frag& f) {
    const Factors F = record(k);
#pragma unroll
    for (int t = 0; t < NT; ++t) { load_w(F, f, t); load_q(F, f, t); load_k(F, f, t); load_e(F, f, t); }
#pragma unroll
    for (int i = 0; i < 3; ++i) load_rest(F, f, i);
  };
  auto meet = [] {      // one barrier a chunk, for LDS alone: the loads of later chunks stay in flight across it
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto emit = [&](int k, int b) {      // a chunk's output in place of its values: its partial sums lie in ps[b][1]
    const float* po = reinterpret_cast<const float*>(&ps[b][1][0][0]);
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) s += po[(w * 64 + lane) * 4 + wave];
    *reinterpret_cast<float*>(at(record(k).v + vt * 256, ooff)) = s;
  };
  f32x4_t ov = {0.f, 0.f, 0.f, 0.f};
  // u's partial sums go out first; o's products and the scaling of S run while they do.  o's own meet at the next chunk's barrier.
  // A CU takes a wave's 16-byte loads in at one per 16 clocks: they are dealt out between the products, each as soon as what it
  // replaces is used up (K' and exp L_end of the chunk before behind the first products).
  auto pin = [] { __builtin_amdgcn_sched_barrier(0x6); };       // (ALU instructions may cross)
  auto step = [&](int k, Frag& f, Frag& before, bool more, bool more_before) {
    const int b = k & 1;
    const Factors Fn = record(k + kAhead), Fb = record(k - 1 + kAhead);
    f32x4_t u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        u = __builtin_amdgcn_mfma_f32_16x16x4f32(f.w[t][r], S[t][r], u, 0, 0, 0);
        if (r & 1) {
          pin();
          if (more_before) { if (r == 1) load_k(Fb, before, t); else load_e(Fb, before, t); }
          pin();
        }
      }
    }
    u = __builtin_amdgcn_mfma_f32_16x16x4f32(f.t, f.x, u, 0, 0, 0);
    ps[b][1][wave][lane] = ov;
    ps[b][0][wave][lane] = u;
    pin();
    ov = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
      for (int r = 0; r < 4; ++r) ov = __builtin_amdgcn_mfma_f32_16x16x4f32(f.q[t][r], S[t][r], ov, 0, 0, 0);
      pin();
      if (more) load_w(Fn, f, t);
      pin();
    }
    ov = __builtin_amdgcn_mfma_f32_16x16x4f32(f.m, f.x, ov, 0, 0, 0);
    f32x4_t Sg[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) Sg[t] = f32x4_t{S[t][0] * f.e[t][0], S[t][1] * f.e[t][1], S[t][2] * f.e[t][2], S[t][3] * f.e[t][3]};
    meet();
    u = ps[b][0][0][lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      const f32x4_t a = ps[b][0][w][lane];
      u[0] += a[0]; u[1] += a[1]; u[2] += a[2]; u[3] += a[3];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
      for (int t = 0; t < NT; ++t)     // (a tile past the last one stays zero)
        Sg[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wave * NT + t < tiles ? f.k[t][r] : 0.f, u[r], Sg[t], 0, 0, 0);
      pin();
      if (more) {
        if (r < NT) load_q(Fn, f, r);
        if (r < 3) load_rest(Fn, f, r);
      }
      pin();
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) S[t] = Sg[t];
    if (k > k0) emit(k - 1, b);
  };
  Frag f[kAhead];
#pragma unroll
  for (int i = 0; i < kAhead; ++i) load(min(k0 + i, k1 - 1), f[i]);
  int k = k0;
  for (; k + 2 * kAhead <= k1; k += kAhead) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) step(k + i, f[i], f[(i + kAhead - 1) % kAhead], true, i > 0 || k > k0);
  }
  // up to 2 kAhead - 1 chunks are left
  const bool was = k > k0;
  for (int j = 0; j < 2; ++j) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int n = k + j * kAhead + i;
      if (n < k1) step(n, f[i], f[(i + kAhead - 1) % kAhead], n + kAhead < k1, (n > k || was) && n - 1 + kAhead < k1);
    }
  }
  ps[k1 & 1][1][wave][lane] = ov;
  __syncthreads();
  emit(k1 - 1, k1 & 1);
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (wave * NT + t < tiles) S0[(size_t)((wave * NT + t) * 16 + 4 * g4 + r) * g.dvp] = S[t][r];
}

// The same for up to two tiles of channels a wave (keys of up to 128), two chunks to a barrier.  A chunk's chain is 26 matrix products of 32 cycles a wave,
// then the meeting of the partial sums (write, barrier, read, add) with the matrix core idle: 0.84 us of which 0.39 are products (2048 tokens of 16 heads,
// 108 us; half the chip's CUs have no work-group, and a head's state cannot be split further).  The second chunk's u needs the first one's state
// S1 = e1 S + K1' u1, so with W2 e1 in place of W2 its product with S joins the first chunk's, and what is missing is (-W2 K1') u1, a 16 x 16 matrix
// that does not depend on the state: it is made one pair ahead, while the partial sums of u come out of LDS.  One meeting and 64 products per
// pair: 1.46 us, 94 us.  Two pairs of chunks are in registers (248: a bound of two waves a SIMD keeps the compiler from moving some to the other file and back, 99 -> 96 us); a load of the pair after the next is issued as soon as what it replaces is used up.
// (Its own set of registers for a third pair, or the first chunk's o behind the barrier: 115 and 98 us.)
constexpr int kOutside = 0x7fff0000;      // beyond any buffer of records
template <typename F, int... I> __device__ __forceinline__ void each_of(std::integer_sequence<int, I...>, F&& f) { (f(std::integral_constant<int, I>()), ...); }
template <int N, typename F> __device__ __forceinline__ void each(F&& f) { each_of(std::make_integer_sequence<int, N>(), f); }

// The 16 columns vt of a head over n chunks from `base` on.  REPLY (the second part of a segment, delta_scan_split_kernel): columns of the identity in place of a
// state and no values; what they answer goes to `replies`, their last state is the product of the chunks' transitions.
using PairParts = f32x4_t[5][4][64];       // o of the pair before (two chunks), G, u1, what u2 has without G u1
template <int NT, bool REPLY, typename Load, typename Store>
__device__ __forceinline__ void delta_scan_pairs(PairParts* ps, const DeltaGeom& g, float* base, int n, int vt, float* replies, Load&& load_state, Store&& store_state) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, g4 = lane >> 4, c = lane & 15, tiles = g.dkp / 16;
  const int pairs = n / 4 * 2;                   // pairs of chunks, an even number of them; up to three chunks by themselves
  struct Chunk { f32x4_t w[NT], q[NT], k[NT], e[NT]; float t, m, x; };
  struct Pair { Chunk a, b; };
  f32x4_t kt[NT];            // K' of the next pair's first chunk, with a token per lane
  f32x4_t S[NT];
  // The records of this segment's chunks as a buffer: a load is one instruction (lane offsets that do not change, a scalar one per chunk), and tiles
  // past the last one lie outside of it, so that they read as zero and their part of S stays zero.
  const size_t rec = record_floats(g.dkp, g.dvp) * sizeof(float);
  const auto buf = __builtin_amdgcn_make_buffer_rsrc(base, 0, (int)(n * rec), 0x00020000);
  const int reply = 16 * g.dkp * (int)sizeof(float);
  const auto rbuf = __builtin_amdgcn_make_buffer_rsrc(replies, 0, REPLY ? n * reply : 0, 0x00020000);
  const int region = 16 * g.dkp * (int)sizeof(float);
  int woff[NT], qoff[NT], koff[NT], eoff[NT], ktoff[NT];
  bool live[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int tile = wave * NT + t, in_tile = (tile * 256 + c * 16 + 4 * g4) * 4;
    live[t] = tile < tiles;
    woff[t] = live[t] ? in_tile : kOutside;
    qoff[t] = live[t] ? region + in_tile : kOutside;
    koff[t] = live[t] ? 2 * region + in_tile : kOutside;
    ktoff[t] = live[t] ? 2 * region + (tile * 256 + 4 * g4 * 16 + c) * 4 : kOutside;
    eoff[t] = live[t] ? 3 * region + (tile * 16 + 4 * g4) * 4 : kOutside;
#pragma unroll
    for (int r = 0; r < 4; ++r) S[t][r] = live[t] ? load_state(tile * 16 + 4 * g4 + r, vt * 16 + c) : 0.f;
  }
  const int rest = 49 * g.dkp * (int)sizeof(float), toff = rest + (c * 16 + 4 * wave + g4) * 4, values = rest + 2048 + vt * 1024;
  const int xoff = values + ((4 * wave + g4) * 16 + c) * 4, ooff = values + ((4 * g4 + wave) * 16 + c) * 4;
  auto record = [&](int k) { return min(k, n - 1) * (int)rec; };      // (past the last chunk: its own factors again, not used)
  auto load4 = [&](int at, int from) { return __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(buf, at, from, 0)); };
  auto load1 = [&](int at, int from) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(buf, at, from, 0)); };
  auto load_w = [&](int F, Chunk& f, int t) { f.w[t] = load4(woff[t], F); };
  auto load_q = [&](int F, Chunk& f, int t) { f.q[t] = load4(qoff[t], F); };
  auto load_k = [&](int F, Chunk& f, int t) { f.k[t] = load4(koff[t], F); };
  auto load_e = [&](int F, Chunk& f, int t) { f.e[t] = load4(eoff[t], F); };
  auto load_t = [&](int F, Chunk& f) { if constexpr (!REPLY) f.t = load1(toff, F); };
  auto load_m = [&](int F, Chunk& f) { if constexpr (!REPLY) f.m = load1(toff + 1024, F); };
  auto load_x = [&](int F, Chunk& f) { if constexpr (!REPLY) f.x = load1(xoff, F); };
  auto load_kt = [&](int F, int t) {
#pragma unroll
    for (int r = 0; r < 4; ++r) kt[t][r] = load1(ktoff[t] + r * 64, F);
  };
  auto load_pair = [&](int p, Pair& f) {
    const int A = record(2 * p), B = record(2 * p + 1);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      load_w(A, f.a, t); load_w(B, f.b, t); load_e(A, f.a, t); load_q(A, f.a, t); load_k(A, f.a, t); load_e(B, f.b, t); load_k(B, f.b, t); load_q(B, f.b, t);
    }
    load_t(A, f.a); load_x(A, f.a); load_m(A, f.a);
    load_t(B, f.b); load_x(B, f.b); load_m(B, f.b);
  };
  auto meet = [] {      // LDS alone: the loads of later chunks stay in flight across the barrier
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto pin = [] { __builtin_amdgcn_sched_barrier(0x6); };       // (ALU instructions may cross)
  struct Parts { f32x4_t v[4]; __device__ __forceinline__ f32x4_t sum() const { return f32x4_t{v[0][0] + v[1][0] + v[2][0] + v[3][0], v[0][1] + v[1][1] + v[2][1] + v[3][1], v[0][2] + v[1][2] + v[2][2] + v[3][2], v[0][3] + v[1][3] + v[2][3] + v[3][3]}; } };
  auto parts = [&](const f32x4_t (&p)[4][64]) { return Parts{{p[0][lane], p[1][lane], p[2][lane], p[3][lane]}}; };
  auto out_parts = [&](const f32x4_t (&p)[4][64]) {      // this thread's number of a chunk's output
    const float* po = reinterpret_cast<const float*>(&p[0][0]) + lane * 4 + wave;
    return f32x4_t{po[0], po[256], po[512], po[768]};
  };
  auto all4 = [](f32x4_t v) { return v[0] + v[1] + v[2] + v[3]; };
  const int roff = (vt * 256 + (4 * g4 + wave) * 16 + c) * 4;
  auto put_out = [&](int k, float v) {
    if constexpr (REPLY) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), rbuf, roff, __builtin_amdgcn_readfirstlane(k * reply), 0);
    else __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), buf, ooff, __builtin_amdgcn_readfirstlane(record(k)), 0);      // in place of the chunk's values
  };
  // (REPLY: no values, so no products with them)
  auto with_values = [&](float m, float x, f32x4_t& acc) { if constexpr (!REPLY) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(m, x, acc, 0, 0, 0); };
  auto coupling = [&](const Chunk& second, auto&& between) {      // this wave's part of (-W2 K1')^T: what it leaves in a lane is the A operand of G u1
    f32x4_t gt = {0.f, 0.f, 0.f, 0.f};
    each<4 * NT>([&](auto i) {
      constexpr int t = decltype(i)::value / 4, r = decltype(i)::value % 4;
      gt = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[t][r], second.w[t][r], gt, 0, 0, 0);
      between(i);
    });
    return gt;
  };
  f32x4_t o1 = {0.f, 0.f, 0.f, 0.f}, o2 = o1, gt = o1;
  Pair f[2];
  auto step = [&](int p, Pair& now, Pair& next) {
    const int b = p & 1, A = record(2 * p + 4), B = record(2 * p + 5), Bn = record(2 * p + 3);
    const float xb = now.b.x;
    ps[b][0][wave][lane] = o1;
    ps[b][1][wave][lane] = o2;
    ps[b][2][wave][lane] = gt;
    f32x4_t u1 = {0.f, 0.f, 0.f, 0.f}, u2 = u1, Sg[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) now.b.w[t][r] *= now.a.e[t][r];
    each<4 * NT>([&](auto i) {
      constexpr int I = decltype(i)::value, t = I / 4, r = I % 4;
      u1 = __builtin_amdgcn_mfma_f32_16x16x4f32(now.a.w[t][r], S[t][r], u1, 0, 0, 0);
      u2 = __builtin_amdgcn_mfma_f32_16x16x4f32(now.b.w[t][r], S[t][r], u2, 0, 0, 0);
      pin();
      if (r == 0) load_q(Bn, next.b, t);       // (what the step before used up last)
      if (r == 3) { load_w(B, now.b, t); load_w(A, now.a, t); }
      pin();
    });
    with_values(now.a.t, now.a.x, u1);
    with_values(now.b.t, now.b.x, u2);
    ps[b][3][wave][lane] = u1;
    ps[b][4][wave][lane] = u2;
    pin();
    o1 = f32x4_t{0.f, 0.f, 0.f, 0.f};
    each<4 * NT>([&](auto i) {
      constexpr int I = decltype(i)::value, t = I / 4, r = I % 4;
      o1 = __builtin_amdgcn_mfma_f32_16x16x4f32(now.a.q[t][r], S[t][r], o1, 0, 0, 0);
      pin();
      if (I == 0) load_m(Bn, next.b);
      if (I == 1) load_t(A, now.a);
      if (I == 2) load_t(B, now.b);
      if (r == 3) load_q(A, now.a, t);
      pin();
    });
    with_values(now.a.m, now.a.x, o1);
#pragma unroll
    for (int t = 0; t < NT; ++t) Sg[t] = f32x4_t{S[t][0] * now.a.e[t][0], S[t][1] * now.a.e[t][1], S[t][2] * now.a.e[t][2], S[t][3] * now.a.e[t][3]};
    meet();
    const Parts p1 = parts(ps[b][3]), pg = parts(ps[b][2]), p2 = parts(ps[b][4]);
    const f32x4_t q1 = out_parts(ps[b][0]), q2 = out_parts(ps[b][1]);
    __builtin_amdgcn_sched_barrier(0);         // (the reads leave together, and the products of the coupling run while they are on their way)
    gt = coupling(next.b, [&](auto i) {
      constexpr int I = decltype(i)::value;
      pin();
      if (I == 0) load_x(B, now.b);
      if (I == 1) load_m(A, now.a);
      if (I == 2) load_x(A, now.a);
      if (I % 4 == 3) load_e(A, now.a, I / 4);
      pin();
    });
    const float out1 = all4(q1), out2 = all4(q2);
    u1 = p1.sum();
    const f32x4_t G = pg.sum();
    u2 = p2.sum();
    each<4>([&](auto i) {
      constexpr int r = decltype(i)::value;
#pragma unroll
      for (int t = 0; t < NT; ++t) Sg[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.a.k[t][r], u1[r], Sg[t], 0, 0, 0);
      u2 = __builtin_amdgcn_mfma_f32_16x16x4f32(G[r], u1[r], u2, 0, 0, 0);
      pin();
      if (r < NT) load_kt(A, r);
      pin();
    });
#pragma unroll
    for (int t = 0; t < NT; ++t) S[t] = f32x4_t{Sg[t][0] * now.b.e[t][0], Sg[t][1] * now.b.e[t][1], Sg[t][2] * now.b.e[t][2], Sg[t][3] * now.b.e[t][3]};
    each<4>([&](auto i) {
      constexpr int r = decltype(i)::value;
#pragma unroll
      for (int t = 0; t < NT; ++t) S[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.b.k[t][r], u2[r], S[t], 0, 0, 0);
      pin();
      if (r < NT) load_k(A, now.a, r);
      else if (r < 2 * NT) load_e(B, now.b, r - NT);
      pin();
    });
    o2 = f32x4_t{0.f, 0.f, 0.f, 0.f};
    each<4 * NT>([&](auto i) {
      constexpr int I = decltype(i)::value, t = I / 4, r = I % 4;
      o2 = __builtin_amdgcn_mfma_f32_16x16x4f32(now.b.q[t][r], Sg[t][r], o2, 0, 0, 0);
      pin();
      if (r == 1) load_k(B, now.b, t);
      pin();
    });
    with_values(now.b.m, xb, o2);
    if (p > 0) {
      put_out(2 * p - 2, out1);
      put_out(2 * p - 1, out2);
    }
  };
  load_pair(0, f[0]);
  load_pair(1, f[1]);
  if (pairs > 0) {
#pragma unroll
    for (int t = 0; t < NT; ++t) load_kt(record(0), t);
    gt = coupling(f[0].b, [](auto) {});
#pragma unroll
    for (int t = 0; t < NT; ++t) load_kt(record(2), t);
    int p = 0;
    do {
      step(p, f[0], f[1]);
      step(p + 1, f[1], f[0]);
      p += 2;
    } while (p < pairs);
    ps[0][0][wave][lane] = o1;
    ps[0][1][wave][lane] = o2;
    __syncthreads();
    put_out(2 * pairs - 2, all4(out_parts(ps[0][0])));
    put_out(2 * pairs - 1, all4(out_parts(ps[0][1])));
  }
  auto single = [&](int k, int b, const Chunk& f) {
    f32x4_t u = {0.f, 0.f, 0.f, 0.f}, o = u;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        u = __builtin_amdgcn_mfma_f32_16x16x4f32(f.w[t][r], S[t][r], u, 0, 0, 0);
        o = __builtin_amdgcn_mfma_f32_16x16x4f32(f.q[t][r], S[t][r], o, 0, 0, 0);
      }
    with_values(f.t, f.x, u);
    with_values(f.m, f.x, o);
    ps[b][3][wave][lane] = u;
    ps[b][4][wave][lane] = o;
    __syncthreads();
    u = parts(ps[b][3]).sum();
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      S[t] = f32x4_t{S[t][0] * f.e[t][0], S[t][1] * f.e[t][1], S[t][2] * f.e[t][2], S[t][3] * f.e[t][3]};
#pragma unroll
      for (int r = 0; r < 4; ++r) S[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.k[t][r], u[r], S[t], 0, 0, 0);
    }
    put_out(k, all4(out_parts(ps[b][4])));
  };
  if (2 * pairs < n) single(2 * pairs, 0, f[0].a);
  if (2 * pairs + 1 < n) single(2 * pairs + 1, 1, f[0].b);
  if (2 * pairs + 2 < n) single(2 * pairs + 2, 0, f[1].a);
#pragma unroll
  for (int t = 0; t < NT; ++t)
    if (live[t]) store_state(wave * NT + t, S[t]);
}

// the head and block of value columns of work-group id among H nvt: the column blocks of a head on one XCD, they read the same factors
__device__ __forceinline__ void scan_columns(const DeltaGeom& g, int id, int nvt, int& h, int& vt) {
  if (g.H % 8 == 0) {
    const int k = id >> 3;
    h = (id & 7) + 8 * (k / nvt);
    vt = k % nvt;
  } else {
    h = id / nvt;
    vt = id % nvt;
  }
}

template <int NT>
__global__ __launch_bounds__(256, 2) void delta_scan_pairs_kernel(DeltaGeom g, float* __restrict__ state, const int32_t* __restrict__ slots,
                                                               const AttnSeg* __restrict__ segs, int c0, int nchunks, int nvt, float* __restrict__ records) {
  __shared__ PairParts ps[2];
  int h, vt;
  scan_columns(g, blockIdx.x, nvt, h, vt);
  const int si = blockIdx.y;
  const AttnSeg sg = segs[si];
  if (sg.n < 2) return;
  int first = 0;             // the segment's first chunk among all
  for (int i = 0; i < si; ++i) first += segs[i].n < 2 ? 0 : ceil_div(segs[i].n, kC);
  const int k0 = max(c0 - first, 0), k1 = min(c0 + nchunks - first, ceil_div(sg.n, kC));
  if (k0 >= k1) return;
  const int lane = threadIdx.x & 63;
  float* S0 = state + ((size_t)slots[sg.seq] * g.H + h) * g.dkp * g.dvp;
  const bool begun = sg.pos0 + k0 > 0;
  delta_scan_pairs<NT, false>(ps, g, records + ((size_t)h * nchunks + (first + k0 - c0)) * record_floats(g.dkp, g.dvp), k1 - k0, vt, nullptr,
                          [&](int d, int v) { return begun ? S0[(size_t)d * g.dvp + v] : 0.f; },
                          [&](int tile, const f32x4_t& s) {
#pragma unroll
                            for (int r = 0; r < 4; ++r) S0[(size_t)(tile * 16 + 4 * (lane >> 4) + r) * g.dvp + vt * 16 + (lane & 15)] = s[r];
                          });
}

// One long segment on a chip whose CUs the kernel above leaves half idle: its chunks in two parts at the same time.  The transition of a chunk is linear in the state:
// with S1 the state between the parts, an output of the second one is the output from a state of zeros plus q^T (the product of the transitions so far) S1, and that
// row of replies is what the same recurrence makes of the columns of the identity.  So the second part has two work-groups for 16 columns, which share a CU and take 2.7 us
// a pair between them (fp32 matrix products leave no room for vector instructions beside them: 32 cycles and 5 - 9 for each of those), and it is the shorter one; the order of the
// work-groups puts both on the CUs that the first part leaves.  delta_out_kernel adds replies S1 and makes the last state.  Everything stays fp32.
// 16 heads of 128, 2048 tokens, us: scan 98 -> 66, output norm 15.5 -> 21 (31 at first, a call 2142 -> 2020; 3000 tokens 2993 -> 2768).  The cut is for parts that share CUs (16 heads of 128 take 256 of them); where each
// has its own, one half would be the even one.  All kernels of a launch of 8 heads there: 2048 tokens 139 -> 116, 4096 251 -> 200; 2 heads 119 -> 96, 215 -> 160.
// Behind the records: [chunk][16 dkp] replies a head, those of the first part unused: there the states, S1 as fragments, the second part's own (L) and its transition (P).
// From 48 chunks on (16 dkp numbers each: room for the three states in those of the first part): below, the joining costs what the parts save.  us of all kernels, one scan -> two parts,
// 640, 768, 1008 tokens: 16 heads of 128 69.5 -> 70.1, 75.8 -> 74.7, 91.5 -> 84.1; 12 heads 64.4 -> 67.1, 73.8 -> 72.4, 86.0 -> 80.8; 2 heads 53.3 -> 53.3, 59.2 -> 58.6, 71.4 -> 64.7;
// 20 heads of 96 66.7 -> 68.4, 74.4 -> 73.1, 91.3 -> 86.7; 32 of 64 61.4 -> 56.5, 64.8 -> 63.4, 81.0 -> 73.0.  8 layers of 16 heads of 128, 1100 tokens: 1445 -> 1377 a call.
constexpr int kSplitChunks = 48;
__host__ __device__ __forceinline__ int split_first(int n) { return (n * 41 + 127) / 256 * 4; }     // chunks of the first part: 0.64 of them, whole turns of the loop
struct SplitMem { float *replies, *s1, *l, *p; };
__host__ __device__ __forceinline__ SplitMem split_mem(float* records, const DeltaGeom& g, int n, int h) {
  float* r = records + (size_t)g.H * n * record_floats(g.dkp, g.dvp) + (size_t)h * n * 16 * g.dkp;
  return SplitMem{r, r, r + g.dkp * g.dvp, r + 2 * g.dkp * g.dvp};
}
template <int NT>
__global__ __launch_bounds__(256, 2) void delta_scan_split_kernel(DeltaGeom g, const float* __restrict__ state, const int32_t* __restrict__ slots,
                                                                  const AttnSeg* __restrict__ segs, int c0, int n, int nvt, float* __restrict__ records) {
  __shared__ PairParts ps[2];
  const int cols = g.H * nvt, slot = (int)blockIdx.x / cols, part = slot == 0 ? 1 : slot == 1 ? 0 : 2, first = split_first(n), lane = threadIdx.x & 63, g4 = lane >> 4, c = lane & 15;
  int h, vt;
  scan_columns(g, (int)blockIdx.x - slot * cols, nvt, h, vt);
  const AttnSeg sg = segs[0];
  const SplitMem m = split_mem(records, g, n, h);
  float* base = records + (size_t)h * n * record_floats(g.dkp, g.dvp);
  auto put = [&](float* to, int tile, const f32x4_t& s) {
#pragma unroll
    for (int r = 0; r < 4; ++r) to[(size_t)(tile * 16 + 4 * g4 + r) * g.dvp + vt * 16 + c] = s[r];
  };
  if (part < 2) {
    const float* S0 = state + ((size_t)slots[sg.seq] * g.H + h) * g.dkp * g.dvp;
    const bool begun = part == 0 && sg.pos0 + c0 > 0;
    const int at = part ? first : 0;
    delta_scan_pairs<NT, false>(ps, g, base + (size_t)at * record_floats(g.dkp, g.dvp), part ? n - first : first, vt, nullptr,
                                [&](int d, int v) { return begun ? S0[(size_t)d * g.dvp + v] : 0.f; },
                                [&](int tile, const f32x4_t& s) {
                                  if (part) put(m.l, tile, s);
                                  else *reinterpret_cast<f32x4_t*>(m.s1 + ((vt * (g.dkp / 16) + tile) * 64 + lane) * 4) = s;
                                });
  } else {
    delta_scan_pairs<NT, true>(ps, g, base + (size_t)first * record_floats(g.dkp, g.dvp), n - first, vt, m.replies + (size_t)first * 16 * g.dkp,
                               [&](int d, int v) { return d == v ? 1.f : 0.f; }, [&](int tile, const f32x4_t& s) { put(m.p, tile, s); });
  }
}
// the state behind a segment in two parts: L + P S1, a wave per 16 x 16 tile
__device__ __forceinline__ void delta_join(const DeltaGeom& g, float* __restrict__ state, int slot, int n, float* __restrict__ records, int at) {
  const int tiles = g.dkp / 16, lane = threadIdx.x & 63, g4 = lane >> 4, c = lane & 15, h = at / (tiles * tiles), rt = at / tiles % tiles, ct = at % tiles;
  if (h >= g.H) return;
  const SplitMem m = split_mem(records, g, n, h);
  const float* l = m.l + (size_t)(rt * 16 + 4 * g4) * g.dvp + ct * 16 + c;
  f32x4_t a[4] = {};             // (short chains, added pairwise: the join adds little to the rounding of its parts)
  for (int t = 0; t < tiles; ++t) {
    const f32x4_t p = *reinterpret_cast<const f32x4_t*>(m.p + (size_t)(rt * 16 + c) * g.dvp + t * 16 + 4 * g4), s1 = *reinterpret_cast<const f32x4_t*>(m.s1 + ((ct * tiles + t) * 64 + lane) * 4);
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[r], s1[r], a[r], 0, 0, 0);
  }
  float* to = state + ((size_t)slot * g.H + h) * g.dkp * g.dvp + (size_t)(rt * 16 + 4 * g4) * g.dvp + ct * 16 + c;
#pragma unroll
  for (int r = 0; r < 4; ++r) to[(size_t)r * g.dvp] = l[(size_t)r * g.dvp] + ((a[0][r] + a[1][r]) + (a[2][r] + a[3][r]));
}

// Norm and gate: a wave per head and chunk, a lane four columns of every value tile of one token, all of them requested together; the work-groups of a
// segment's last chunk renew its ring.  WIDE: rows of z and y in 16 and 8 bytes.  Bound by memory: 16 heads of 128, 2048 tokens, 42 MB in 16.3 us (19.5 with
// a lane per column and eight tokens after each other).
// SPLIT: a segment in two parts (delta_scan_split_kernel) -- chunks of the second one get their replies times S1, four of a head in a work-group, so that S1's
// fragments come out of memory once for four waves; the second part takes longer and comes first, then the first one's chunks, four a work-group whatever the number of
// heads, then those that make the last state.  Bound by the round of requests and the fp32 products behind it: everything that a wave needs from memory is asked for in front of the
// barrier, S1 goes to LDS without registers, and where every tile is there no branch stands around a product.  16 heads of 128, 2048 tokens: 31.2 -> 21.2 us a launch; eight chunks to one S1
// 24.7 (half as many CUs multiply; 28.8 with registers for two such work-groups a CU, which spill).
constexpr int kOutWaves = 4;
__device__ __forceinline__ void lds_dma16(const void* g, void* l) {      // 16 bytes a lane, to l + 16 lane
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g, (__attribute__((address_space(3))) void*)l, 16, 0, 0);
}
__host__ __device__ __forceinline__ int split_groups(int n, int H) { return ceil_div(n - split_first(n), kOutWaves) * H; }     // work-groups of the second part
__host__ __device__ __forceinline__ int first_groups(int n, int H) { return ceil_div(split_first(n) * H, kOutWaves); }         // and of the first
template <typename T, int NT, bool WIDE, bool SPLIT = false>
__global__ __launch_bounds__(SPLIT ? kOutWaves * 64 : 256, SPLIT ? 2 : 1) void delta_out_kernel(DeltaGeom g, DeltaIn in, const AttnSeg* __restrict__ segs, int nseg, int c0, int n,
                                                                                                 float* __restrict__ records, T* __restrict__ y, int ldy) {
  const int wave = SPLIT ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x >> 6, lane = threadIdx.x & 63;
  int chunk = blockIdx.x, h = blockIdx.y * 4 + wave;
  __shared__ f32x4_t s1[SPLIT ? NT * NT * 64 : 1];      // the state between the parts, as fragments: one round of requests
  f32x4_t rep[SPLIT ? NT : 1];                           // the chunk's replies
  bool second = false;
  if constexpr (SPLIT) {
    const int first = split_first(n), seconds = split_groups(n, g.H), firsts = first_groups(n, g.H), b = blockIdx.x;
    if (b >= seconds + firsts) {
      delta_join(g, in.state, in.slots[segs[0].seq], n, records, (b - seconds - firsts) * kOutWaves + wave);
      return;
    }
    second = b < seconds;
    const int unit = (b - seconds) * kOutWaves + wave;
    chunk = second ? first + b / g.H * kOutWaves + wave : unit / g.H;
    h = second ? b % g.H : unit % g.H;
    if (!second && chunk >= first) return;
    if (second) {
      const SplitMem m = split_mem(records, g, n, h);
      const float* replies = m.replies + (size_t)min(chunk, n - 1) * 16 * g.dkp + (lane & 15) * 16 + (lane >> 4) * 4;
      const f32x4_t* from = reinterpret_cast<const f32x4_t*>(m.s1);
      const int all = g.dkp * g.dvp / 4;
#pragma unroll
      for (int i = 0; i < NT * NT / kOutWaves; ++i)
        lds_dma16(from + min(i * kOutWaves * 64 + (int)threadIdx.x, all - 1), s1 + i * kOutWaves * 64 + wave * 64);
#pragma unroll
      for (int d = 0; d < NT; ++d) rep[d] = *reinterpret_cast<const f32x4_t*>(replies + min(d, g.dkp / 16 - 1) * 256);
    }
  }
  const int known = min(chunk, n - 1);
  const ChunkAt at = chunk_at(segs, nseg, c0 + known);
  if (!SPLIT && (!at.ok || chunk >= n)) return;
  const int t = lane >> 2, q = (lane & 3) * 4, tiles = g.dvp / 16;
  const size_t row = at.sg.row0 + at.t0 + min(t, at.n - 1);
  f32x4_t x[NT], z[NT];
  if (h < g.H) {
    const float *src = factors_at(records, (size_t)h * n + known, g.dkp, g.dvp).v, *zr = in.z + row * in.ldz + in.gate + h * g.dv;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int tile = min(i, tiles - 1), v = tile * 16 + q;
      x[i] = *reinterpret_cast<const f32x4_t*>(src + tile * 256 + lane * 4);
      if constexpr (WIDE) z[i] = *reinterpret_cast<const f32x4_t*>(zr + min(v, g.dv - 4));
      else z[i] = f32x4_t{zr[min(v, g.dv - 1)], zr[min(v + 1, g.dv - 1)], zr[min(v + 2, g.dv - 1)], zr[min(v + 3, g.dv - 1)]};
    }
  }
  if constexpr (SPLIT) {
    if (second) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
    if (chunk >= n) return;
  }
  if (h < g.H) {
    if constexpr (SPLIT) {
      if (second) {     // the products leave a column's quad of token (lane & 15) in lane >> 4: four lanes trade places
        auto products = [&](auto whole) {      // (every tile there: no branch around a product)
#pragma unroll
          for (int i = 0; i < NT; ++i) {
            f32x4_t add[2] = {};
#pragma unroll
            for (int d = 0; d < NT; ++d) {
              if (!decltype(whole)::value && max(i, d) >= tiles) continue;
              const f32x4_t f = s1[(i * (decltype(whole)::value ? NT : tiles) + d) * 64 + lane];
#pragma unroll
              for (int r = 0; r < 4; ++r) add[d & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[r], rep[d][r], add[d & 1], 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) x[i][r] += __shfl(add[0][r] + add[1][r], (lane & 3) * 16 + t);
          }
        };
        if (tiles == NT) products(std::true_type());
        else products(std::false_type());
      }
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) ss = __builtin_fmaf(x[i][r], i * 16 + q + r < g.dv ? x[i][r] : 0.f, ss);
    const float f = 1.f / sqrtf(group_sum<4>(ss) / (float)g.dv + in.eps);
    if (t < at.n) {
      T* to = y + row * ldy + h * g.dv;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int v = i * 16 + q;
        if (v >= g.dv) break;
        float o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = x[i][r] * f * in.norm[min(v + r, g.dv - 1)] * gate(z[i][r]);
        if constexpr (WIDE) {
          put4(to + v, o);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (v + r < g.dv) put1(to + v + r, o[r]);
        }
      }
    }
  }
  if (!at.last) return;
  const int C = g.channels();
  float* ring = in.ring + (size_t)in.slots[at.sg.seq] * g.taps * C;
  // (SPLIT: the last chunk is of the second part, and a wave a head has it, not ceil(H / 4) work-groups)
  for (int ch = SPLIT ? h * 64 + lane : blockIdx.y * 256 + threadIdx.x; ch < C; ch += SPLIT ? g.H * 64 : gridDim.y * 256)
    for (int i = max(0, at.sg.n - g.taps); i < at.sg.n; ++i)
      ring[(size_t)((at.sg.pos0 + i) % g.taps) * C + ch] = in.proj[(size_t)(at.sg.row0 + i) * in.ldp + ch];
}

int check_in(const DeltaGeom& g, const DeltaIn& in) {
  MI_CHECK(delta_supported(g), "delta rule: heads must be a multiple of the key heads, head sizes 1 .. 256, 1 .. 16 taps");
  MI_CHECK(g.dkp % 16 == 0 && g.dkp >= g.dk && g.dkp < g.dk + 16 && g.dvp % 16 == 0 && g.dvp >= g.dv && g.dvp < g.dv + 16, "delta rule: padding");
  MI_CHECK(in.proj && in.z && in.conv && in.a_log && in.dt && in.norm && in.state && in.ring && in.slots && in.pos, "delta rule: null argument");
  MI_CHECK(in.beta >= g.channels() && in.ldp >= in.beta + g.H && in.gate >= g.H * g.dk && in.ldz >= in.gate + g.H * g.dv, "delta rule: columns");
  return MI_OK;
}

}  // namespace

bool delta_supported(const DeltaGeom& g) {
  return g.H >= 1 && g.G >= 1 && g.H % g.G == 0 && g.dk >= 1 && g.dk <= 256 && g.dv >= 1 && g.dv <= 256 && g.taps >= 1 && g.taps <= 16;
}
// whether a segment may go in two parts (delta_scan_split_kernel): states as wide as they are high, keys the paired scan takes, CUs for both parts (32 heads of 128 have none to spare, and no replies)
static bool split_fits(const DeltaGeom& g, int num_cu) { return g.dkp == g.dvp && g.dkp <= 128 && 2 * g.H * (g.dvp / 16) <= num_cu; }
size_t delta_chunk_floats(const DeltaGeom& g) {
  int num_cu = 0;
  return (size_t)g.H * (record_floats(g.dkp, g.dvp) + (device_num_cu(&num_cu) != MI_OK || split_fits(g, num_cu) ? 16 * g.dkp : 0));
}

int launch_delta_token(const DeltaGeom& g, const DeltaIn& in, int rows, const AttnSeg* segs, void* y, int ldy, bool f32, hipStream_t s) {
  int rc = check_in(g, in);
  if (rc != MI_OK) return rc;
  MI_CHECK(rows >= 1 && rows <= 65535 && y && ldy >= g.H * g.dv, "delta rule: rows");
  const dim3 grid(g.H, rows);
  const int vq = g.dvp <= 16 ? 4 : g.dvp <= 32 ? 8 : g.dvp <= 64 ? 16 : g.dvp <= 128 ? 32 : 64, need = ceil_div(g.dkp, kTokenThreads / vq);
#define MI_DT(VQ, RPT) \
  if (f32) hipLaunchKernelGGL((delta_token_kernel<float, VQ, RPT>), grid, dim3(kTokenThreads), 0, s, g, in, segs, (float*)y, ldy); \
  else hipLaunchKernelGGL((delta_token_kernel<uint16_t, VQ, RPT>), grid, dim3(kTokenThreads), 0, s, g, in, segs, (uint16_t*)y, ldy)
  if (vq == 4) { if (need <= 1) { MI_DT(4, 1); } else { MI_DT(4, 2); } }
  else if (vq == 8) { if (need <= 1) { MI_DT(8, 1); } else if (need <= 2) { MI_DT(8, 2); } else { MI_DT(8, 4); } }
  else if (vq == 16) { if (need <= 2) { MI_DT(16, 2); } else if (need <= 4) { MI_DT(16, 4); } else { MI_DT(16, 8); } }
  else if (vq == 32) { if (need <= 4) { MI_DT(32, 4); } else if (need <= 8) { MI_DT(32, 8); } else { MI_DT(32, 16); } }
  else { if (need <= 8) { MI_DT(64, 8); } else if (need <= 16) { MI_DT(64, 16); } else { MI_DT(64, 32); } }
#undef MI_DT
  MI_HIP(hipGetLastError());
  return MI_OK;
}

int launch_delta_prompt(const DeltaGeom& g, const DeltaIn& in, const AttnSeg* sd, const AttnSeg* sh, int nseg, float* records, int max_chunks,
                        void* y, int ldy, bool f32, hipStream_t s) {
  int rc = check_in(g, in);
  if (rc != MI_OK) return rc;
  MI_CHECK(nseg >= 1 && nseg <= 65535 && records && max_chunks >= 1 && y && ldy >= g.H * g.dv, "delta rule: segments / workspace");
  int chunks = 0;
  for (int i = 0; i < nseg; ++i) chunks += sh[i].n < 2 ? 0 : ceil_div(sh[i].n, kC);
  const int nvt = g.dvp / 16, nt = ceil_div(g.dkp / 16, 4);
  int num_cu = 0;
  if (device_num_cu(&num_cu) != MI_OK) return MI_EHIP;
  const size_t lds = (size_t)(3 * kC * (g.dkp + 4) + std::max(kC * (g.dkp + 4), kPairParts * kPairTiles * 8)) * sizeof(float);
  for (int c0 = 0; c0 < chunks; c0 += max_chunks) {
    const int n = std::min(max_chunks, chunks - c0);
    const bool split = nseg == 1 && split_fits(g, num_cu) && n >= kSplitChunks;
    const int joins = ceil_div(g.H * nvt * nvt, kOutWaves);       // work-groups for the last state
    const dim3 gf(n, g.H), gs(g.H * nvt, nseg), go(split ? split_groups(n, g.H) + first_groups(n, g.H) + joins : n, split ? 1 : ceil_div(g.H, 4));
#define MI_DF(TAPS) { \
    if (lds > 48 * 1024) { rc = ensure_dynamic_lds(reinterpret_cast<const void*>(delta_factors_kernel<TAPS>), (int)lds); if (rc != MI_OK) return rc; } \
    hipLaunchKernelGGL((delta_factors_kernel<TAPS>), gf, dim3(256), lds, s, g, in, sd, nseg, c0, records); }
#define MI_DS(NT) hipLaunchKernelGGL((delta_scan_kernel<NT>), gs, dim3(256), 0, s, g, in.state, in.slots, sd, c0, n, nvt, records)
    switch (g.taps) {
      case 1: MI_DF(1); break;
      case 2: MI_DF(2); break;
      case 3: MI_DF(3); break;
      case 4: MI_DF(4); break;
      default: MI_DF(0);
    }
#undef MI_DF
#define MI_DP(NT) hipLaunchKernelGGL((delta_scan_pairs_kernel<NT>), gs, dim3(256), 0, s, g, in.state, in.slots, sd, c0, n, nvt, records)
    if (split && nt == 1) hipLaunchKernelGGL((delta_scan_split_kernel<1>), dim3(3 * g.H * nvt), dim3(256), 0, s, g, in.state, in.slots, sd, c0, n, nvt, records);
    else if (split) hipLaunchKernelGGL((delta_scan_split_kernel<2>), dim3(3 * g.H * nvt), dim3(256), 0, s, g, in.state, in.slots, sd, c0, n, nvt, records);
    else if (nt == 1) MI_DP(1);
    else if (nt == 2) MI_DP(2);
    else if (nt == 3) MI_DS(3);      // (three sets of two chunks do not fit the registers)
    else MI_DS(4);
#undef MI_DP
#undef MI_DS
#define MI_DO(NT, ...) \
    if (f32) hipLaunchKernelGGL((delta_out_kernel<float, NT, __VA_ARGS__>), go, dim3(split ? kOutWaves * 64 : 256), 0, s, g, in, sd, nseg, c0, n, records, (float*)y, ldy); \
    else hipLaunchKernelGGL((delta_out_kernel<uint16_t, NT, __VA_ARGS__>), go, dim3(split ? kOutWaves * 64 : 256), 0, s, g, in, sd, nseg, c0, n, records, (uint16_t*)y, ldy)
    const bool wide = g.dv % 4 == 0 && in.ldz % 4 == 0 && in.gate % 4 == 0 && ldy % 4 == 0 && reinterpret_cast<uintptr_t>(in.z) % 16 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0;
    if (split) { if (wide && g.dv <= 64) { MI_DO(4, true, true); } else if (wide) { MI_DO(8, true, true); } else { MI_DO(8, false, true); } }
    else if (!wide) { MI_DO(16, false); } else if (g.dv <= 64) { MI_DO(4, true); } else if (g.dv <= 128) { MI_DO(8, true); } else { MI_DO(16, true); }
#undef MI_DO
    MI_HIP(hipGetLastError());
  }
  return MI_OK;
}

}  // namespace mi
