// Sequence mixers that carry a matrix state per head: the gated delta rule with a decay per key channel, and retention
// (one fixed decay per head).  State, decays, step sizes, unit norms and the products with the state are float32.
//
// One token (decode): k_delta_step / k_retention_step.  A workgroup owns one head and 32 of its value columns; the
// state's columns are independent but for the vectors every workgroup of a head makes for itself (convolution, unit
// norms, decay), so no workgroup waits for another.
//
// A portion of a prompt: two launches.  The first (k_delta_prep / k_retention_prep, a workgroup per head and chunk of
// 16 tokens, all chunks at once) writes what a chunk does to the state as dense operands; the second (k_chunk_scan, a
// workgroup per head and 16 value columns) walks over the chunks with the state in the accumulators of the float32
// matrix instruction.  With b_t the step size, G_t the product of the decays up to token t of the chunk and S the state
// ahead of it:
//   A[t,s] = sum_d k_t k_s G_t / G_s  (s < t),   T = (I + diag(b) A)^-1,   U = T diag(b) (V - (G k) S)
//   o_t = S^T (G_t q_t) + sum_{s <= t} B[t,s] u_s,   B[t,s] = sum_d q_t k_s G_t / G_s
//   S  <- G_last S + sum_s (G_last / G_s) k_s u_s^T
// (retention: U = V).  Decays are kept as logarithms and every quotient is the exponential of a difference that is <= 0,
// so a decay as strong as float32 can hold neither overflows nor loses the tokens behind it.
#include "recurrent_common.h"
#include <algorithm>

namespace adamah {


typedef AdamahDeltaSpec DSpec;
typedef AdamahRetentionSpec RSpec;

// sums over a workgroup of NW waves of up to three values at once; sh: 3 NW floats
template <int NW>
__device__ __forceinline__ void block_add3(float& a, float& b, float& c, float* sh) {
  a = wave_add(a); b = wave_add(b); c = wave_add(c);
  const uint32_t w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63u) == 0) { sh[w] = a; sh[NW + w] = b; sh[2 * NW + w] = c; }
  __syncthreads();
  a = b = c = 0.f;
#pragma unroll
  for (int i = 0; i < NW; i++) { a += sh[i]; b += sh[NW + i]; c += sh[2 * NW + i]; }
}

// dot product of a bf16 matrix row of kp columns (a multiple of 64, zeros at the end) with a float32 vector of as many,
// by 8 neighbouring lanes (all get the sum)
__device__ __forceinline__ float dot8(const bf16_t* w, const float* x, uint32_t kp, uint32_t sub) {
  float a = 0.f;
  for (uint32_t c = sub * 8u; c < kp; c += 64u) {
    const uint4 p = *(const uint4*)(w + c);
    const uint32_t u[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
    for (int i = 0; i < 4; i++) { a = fmaf(bf_lo(u[i]), x[c + 2 * i], a); a = fmaf(bf_hi(u[i]), x[c + 2 * i + 1], a); }
  }
  a += __shfl_xor(a, 1, 64); a += __shfl_xor(a, 2, 64); a += __shfl_xor(a, 4, 64);
  return a;
}

struct LowRank { uint32_t w, k, k_stride, src, src_stride, out, out_stride; };   // what a step needs of a linear spec

// the same for a row held in registers: NC 16-byte words of it per lane (zeros beyond the row), x as long
template <int NC>
__device__ __forceinline__ float dot8_regs(const uint4 (&w)[NC], const float* x, uint32_t kp, uint32_t sub) {
  float a = 0.f;
#pragma unroll
  for (int n = 0; n < NC; n++) {
    const uint32_t c = sub * 8u + 64u * n, u[4] = {w[n].x, w[n].y, w[n].z, w[n].w};
    if (c >= kp) break;
#pragma unroll
    for (int i = 0; i < 4; i++) { a = fmaf(bf_lo(u[i]), x[c + 2 * i], a); a = fmaf(bf_hi(u[i]), x[c + 2 * i + 1], a); }
  }
  a += __shfl_xor(a, 1, 64); a += __shfl_xor(a, 2, 64); a += __shfl_xor(a, 4, 64);
  return a;
}

// One token of one sequence per blockIdx.z; DN: state rows a thread holds (dim <= 16 DN); TM >= taps.  Everything a
// workgroup reads is asked for at the start: the state, the convolution's inputs, the rows of the low-rank factors (in
// registers where their rank is at most 128).
//
// CW: value columns of a thread, VC of them beside each other in a workgroup.  With one, a head of 128 columns is four
// workgroups, each of which repeats the head's decay and convolution: latency decides, and more of them is better.  With
// four, one workgroup does the head: a quarter of the repeated work, and the state moves 16 bytes a lane.  The state's
// rows go to the same sums in the same order either way, so a result does not depend on the sequences beside it.
#define DSTEP 512u
template <int CW> struct alignas(4 * CW) Cols { float x[CW]; };
template <int DN, int TM, int CW>
__global__ void __launch_bounds__(DSTEP)
k_delta_step(const DSpec s, const LowRank da, const LowRank ga, float* act, const bf16_t* __restrict__ W, float* state, uint32_t seq0,
             uint32_t pos) {
  constexpr int NP = DN / 4 > 0 ? DN / 4 : 1;          // decay rows of 8 lanes: 64 a pass
  constexpr uint32_t NG = DSTEP / VC, NV = VC * CW;
  constexpr int NR = CW > 2 ? CW / 2 : 1;              // gate rows of 8 lanes: 64 a pass
  extern __shared__ float lds[];
  __shared__ float sh[3 * DSTEP / 64];
  __shared__ __align__(16) float red[2][NG][NV];
  __shared__ __align__(16) float vs[NV];
  const uint32_t D = s.dim, V = s.vdim, tid = threadIdx.x, h = blockIdx.x, v0 = blockIdx.y * NV, row = blockIdx.z;
  float *qs = lds, *ks = qs + D, *gs = ks + D, *la = gs + D, *lg = la + da.k_stride;
  const uint32_t n_ch = 2u * s.kv_heads * D + s.heads * V, rep = s.heads / s.kv_heads, kv = h / rep, sub = tid & 7u;
  const float* x = act + s.x + (uint64_t)row * s.x_stride;
  float* ring = state + (uint64_t)(seq0 + row) * s.seq_stride + s.conv_off;
  float* S = state + (uint64_t)(seq0 + row) * s.seq_stride + s.s_off + (uint64_t)h * D * V;
  const uint32_t qc = kv * D, kc = s.kv_heads * D + kv * D, vc = 2u * s.kv_heads * D + h * V;
  const uint32_t col = (tid & (VC - 1u)) * CW, dg = tid / VC, v = v0 + col;
  const bool small = da.k_stride <= 128u && ga.k_stride <= 128u;
  const uint32_t gt = DSTEP - 1u - tid;                // gate rows: the last threads
  Cols<CW> st[DN];
#pragma unroll
  for (int i = 0; i < DN; i++) {
    const uint32_t d = dg + NG * i;
    st[i] = {};
    if (pos != 0u && d < D && v < V) st[i] = *(const Cols<CW>*)(S + (uint64_t)d * V + v);
  }
  for (uint32_t i = tid; i < da.k_stride; i += DSTEP) la[i] = i < da.k ? act[da.src + (uint64_t)row * da.src_stride + i] : 0.f;
  for (uint32_t i = gt; i < ga.k_stride; i += DSTEP) lg[i] = i < ga.k ? act[ga.src + (uint64_t)row * ga.src_stride + i] : 0.f;
  uint4 wa[NP][2], wg[NR][2];
  float bias[NP];
#pragma unroll
  for (int i = 0; i < NP; i++) {
    const uint32_t r = h * D + min((tid >> 3) + 64u * i, D - 1u);
    bias[i] = act[s.dt_bias + r];
    if (small)
#pragma unroll
      for (int n = 0; n < 2; n++)
        wa[i][n] = sub * 8u + 64u * n < da.k_stride ? *(const uint4*)(W + da.w + (uint64_t)r * da.k_stride + sub * 8u + 64u * n) : make_uint4(0, 0, 0, 0);
  }
  const float a_log = act[s.a_log + h], step = x[s.x_b + h];
  const auto gate_row = [&](int i) { return h * V + min(v0 + (gt >> 3) + 64u * i, V - 1u); };
  if (small && gt < 8u * NV)
#pragma unroll
    for (int i = 0; i < NR; i++)
#pragma unroll
      for (int n = 0; n < 2; n++)
        wg[i][n] = (gt & 7u) * 8u + 64u * n < ga.k_stride ? *(const uint4*)(W + ga.w + (uint64_t)gate_row(i) * ga.k_stride + (gt & 7u) * 8u + 64u * n) : make_uint4(0, 0, 0, 0);
  float sq = 0.f, sk = 0.f, qk = 0.f;
  for (uint32_t i = tid; i < 2u * D; i += DSTEP) {
    const bool is_k = i >= D;
    const uint32_t d = is_k ? i - D : i;
    const float a = conv_silu_ring<TM>(x, ring, n_ch, (is_k ? kc : qc) + d, pos, act + (is_k ? s.ck : s.cq) + (uint64_t)(kv * D + d) * s.taps, s.taps);
    (is_k ? ks : qs)[d] = a;
    if (is_k) sk = fmaf(a, a, sk); else sq = fmaf(a, a, sq);
  }
  if (gt < NV && v0 + gt < V)
    vs[gt] = conv_silu_ring<TM>(x, ring, n_ch, vc + v0 + gt, pos, act + s.cv + (uint64_t)(h * V + v0 + gt) * s.taps, s.taps);
  const float ea = expf(a_log), beta = sigmoid_f(step);
  __syncthreads();
  for (uint32_t d = tid; d < D; d += DSTEP) qk = fmaf(qs[d], ks[d], qk);
  if (small) {
#pragma unroll
    for (int i = 0; i < NP; i++) {
      const uint32_t d = (tid >> 3) + 64u * i;
      const float a = dot8_regs<2>(wa[i], la, da.k_stride, sub);
      if (sub == 0 && d < D) gs[d] = expf(-ea * softplus_f(a + bias[i]));
    }
  } else {
    for (uint32_t d = tid >> 3; d < ((D + 63u) & ~63u); d += 64u) {      // whole waves take part in the dot products
      const uint32_t r = h * D + min(d, D - 1u);
      const float a = dot8(W + da.w + (uint64_t)r * da.k_stride, la, da.k_stride, sub);
      if (sub == 0 && d < D) gs[d] = expf(-ea * softplus_f(a + act[s.dt_bias + r]));
    }
  }
  if (gt < 8u * NV)
#pragma unroll
    for (int i = 0; i < NR; i++) {
      const uint32_t grow = gate_row(i);
      const float a = small ? dot8_regs<2>(wg[i], lg, ga.k_stride, gt & 7u) : dot8(W + ga.w + (uint64_t)grow * ga.k_stride, lg, ga.k_stride, gt & 7u);
      if ((gt & 7u) == 0 && v0 + (gt >> 3) + 64u * i < V) act[ga.out + (uint64_t)row * ga.out_stride + grow] = a;
    }
  block_add3<DSTEP / 64>(sq, sk, qk, sh);      // (its barriers also publish gs)
  const float iq = 1.0f / sqrtf(sq + 1e-6f) / sqrtf((float)D), ik = 1.0f / sqrtf(sk + 1e-6f);
  qk = qk * iq * ik;
  Cols<CW> pk = {}, pq = {};
#pragma unroll
  for (int i = 0; i < DN; i++) {
    const uint32_t d = dg + NG * i;
    if (d < D) {
      const float g = gs[d], k = ks[d], q = qs[d];
#pragma unroll
      for (int c = 0; c < CW; c++) {
        st[i].x[c] *= g;
        pk.x[c] = fmaf(st[i].x[c], k, pk.x[c]); pq.x[c] = fmaf(st[i].x[c], q, pq.x[c]);
      }
    }
  }
  *(Cols<CW>*)&red[0][dg][col] = pk; *(Cols<CW>*)&red[1][dg][col] = pq;
  __syncthreads();
  pk = {}; pq = {};
#pragma unroll CW == 1 ? 16 : 4
  for (int i = 0; i < (int)NG; i++) {
    const Cols<CW> a = *(const Cols<CW>*)&red[0][i][col], b = *(const Cols<CW>*)&red[1][i][col];
#pragma unroll
    for (int c = 0; c < CW; c++) { pk.x[c] += a.x[c]; pq.x[c] += b.x[c]; }
  }
  if (v < V) {
    float uk[CW];
#pragma unroll
    for (int c = 0; c < CW; c++) {
      const float u = beta * (vs[col + c] - pk.x[c] * ik);
      if (dg == 0) act[s.out + (uint64_t)row * s.out_stride + h * V + v + c] = fmaf(u, qk, pq.x[c] * iq);
      uk[c] = u * ik;
    }
#pragma unroll
    for (int i = 0; i < DN; i++) {
      const uint32_t d = dg + NG * i;
      if (d < D) {
        const float k = ks[d];
#pragma unroll
        for (int c = 0; c < CW; c++) st[i].x[c] = fmaf(k, uk[c], st[i].x[c]);
        *(Cols<CW>*)(S + (uint64_t)d * V + v) = st[i];
      }
    }
  }
  float* slot = ring + (uint64_t)(pos % s.taps) * n_ch;
  if (blockIdx.y == 0 && h % rep == 0)
    for (uint32_t d = tid; d < D; d += DSTEP) { slot[qc + d] = x[qc + d]; slot[kc + d] = x[kc + d]; }
  if (tid < NV && v0 + tid < V) slot[vc + v0 + tid] = x[vc + v0 + tid];
}

__device__ __forceinline__ float rotated(const float* x, const float* freq, uint32_t d, uint32_t dims, uint32_t p) {
  const uint32_t half = dims >> 1;
  if (d >= dims) return x[d];
  const uint32_t i = d < half ? d : d - half;
  float sn, cs;
  sincosf((float)p * freq[i], &sn, &cs);
  return d < half ? x[d] * cs - x[d + half] * sn : x[d] * cs + x[d - half] * sn;
}

template <int DN>
__global__ void __launch_bounds__(256)
k_retention_step(const RSpec s, float* act, float* state, uint32_t seq0, uint32_t pos) {
  extern __shared__ float lds[];
  __shared__ float sh[12];
  __shared__ float red[8][VC];
  const uint32_t D = s.dim, V = s.vdim, tid = threadIdx.x, h = blockIdx.x, v0 = blockIdx.y * VC, row = blockIdx.z;
  float *qs = lds, *ks = qs + D;
  const float* x = act + s.x + (uint64_t)row * s.x_stride;
  float* S = state + (uint64_t)(seq0 + row) * s.seq_stride + s.s_off + (uint64_t)h * D * V;
  const uint32_t col = tid & 31u, dg = tid >> 5, v = v0 + col;
  const float dec = act[s.decay + h], kscale = 1.0f / sqrtf((float)D);
  float st[DN];
#pragma unroll
  for (int i = 0; i < DN; i++) {
    const uint32_t d = dg + 8u * i;
    st[i] = (pos != 0u && d < D && v < V) ? S[(uint64_t)d * V + v] : 0.f;
  }
  const float vv = v < V ? x[s.x_v + h * V + v] : 0.f;
  float qk = 0.f, z0 = 0.f, z1 = 0.f;
  for (uint32_t d = tid; d < D; d += 256u) {
    qs[d] = rotated(x + s.x_q + h * D, act + s.freq, d, s.rot_dims, pos);
    ks[d] = rotated(x + s.x_k + h * D, act + s.freq, d, s.rot_dims, pos) * kscale;
    qk = fmaf(qs[d], ks[d], qk);
  }
  block_add3<4>(qk, z0, z1, sh);
  float pq = 0.f;
#pragma unroll
  for (int i = 0; i < DN; i++) {
    const uint32_t d = dg + 8u * i;
    if (d < D && v < V) {
      const float t = dec * st[i];
      pq = fmaf(t, qs[d], pq);
      S[(uint64_t)d * V + v] = fmaf(ks[d], vv, t);
    }
  }
  red[dg][col] = pq;
  __syncthreads();
  if (dg == 0 && v < V) {
    pq = 0.f;
#pragma unroll
    for (int i = 0; i < 8; i++) pq += red[i][col];
    act[s.out + (uint64_t)row * s.out_stride + h * V + v] = fmaf(vv, qk, pq);
  }
}

// ---- chunk operands -------------------------------------------------------------------------------------------------
// Block of one (head, chunk): W = T diag(b) (G k) [16][Dp], Q = G q [16][Dp], K^T [Dp][16], B [16][16], U0 [16][Vp], G_last [Dp].
struct ChunkDims { uint32_t Dp, Vp, n_chunks; };
__host__ __device__ inline uint32_t chunk_floats(uint32_t Dp, uint32_t Vp) { return 49u * Dp + 256u + 16u * Vp; }

// Columns of q and k (a thread each) run through their convolution in registers, then those of v and of the decay.
// Exponentials and LDS reads bound it; four workgroups a compute unit (by LDS) hide one another's barriers as long as a thread has
// at most 128 registers (2048 tokens in 32 heads of 128: 194 us with 201 registers, two workgroups; 143 with 69).
template <int TM>
__global__ void __launch_bounds__(256)
k_delta_prep(const DSpec s, uint32_t dec_out, uint32_t dec_stride, const float* __restrict__ act, const float* __restrict__ state,
             float* __restrict__ scratch, ChunkDims cd, uint32_t m, uint32_t seq0, uint32_t pos) {
  extern __shared__ float lds[];
  __shared__ __attribute__((aligned(16))) float A[CH][CH + 4], M[CH][CH + 4];
  __shared__ float beta[CH], iq[CH], ik[CH];
  const uint32_t D = s.dim, V = s.vdim, tid = threadIdx.x, c0 = blockIdx.x * CH, h = blockIdx.y, P = D + 1u;
  float *qs = lds, *ks = qs + CH * P, *G = ks + CH * P, *vs = G + CH * P;             // G: log2 of the running decay; vs [CH][Vp]
  const uint32_t n_ch = 2u * s.kv_heads * D + s.heads * V, kv = h / (s.heads / s.kv_heads);
  const uint32_t qc = kv * D, kc = s.kv_heads * D + kv * D, vc = 2u * s.kv_heads * D + h * V;
  const uint32_t sq = blockIdx.z;                            // sequence: rows sq m ..
  const float* x = act + s.x + (uint64_t)sq * m * s.x_stride;
  const float* ring = state + (uint64_t)(seq0 + sq) * s.seq_stride + s.conv_off;
  const float* dec = act + dec_out + (uint64_t)sq * m * dec_stride;
  float* out = scratch + (((uint64_t)sq * s.heads + h) * cd.n_chunks + blockIdx.x) * chunk_floats(cd.Dp, cd.Vp);
  float *oW = out, *oQ = oW + CH * cd.Dp, *oK = oQ + CH * cd.Dp, *oB = oK + CH * cd.Dp, *oU = oB + 256u, *oG = oU + CH * cd.Vp;
  for (uint32_t i = tid; i < 2u * D; i += 256u) {
    const bool is_k = i >= D;
    const uint32_t d = is_k ? i - D : i;
    float* to = (is_k ? ks : qs) + d;
    conv_silu_rows<TM>(x, s.x_stride, c0, m, ring, n_ch, (is_k ? kc : qc) + d, pos, act + (is_k ? s.ck : s.cq) + (uint64_t)(kv * D + d) * s.taps,
                       s.taps, [&](int t, float v) { to[t * P] = v; });
  }
  if (tid < CH) beta[tid] = c0 + tid < m ? sigmoid_f(x[(uint64_t)(c0 + tid) * s.x_stride + s.x_b + h]) : 0.f;
  const float ea = expf(act[s.a_log + h]);
  const uint32_t v_items = (V + 63u) & ~63u;                 // whole waves do one or the other
  for (uint32_t i = tid; i < v_items + D; i += 256u) {
    if (i < v_items) {
      if (i < V) conv_silu_rows<TM>(x, s.x_stride, c0, m, ring, n_ch, vc + i, pos, act + s.cv + (uint64_t)(h * V + i) * s.taps, s.taps,
                                    [&](int t, float v) { vs[t * cd.Vp + i] = v; });
    } else {
      const uint32_t d = i - v_items;
      const float bias = act[s.dt_bias + h * D + d];
      float z[CH];
#pragma unroll
      for (int t = 0; t < (int)CH; t++) z[t] = dec[(uint64_t)min(c0 + t, m - 1u) * dec_stride + h * D + d];
      const auto decay = [&](int t) { return fminf(ea * softplus_f(z[t] + bias), NO_MEMORY) * 1.44269504f; };
      if (m - c0 >= CH) {                                    // (as in conv_silu_rows)
#pragma unroll
        for (int t = 0; t < (int)CH; t++) z[t] = decay(t);
      } else {
#pragma unroll
        for (int t = 0; t < (int)CH; t++) if (c0 + t < m) z[t] = decay(t);
      }
      float lg = 0.f;
#pragma unroll
      for (int t = 0; t < (int)CH; t++) {
        lg -= c0 + t < m ? z[t] : 0.f;
        G[t * P + d] = lg;
      }
    }
  }
  __syncthreads();
  {                                                          // lengths of q and k: 8 threads a row, 32 rows
    const uint32_t rr = tid >> 3, sub = tid & 7u;
    const float* v = (rr < CH ? qs : ks) + (rr & (CH - 1u)) * P;
    float ss = 0.f;
    for (uint32_t d = sub; d < D; d += 8u) ss = fmaf(v[d], v[d], ss);
    ss += __shfl_xor(ss, 1, 64); ss += __shfl_xor(ss, 2, 64); ss += __shfl_xor(ss, 4, 64);
    if (sub == 0) (rr < CH ? iq : ik)[rr & (CH - 1u)] = 1.0f / sqrtf(ss + 1e-6f) / (rr < CH ? sqrtf((float)D) : 1.0f);
  }
  __syncthreads();
  {
    const uint32_t t = tid >> 4, r = tid & 15u;
    float a = 0.f, b = 0.f;
    if (r <= t) {
#pragma unroll 4
      for (uint32_t d = 0; d < D; d++) {
        const float e = __builtin_amdgcn_exp2f(G[t * P + d] - G[r * P + d]) * ks[r * P + d];
        a = fmaf(ks[t * P + d], e, a); b = fmaf(qs[t * P + d], e, b);
      }
    }
    A[t][r] = r < t ? a * ik[t] * ik[r] * beta[t] : 0.f;
    oB[place16(t, r)] = b * iq[t] * ik[r];
  }
  __syncthreads();
  if (tid < CH) {                                            // column tid of the inverse, forward substitution
    float y[CH];
#pragma unroll
    for (int t = 0; t < (int)CH; t++) {
      float a = (uint32_t)t == tid ? 1.f : 0.f;
#pragma unroll
      for (int r = 0; r < t; r++) a = fmaf(-A[t][r], y[r], a);
      y[t] = a;
      M[t][tid] = a * beta[tid];
    }
  }
  __syncthreads();
  for (uint32_t i = tid; i < 2u * cd.Dp + cd.Vp; i += 256u) {
    if (i < cd.Dp) {
      const uint32_t d = i;
      const bool in = d < D;
      const float gl = in ? G[15u * P + d] : 0.f;
      float qt[CH], kt[CH];
#pragma unroll
      for (int t = 0; t < (int)CH; t++) {
        const float lg = in ? G[t * P + d] : 0.f;
        qt[t] = in ? qs[t * P + d] * iq[t] * __builtin_amdgcn_exp2f(lg) : 0.f;
        kt[t] = in ? ks[t * P + d] * ik[t] * __builtin_amdgcn_exp2f(gl - lg) : 0.f;
      }
      store_rows(oQ, d, qt);
      store_cols(oK, d, kt);
      oG[d] = __builtin_amdgcn_exp2f(gl);
    } else {
      const bool is_u = i >= 2u * cd.Dp;
      const uint32_t d = is_u ? i - 2u * cd.Dp : i - cd.Dp;
      float y[CH];
#pragma unroll
      for (int t = 0; t < (int)CH; t++)
        y[t] = is_u ? (d < V ? vs[t * cd.Vp + d] : 0.f) : d < D ? ks[t * P + d] * ik[t] * __builtin_amdgcn_exp2f(G[t * P + d]) : 0.f;
      float o[CH];
#pragma unroll
      for (int t = 0; t < (int)CH; t++) {
        if (!(t & 3)) asm volatile("" ::: "memory");         // four rows of M at a time: all of them would take 136 registers
        float a = 0.f;
#pragma unroll
        for (int r = 0; r <= t; r++) a = fmaf(M[t][r], y[r], a);
        o[t] = a;
      }
      if (is_u) store_cols(oU, d, o); else store_rows(oW, d, o);
    }
  }
}

__global__ void __launch_bounds__(256)
k_retention_prep(const RSpec s, const float* __restrict__ act, float* __restrict__ scratch, ChunkDims cd, uint32_t m, uint32_t pos) {
  extern __shared__ float lds[];
  __shared__ float pw[CH + 1];
  const uint32_t D = s.dim, V = s.vdim, tid = threadIdx.x, c0 = blockIdx.x * CH, h = blockIdx.y, P = D + 1u, half = s.rot_dims >> 1;
  const uint32_t L = min(CH, m - c0);
  float *qs = lds, *ks = qs + CH * P, *cs = ks + CH * P, *sn = cs + CH * half;
  const float* x = act + s.x + (uint64_t)blockIdx.z * m * s.x_stride;          // z: the sequence
  float* out = scratch + (((uint64_t)blockIdx.z * s.heads + h) * cd.n_chunks + blockIdx.x) * chunk_floats(cd.Dp, cd.Vp);
  float *oQ = out + CH * cd.Dp, *oK = oQ + CH * cd.Dp, *oB = oK + CH * cd.Dp, *oU = oB + 256u, *oG = oU + CH * cd.Vp;
  const float kscale = 1.0f / sqrtf((float)D);
  if (tid == 0) {
    const float dec = act[s.decay + h];
    pw[0] = 1.f;
    for (uint32_t i = 1; i <= CH; i++) pw[i] = pw[i - 1] * dec;
  }
  for (uint32_t i = tid; i < 2u * D; i += 256u) {
    const bool is_k = i >= D;
    const uint32_t d = is_k ? i - D : i;
    const float* src = x + (is_k ? s.x_k : s.x_q) + h * D + d;
    float* to = (is_k ? ks : qs) + d;
    float v[CH];
#pragma unroll
    for (int t = 0; t < (int)CH; t++) v[t] = src[(uint64_t)min(c0 + t, m - 1u) * s.x_stride];      // (a load on every path)
#pragma unroll
    for (int t = 0; t < (int)CH; t++) to[t * P] = c0 + t >= m ? 0.f : is_k ? v[t] * kscale : v[t];
  }
  for (uint32_t i = tid; i < CH * half; i += 256u) {
    const uint32_t t = i / half, d = i - t * half;
    float a, b;
    sincosf((float)(pos + c0 + t) * act[s.freq + d], &a, &b);
    sn[i] = a; cs[i] = b;
  }
  for (uint32_t v = tid; v < cd.Vp; v += 256u) {
    float y[CH];
#pragma unroll
    for (int t = 0; t < (int)CH; t++) y[t] = x[(uint64_t)min(c0 + t, m - 1u) * s.x_stride + s.x_v + h * V + min(v, V - 1u)];
#pragma unroll
    for (int t = 0; t < (int)CH; t++) y[t] = c0 + t < m && v < V ? y[t] : 0.f;
    store_cols(oU, v, y);
  }
  __syncthreads();
  for (uint32_t i = tid; i < 2u * CH * half; i += 256u) {     // turn the pairs in place
    const bool is_k = i >= CH * half;
    const uint32_t j = is_k ? i - CH * half : i, t = j / half, d = j - t * half;
    float* r = (is_k ? ks : qs) + t * P;
    const float a = r[d], b = r[d + half];
    r[d] = a * cs[j] - b * sn[j];
    r[d + half] = b * cs[j] + a * sn[j];
  }
  __syncthreads();
  {
    const uint32_t t = tid >> 4, r = tid & 15u;
    float b = 0.f;
    if (r <= t) {
#pragma unroll 4
      for (uint32_t d = 0; d < D; d++) b = fmaf(qs[t * P + d], ks[r * P + d], b);
      b *= pw[t - r];
    }
    oB[place16(t, r)] = b;
  }
  for (uint32_t d = tid; d < cd.Dp; d += 256u) {
    float qt[CH], kt[CH];
#pragma unroll
    for (int t = 0; t < (int)CH; t++) {
      qt[t] = d < D ? qs[t * P + d] * pw[t + 1] : 0.f;
      kt[t] = (d < D && (uint32_t)t < L) ? ks[t * P + d] * pw[L - 1u - min((uint32_t)t, L - 1u)] : 0.f;
    }
    store_rows(oQ, d, qt);
    store_cols(oK, d, kt);
    oG[d] = pw[L];
  }
}

// ---- the walk over the chunks ---------------------------------------------------------------------------------------
// A serial chain, so what counts is a chunk's latency, or how much of it other workgroups hide (scan_form).  Four waves share the
// state rows (NT tiles of 16 each); a tile's accumulator holds rows 4 g + i of lane group g, which is also how instruction i wants its
// right operand when the left one is read as four consecutive columns per lane.  On their chain are only the products that the state
// needs (delta: W S, its sum through LDS, K u); Q S goes out while that sum is on its way.  A fifth wave adds up the four shares of
// Q S, adds B u from what they leave in LDS and stores: loads and stores share a counter, and a wave that does both waits
// for its stores.  2048 tokens in 32 heads of 128: outputs by the first of four waves, ahead of its part of the state, 136 us,
// retention 97; so 114 and 79.
// In every form one product behind the other by wave, the waves' parts as (0 + 1) + (2 + 3), B u behind that sum in order: a router behind
// these sums turns another order into another choice of experts (with two sums a wave and a quarter of B u in each share 111 and 79
// us, and 3e-2 in a mixture's logits).
struct ScanArgs {
  uint32_t heads, dim, vdim, out, out_stride, s_off, m, pos;
  ChunkDims cd;
  uint32_t kv_heads, taps, conv_off, x, x_stride;     // delta: the convolution's ring is brought up to date here
  uint32_t seq_stride;                                // of the state; grid z: the sequence, its rows m z .. of the activations
};
template <int NT, int FORM> struct ChunkOps { f4_t w[NT], q[NT], k[NT], gl[NT], u; std::conditional_t<FORM == SCAN_TURNS, f4_t, float> b; };

template <bool DELTA, int NT, int FORM>
__device__ __forceinline__ void load_ops(ChunkOps<NT, FORM>& o, const float* blk, const ChunkDims& cd, uint32_t wave, uint32_t lane, uint32_t v0) {
  const float *pQ = blk + CH * cd.Dp, *pK = pQ + CH * cd.Dp, *pB = pK + CH * cd.Dp, *pU = pB + 256u, *pG = pU + CH * cd.Vp;
#pragma unroll
  for (int j = 0; j < NT; j++) {
    const uint32_t T = wave * NT + j, at = T * 256u + lane * 4u;
    if (DELTA) o.w[j] = *(const f4_t*)(blk + at);
    o.q[j] = *(const f4_t*)(pQ + at);
    o.k[j] = *(const f4_t*)(pK + at);
    o.gl[j] = *(const f4_t*)(pG + T * 16u + (lane >> 4) * 4u);
  }
  o.u = *(const f4_t*)(pU + v0 * 16u + lane * 4u);
  if constexpr (FORM == SCAN_TURNS) o.b = *(const f4_t*)(pB + lane * 4u);
  else o.b = pB[lane * 4u + wave];
}

template <bool DELTA, int NT, int FORM>
__global__ void __launch_bounds__(SCAN_T(FORM), FORM == SCAN_TURNS ? 2 : 1)
k_chunk_scan(const ScanArgs a, const float* __restrict__ scratch, float* act, float* state) {
  __shared__ f4_t p1[2][4][64], p2[2][4][64];                // [chunk & 1][wave][lane]
  __shared__ f4_t pb[2][64], pu[2][64];                      // B and u for the fifth wave, one of a lane's four by each wave
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6)), c = lane & 15u, kg = lane >> 4;
  const uint32_t h = blockIdx.x, v0 = blockIdx.y * 16u, D = a.dim, V = a.vdim, v = v0 + c;
  const uint32_t bs = chunk_floats(a.cd.Dp, a.cd.Vp), n = a.cd.n_chunks;
  const float* blk = scratch + ((uint64_t)blockIdx.z * a.heads + h) * n * bs;
  state += (uint64_t)blockIdx.z * a.seq_stride;
  float* out = act + a.out + (uint64_t)blockIdx.z * a.m * a.out_stride + h * V + v;
  const auto put = [&](uint32_t ci, f4_t b, f4_t u) {        // the outputs of chunk ci
    const f4_t (*p)[64] = p2[ci & 1u];
    f4_t o = (p[0][lane] + p[1][lane]) + (p[2][lane] + p[3][lane]);
#pragma unroll
    for (int i = 0; i < 4; i++) o = __builtin_amdgcn_mfma_f32_16x16x4f32(b[i], u[i], o, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t r = ci * CH + 4u * kg + i;
      if (r < a.m && v < V) out[(uint64_t)r * a.out_stride] = o[i];
    }
  };
  if (FORM != SCAN_TURNS && wave == 4u) {
    if (DELTA) __syncthreads();                              // (there a chunk's shares are whole at the next one's barrier)
    for (uint32_t ci = 0; ci < n; ci++) {
      __syncthreads();
      put(ci, pb[ci & 1u][lane], pu[ci & 1u][lane]);
    }
  } else {
    float* S = state + a.s_off + (uint64_t)h * D * V;
    f4_t st[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) st[j] = (f4_t){0, 0, 0, 0};
    if (a.pos != 0u) {
#pragma unroll
      for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) st[j][i] = S[(uint64_t)min((wave * NT + j) * 16u + 4u * kg + i, D - 1u) * V + min(v, V - 1u)];
#pragma unroll
      for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) if ((wave * NT + j) * 16u + 4u * kg + i >= D || v >= V) st[j][i] = 0.f;
    }
    // the operands of the chunk two ahead, asked for on every path (past the end: the last one's again)
    const auto ask = [&](ChunkOps<NT, FORM>& o, uint32_t ci) { load_ops<DELTA, NT, FORM>(o, blk + (uint64_t)min(ci, n - 1u) * bs, a.cd, wave, lane, v0); __builtin_amdgcn_sched_barrier(0); };
    const auto chunk = [&](const ChunkOps<NT, FORM>& cur, uint32_t ci) {
      const uint32_t x = ci & 1u;
      f4_t u = cur.u, s = {0, 0, 0, 0}, q_s = {0, 0, 0, 0}, r[4], was[NT];
      const auto k_u = [&](int t) { st[t % NT] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.k[t % NT][t / NT], u[t / NT], st[t % NT], 0, 0, 0); };
      const auto share = [&] {                               // of the outputs
        p2[x][wave][lane] = q_s;
        if constexpr (FORM != SCAN_TURNS) {
          ((float*)&pb[x][lane])[wave] = cur.b;
          ((float*)&pu[x][lane])[wave] = wave & 2u ? (wave & 1u ? u[3] : u[2]) : (wave & 1u ? u[1] : u[0]);
        }
      };
      constexpr bool Q_AHEAD = FORM == SCAN_TURNS;           // of the barrier
      if (DELTA || Q_AHEAD)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
          for (int i = 0; i < 4; i++) {
            if (DELTA) s = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.w[j][i], st[j][i], s, 0, 0, 0);
            if (Q_AHEAD) q_s = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.q[j][i], st[j][i], q_s, 0, 0, 0);
          }
      if (DELTA) p1[x][wave][lane] = s;
      else if (!Q_AHEAD) {                                   // (an instruction waits for the one that it adds to: two sums in turn)
#pragma unroll
        for (int j = 0; j < NT; j++) { was[j] = st[j]; st[j] *= cur.gl[j]; }
#pragma unroll
        for (int t = 0; t < 4 * NT; t++) {
          q_s = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.q[t / 4][t % 4], was[t / 4][t % 4], q_s, 0, 0, 0);
          k_u(t);
        }
      }
      if (!DELTA || Q_AHEAD) share();
      __syncthreads();
      if (DELTA)
#pragma unroll
        for (int w = 0; w < 4; w++) r[w] = p1[x][w][lane];
      __builtin_amdgcn_sched_barrier(0);                     // Q S behind them, not ahead of the barrier
      if (DELTA && !Q_AHEAD)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
          for (int i = 0; i < 4; i++) q_s = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.q[j][i], st[j][i], q_s, 0, 0, 0);
      if (DELTA) u -= (r[0] + r[1]) + (r[2] + r[3]);
      if constexpr (FORM == SCAN_TURNS) if (wave == (ci & 3u)) put(ci, cur.b, u);
      if (DELTA || Q_AHEAD) {
#pragma unroll
        for (int j = 0; j < NT; j++) st[j] *= cur.gl[j];
#pragma unroll
        for (int t = 0; t < 4 * NT; t++) k_u(t);
        if (!Q_AHEAD) share();
      }
    };
    ChunkOps<NT, FORM> o0;
    ask(o0, 0);
    if constexpr (FORM == SCAN_FEW) {
      for (uint32_t ci = 0; ci < n; ci++) {
        if (ci) ask(o0, ci);
        chunk(o0, ci);
      }
    } else {
      // (a loop in one piece: with a way out behind each chunk the loads were moved down to where only the rest of the loop needs them)
      ChunkOps<NT, FORM> o1, o2;
      ask(o1, 1); ask(o2, 2);
      uint32_t ci = 0;
      for (; ci + 3u <= n; ci += 3u) {
        chunk(o0, ci);
        ask(o0, ci + 3u);
        chunk(o1, ci + 1u);
        ask(o1, ci + 4u);
        chunk(o2, ci + 2u);
        ask(o2, ci + 5u);
      }
      if (ci < n) chunk(o0, ci);
      if (ci + 1u < n) chunk(o1, ci + 1u);
    }
    if (DELTA && FORM != SCAN_TURNS) __syncthreads();        // the last chunk's shares are there
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t d = (wave * NT + j) * 16u + 4u * kg + i;
        if (d < D && v < V) S[(uint64_t)d * V + v] = st[j][i];
      }
  }
  if (!DELTA) return;
  const uint32_t n_ch = 2u * a.kv_heads * D + a.heads * V, rep = a.heads / a.kv_heads, kv = h / rep;
  for (uint32_t r = a.m > a.taps ? a.m - a.taps : 0u; r < a.m; r++) {
    float* slot = state + a.conv_off + (uint64_t)((a.pos + r) % a.taps) * n_ch;
    const float* x = act + a.x + ((uint64_t)blockIdx.z * a.m + r) * a.x_stride;
    if (blockIdx.y == 0 && h % rep == 0)
      for (uint32_t d = tid; d < D; d += SCAN_T(FORM)) {
        slot[kv * D + d] = x[kv * D + d];
        slot[(a.kv_heads + kv) * D + d] = x[(a.kv_heads + kv) * D + d];
      }
    const uint32_t vc = 2u * a.kv_heads * D + h * V + v;
    if (wave == 0u && kg == 0u && v < V) slot[vc] = x[vc];
  }
}

static Scratch g_chunks;
void recurrent_release() { scratch_free(g_chunks); }

static bool rows_ok(uint64_t off, uint64_t stride, uint64_t rows, uint64_t width, uint64_t n_elems) {
  return in_range(off, (rows - 1) * stride + width, n_elems);
}

template <bool DELTA>
static int launch_scan(const ScanArgs& a, float* act, float* state, uint32_t n_seq) {
  const dim3 grid(a.heads, cdiv(a.vdim, 16), n_seq);
  const float* sc = (const float*)g_chunks.p;
  const auto go = [&](auto tiles) {
    constexpr int NT = decltype(tiles)::value;
    constexpr bool turns = !DELTA || NT < 4;                 // (that one would spill)
    const int form = scan_form((uint64_t)grid.x * grid.y * grid.z, a.cd.n_chunks, NT, NT == 1 || (!DELTA && NT == 2), turns);
    if (form == SCAN_FEW) k_chunk_scan<DELTA, NT, SCAN_FEW><<<grid, SCAN_T(SCAN_FEW), 0, g.stream>>>(a, sc, act, state);
    else if (form == SCAN_DEEP) k_chunk_scan<DELTA, NT, SCAN_DEEP><<<grid, SCAN_T(SCAN_DEEP), 0, g.stream>>>(a, sc, act, state);
    else if constexpr (turns) k_chunk_scan<DELTA, NT, SCAN_TURNS><<<grid, SCAN_T(SCAN_TURNS), 0, g.stream>>>(a, sc, act, state);
  };
  switch (a.cd.Dp / 64u) {
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 3: go(std::integral_constant<int, 3>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    default: return ADAMAH_ERR_INVALID;
  }
  count_launch();
  return check_launch();
}

static LowRank low_rank(const LinSpec& s) { return {s.w, s.k, s.k_stride, s.src, s.src_stride, s.out, s.out_stride}; }

// n_seq sequences of `rows` tokens each, one behind the other in the activations, their states from slot seq0 on.
static int run_delta_rule(uint32_t map_act, uint32_t map_opnd, uint32_t map_wt, uint32_t h_spec, uint32_t h_decay, uint32_t h_gate,
                          uint32_t n_seq, uint32_t rows, uint32_t seq0, uint32_t pos) {
  Map *ma = get_f32_map(map_act), *mo = get_map(map_opnd), *mw = get_map(map_wt);
  const DSpec* s = spec_of<DSpec>(h_spec);
  const LinSpec *da = spec_of<LinSpec>(h_decay), *ga = spec_of<LinSpec>(h_gate);
  if (!ma || !mw || mw->dtype != DTYPE_BF16 || !s || !da || !ga || n_seq == 0 || rows == 0 || (uint64_t)n_seq * rows > 0xFFFFFFFFull) return ADAMAH_ERR_INVALID;
  Map* ms = get_f32_map(s->state_map);
  const uint64_t D = s->dim, V = s->vdim, H = s->heads, KH = s->kv_heads, n_tok = (uint64_t)n_seq * rows;
  if (!ms || D == 0 || D > 256 || V == 0 || H == 0 || KH == 0 || H % KH || s->taps == 0 || s->taps > MAX_TAPS) return ADAMAH_ERR_INVALID;
  const uint64_t n_ch = 2 * KH * D + H * V;
  if (s->x_stride < n_ch || s->x_b + H > s->x_stride) return ADAMAH_ERR_INVALID;
  if (!rows_ok(s->x, s->x_stride, n_tok, s->x_stride, ma->n_elems) || !rows_ok(s->out, s->out_stride, n_tok, H * V, ma->n_elems)) return ADAMAH_ERR_INVALID;
  if (!in_range(s->cq, KH * D * s->taps, ma->n_elems) || !in_range(s->ck, KH * D * s->taps, ma->n_elems) ||
      !in_range(s->cv, H * V * s->taps, ma->n_elems) || !in_range(s->a_log, H, ma->n_elems) || !in_range(s->dt_bias, H * D, ma->n_elems)) return ADAMAH_ERR_INVALID;
  if ((uint64_t)s->s_off + H * D * V > s->seq_stride || (uint64_t)s->conv_off + n_ch * s->taps > s->seq_stride ||
      !in_range((uint64_t)seq0 * s->seq_stride, (uint64_t)n_seq * s->seq_stride, ms->n_elems)) return ADAMAH_ERR_INVALID;
  for (const LinSpec* l : {da, ga}) {
    const uint64_t n = l == da ? H * D : H * V;
    if (l->n != n || l->k == 0 || l->k_stride < l->k || (l->k_stride & 63u) || (l->w & 7u) || l->epi || l->groups ||
        !in_range(l->w, n * l->k_stride, mw->n_elems) || !rows_ok(l->src, l->src_stride, n_tok, l->k, ma->n_elems) ||
        !rows_ok(l->out, l->out_stride, n_tok, n, ma->n_elems)) return ADAMAH_ERR_INVALID;
  }
  float *act = (float*)ma->buf, *state = (float*)ms->buf;
  if (rows == 1) {
    const size_t lds = (size_t)(3 * D + da->k_stride + ga->k_stride) * 4;
    if (lds > 48000) return ADAMAH_ERR_INVALID;
    const bf16_t* W = (const bf16_t*)mw->buf;
    // Four columns a thread once that alone gives more than every other compute unit a workgroup, and rows start on 16
    // bytes.  Heads of 128 x 128, us with one and four (the state at a large copy's rate): 32 heads 1 sequence 8.4 / 9.6 (0.9),
    // 4 12.0 / 11.6 (3.5), 8 21.6 / 14.7 (6.9), 16 38.5 / 20.9 (13.8), 32 77 / 45 (28); 16 heads 4 8.9 / 10.0, 16 21.8 / 14.6.
    // Beyond 128 rows of state a thread's part of it would leave one workgroup a compute unit.
    const bool wide = s->taps <= 4 && D <= 128 && V > 2 * VC && !((V | s->s_off | s->seq_stride) & 3u) &&
                      2 * H * cdiv(V, 4 * VC) * n_seq > (uint64_t)g.n_cu;
    const dim3 grid((uint32_t)H, cdiv(V, wide ? 4 * VC : VC), n_seq);
#define STEP(DN, TM, CW) k_delta_step<DN, TM, CW><<<grid, DSTEP, lds, g.stream>>>(*s, low_rank(*da), low_rank(*ga), act, W, state, seq0, pos)
    if (wide) { if (D <= 64) STEP(4, 4, 4); else STEP(8, 4, 4); }
    else if (s->taps <= 4) { if (D <= 64) STEP(4, 4, 1); else if (D <= 128) STEP(8, 4, 1); else STEP(16, 4, 1); }
    else { if (D <= 64) STEP(4, MAX_TAPS, 1); else if (D <= 128) STEP(8, MAX_TAPS, 1); else STEP(16, MAX_TAPS, 1); }
#undef STEP
    count_launch();
    return check_launch();
  }
  if (int r = adamah_linear_dev(map_act, map_opnd, map_wt, h_decay, 0, n_seq * rows)) return r;
  if (int r = adamah_linear_dev(map_act, map_opnd, map_wt, h_gate, 0, n_seq * rows)) return r;
  const ChunkDims cd = {(uint32_t)((D + 63) / 64 * 64), (uint32_t)((V + 15) / 16 * 16), cdiv(rows, CH)};
  if (int r = scratch_need(g_chunks, (size_t)n_seq * H * cd.n_chunks * chunk_floats(cd.Dp, cd.Vp) * 4)) return r;
  const size_t lds = (size_t)CH * (3 * (D + 1) + cd.Vp) * 4;
  if (lds > 120000) return ADAMAH_ERR_INVALID;
#define PREP(TM)                                                                                                                      \
  do {                                                                                                                                \
    if (lds > 60000) hipFuncSetAttribute((const void*)k_delta_prep<TM>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);         \
    k_delta_prep<TM><<<dim3(cd.n_chunks, (uint32_t)H, n_seq), 256, lds, g.stream>>>(*s, da->out, da->out_stride, act, state,                 \
                                                                            (float*)g_chunks.p, cd, rows, seq0, pos);                \
  } while (0)
  if (s->taps <= 4) PREP(4); else PREP(MAX_TAPS);
#undef PREP
  count_launch();
  if (int r = check_launch()) return r;
  ScanArgs a = {s->heads, s->dim, s->vdim, s->out, s->out_stride, s->s_off, rows, pos, cd, s->kv_heads, s->taps, s->conv_off, s->x, s->x_stride, s->seq_stride};
  return launch_scan<true>(a, act, state + (uint64_t)seq0 * s->seq_stride, n_seq);
}

static int run_retention(uint32_t map_act, uint32_t h_spec, uint32_t n_seq, uint32_t rows, uint32_t seq0, uint32_t pos) {
  Map* ma = get_f32_map(map_act);
  const RSpec* s = spec_of<RSpec>(h_spec);
  if (!ma || !s || n_seq == 0 || rows == 0 || (uint64_t)n_seq * rows > 0xFFFFFFFFull) return ADAMAH_ERR_INVALID;
  Map* ms = get_f32_map(s->state_map);
  const uint64_t D = s->dim, V = s->vdim, H = s->heads, n_tok = (uint64_t)n_seq * rows;
  if (!ms || D == 0 || D > 256 || V == 0 || H == 0 || s->rot_dims > D || (s->rot_dims & 1u)) return ADAMAH_ERR_INVALID;
  if (s->x_q + H * D > s->x_stride || s->x_k + H * D > s->x_stride || s->x_v + H * V > s->x_stride ||
      !rows_ok(s->x, s->x_stride, n_tok, s->x_stride, ma->n_elems) || !rows_ok(s->out, s->out_stride, n_tok, H * V, ma->n_elems) ||
      !in_range(s->freq, s->rot_dims / 2, ma->n_elems) || !in_range(s->decay, H, ma->n_elems)) return ADAMAH_ERR_INVALID;
  if ((uint64_t)s->s_off + H * D * V > s->seq_stride ||
      !in_range((uint64_t)seq0 * s->seq_stride, (uint64_t)n_seq * s->seq_stride, ms->n_elems)) return ADAMAH_ERR_INVALID;
  float *act = (float*)ma->buf, *state = (float*)ms->buf;
  if (rows == 1) {
    const dim3 grid((uint32_t)H, cdiv(V, VC), n_seq);
    const size_t lds = (size_t)2 * D * 4;
    if (D <= 64) k_retention_step<8><<<grid, 256, lds, g.stream>>>(*s, act, state, seq0, pos);
    else if (D <= 128) k_retention_step<16><<<grid, 256, lds, g.stream>>>(*s, act, state, seq0, pos);
    else k_retention_step<32><<<grid, 256, lds, g.stream>>>(*s, act, state, seq0, pos);
    count_launch();
    return check_launch();
  }
  const ChunkDims cd = {(uint32_t)((D + 63) / 64 * 64), (uint32_t)((V + 15) / 16 * 16), cdiv(rows, CH)};
  if (int r = scratch_need(g_chunks, (size_t)n_seq * H * cd.n_chunks * chunk_floats(cd.Dp, cd.Vp) * 4)) return r;
  k_retention_prep<<<dim3(cd.n_chunks, (uint32_t)H, n_seq), 256, (size_t)CH * (2 * (D + 1) + s->rot_dims) * 4, g.stream>>>(*s, act, (float*)g_chunks.p, cd, rows, pos);
  count_launch();
  if (int r = check_launch()) return r;
  ScanArgs a = {s->heads, s->dim, s->vdim, s->out, s->out_stride, s->s_off, rows, pos, cd, 0, 0, 0, 0, 0, s->seq_stride};
  return launch_scan<false>(a, act, state + (uint64_t)seq0 * s->seq_stride, n_seq);
}

}  // namespace adamah

using namespace adamah;

extern "C" {

int adamah_delta_rule_dev(uint32_t map_act, uint32_t map_opnd, uint32_t map_wt, uint32_t h_spec, uint32_t h_decay, uint32_t h_gate,
                          uint32_t n_seq, uint32_t rows, uint32_t seq0, uint32_t pos) { ADAMAH_API();
  if (n_seq > 1 && rows > 1) return ADAMAH_ERR_INVALID;
  return run_delta_rule(map_act, map_opnd, map_wt, h_spec, h_decay, h_gate, n_seq, rows, seq0, pos);
}

int adamah_hip_delta_rule_seqs_dev(uint32_t map_act, uint32_t map_opnd, uint32_t map_wt, uint32_t h_spec, uint32_t h_decay, uint32_t h_gate,
                                   uint32_t n_seq, uint32_t rows, uint32_t seq0, uint32_t pos) { ADAMAH_API();
  return run_delta_rule(map_act, map_opnd, map_wt, h_spec, h_decay, h_gate, n_seq, rows, seq0, pos);
}

int adamah_retention_dev(uint32_t map_act, uint32_t h_spec, uint32_t n_seq, uint32_t rows, uint32_t seq0, uint32_t pos) { ADAMAH_API();
  if (n_seq > 1 && rows > 1) return ADAMAH_ERR_INVALID;
  return run_retention(map_act, h_spec, n_seq, rows, seq0, pos);
}

int adamah_hip_retention_seqs_dev(uint32_t map_act, uint32_t h_spec, uint32_t n_seq, uint32_t rows, uint32_t seq0, uint32_t pos) { ADAMAH_API();
  return run_retention(map_act, h_spec, n_seq, rows, seq0, pos);
}

}  // extern "C"
