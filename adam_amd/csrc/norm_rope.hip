// RMSNorm (+ residual), half-split RoPE, fused per-head QK-norm + RoPE, and row copy (KV append).
//
// Reference kernels: shaders/src/f32/map_rmsnorm.comp, map_rmsnorm_x.comp:26-48,
// map_rmsnorm_add.comp:14-44, map_rope.comp:11-37, map_qk_norm_rope_x.comp:32-84,
// map_row_copy.comp:13-24; dispatchers adamah.c:7610-7878, 8476-8604, 8061-8085.
// Row bases come from device-resident loc arrays, one entry per row, as in the reference.
#include "common.h"
#include "gemv_common.h"
#include "../../include/adamah_hip.h"

namespace adamah {

__device__ __forceinline__ float block_sum_256(float v, float* sh) {
  v = wave_add(v);
  if ((threadIdx.x & 63u) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  __syncthreads();
  return t;
}

// y = x * (1/sqrt(sum(x^2)/dim + eps)) * w (+ r); one 256-thread workgroup per row
template <bool ADD>
__global__ void __launch_bounds__(256)
k_rmsnorm(const float* act, const float* wt, float* out, const uint32_t* __restrict__ ls,
          const uint32_t* __restrict__ lw, const uint32_t* __restrict__ lr, const uint32_t* __restrict__ ld,
          uint32_t dim, float eps, uint64_t act_elems, uint64_t wt_elems) {
  __shared__ float sh[4];
  const uint32_t ri = blockIdx.x, tid = threadIdx.x;
  const uint64_t sb = ls[ri], wb = lw[ri], db = ld[ri], rb = ADD ? (uint64_t)lr[ri] : 0;
  if (sb + dim > act_elems || db + dim > act_elems || wb + dim > wt_elems || (ADD && rb + dim > act_elems)) return;
  float ss = 0.f;
  for (uint32_t i = tid; i < dim; i += 256u) { float x = act[sb + i]; ss = fmaf(x, x, ss); }
  ss = block_sum_256(ss, sh);
  const float inv = 1.0f / sqrtf(ss / (float)dim + eps);
  for (uint32_t i = tid; i < dim; i += 256u) {
    float y = act[sb + i] * inv * wt[wb + i];
    if (ADD) y += act[rb + i];
    out[db + i] = y;
  }
}

// The same row op with the row held in registers: one trip to memory instead of two dependent passes, for rows of at most 8192.
// WIDE: rows of a multiple of eight, a thread owns the eight neighbours of one word (PER = 8, NT >= dim / 8 threads), loads and
// stores 16 bytes at a time; the squares pass through LDS, where 256 threads add them up in the order of the kernel above.
// Otherwise 256 threads own elements 256 apart (dim <= 256 PER), that kernel's order by itself.  The results are the same bits.
// EMIT: the rows are [n_rows, dim] back to back and a batched matmul follows; its fp16 operand form (row scaled by a power of two,
// two planes, 8-element words in the order (0,4)(1,5)(2,6)(3,7), plus (s, 1/s) per row) is written here as well, which spares that
// matmul its conversion launch.  A launch of few rows is one trip to memory, two sums over the workgroup and the stores: with one
// element a load and 256 threads a row it was 16 pairs of loads and 48 stores a thread.  us behind each other, operand form included,
// that and this: 8 rows of 4096 4.55 and 4.35, of 8192 6.5 and 6.1, 512 rows 7.5 and 7.3, 12.0 and 11.6; 2 rows of 4096 with a residual
// 4.7 and 4.2.  (Each thread's squares summed by itself, in another order: 4.0, 4.8, 6.4 and 10.1.)
struct RowsByValue { uint32_t on, s0, ss, w0, ws, d0, ds, r0, rs; };   // host side only
typedef float f4r_t __attribute__((ext_vector_type(4), aligned(4)));
template <bool ADD, bool EMIT, bool WIDE, int NT, int PER>
__global__ void __launch_bounds__(NT)
k_rmsnorm_rows(const float* act, const float* wt, uint32_t dim_on, float eps, uint32_t s0, uint32_t ss_, uint32_t w0, uint32_t ws,
               uint32_t d0, uint32_t ds, uint32_t r0, uint32_t rs, float* out,
               const uint32_t* __restrict__ ls, const uint32_t* __restrict__ lw, const uint32_t* __restrict__ lr,
               const uint32_t* __restrict__ ld, uint64_t act_elems, uint64_t wt_elems, float* scale, uint4* xf, ActForm form) {
  // (these 14 dwords are in registers when a wave starts.  Top bit of dim_on: row i's source / weights / destination /
  // residual start at x0 + i xs -- the host found the rows evenly spaced -- instead of four loads from the row
  // tables, which the rows' own loads would have to wait for)
  static_assert(WIDE ? PER == 8 : NT == 256 && !EMIT, "the operand form is made of whole words");
  __shared__ __attribute__((aligned(16))) float row[WIDE ? 8 * NT : 4];
  __shared__ float sums[4], tops[NT / 64];
  const uint32_t ri = blockIdx.x, tid = threadIdx.x, dim = dim_on & 0x7FFFFFFFu;
  uint64_t sb, wb, db, rb = 0;
  if (dim_on >> 31) {
    sb = (uint64_t)s0 + (uint64_t)ri * ss_; wb = (uint64_t)w0 + (uint64_t)ri * ws;
    db = (uint64_t)d0 + (uint64_t)ri * ds; if (ADD) rb = (uint64_t)r0 + (uint64_t)ri * rs;
  } else {
    sb = ls[ri]; wb = lw[ri]; db = ld[ri]; if (ADD) rb = lr[ri];
  }
  if (sb + dim > act_elems || db + dim > act_elems || wb + dim > wt_elems || (ADD && rb + dim > act_elems)) return;
  const bool in = tid < (dim >> 3);                          // WIDE: the thread has a word
  float x[PER], w[PER], r[PER], ss = 0.f;
  if (WIDE) {
    const uint32_t i = in ? tid * 8u : 0u;                   // (a thread past the row loads its first word)
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const f4r_t xv = *(const f4r_t*)(act + sb + i + 4 * h), wv = *(const f4r_t*)(wt + wb + i + 4 * h);
      f4r_t rv = {0.f, 0.f, 0.f, 0.f};
      if (ADD) rv = *(const f4r_t*)(act + rb + i + 4 * h);
#pragma unroll
      for (int e = 0; e < 4; e++) { x[4 * h + e] = xv[e]; w[4 * h + e] = wv[e]; r[4 * h + e] = rv[e]; }
    }
    *(f4r_t*)(row + tid * 8u) = (f4r_t){x[0], x[1], x[2], x[3]};
    *(f4r_t*)(row + tid * 8u + 4) = (f4r_t){x[4], x[5], x[6], x[7]};
    __syncthreads();
    if (tid < 256u) {
#pragma unroll
      for (uint32_t u = 0; u < 8u * NT / 256u; u++) {
        const float v = row[tid + 256u * u];
        ss = tid + 256u * u < dim ? fmaf(v, v, ss) : ss;
      }
    }
  } else {
#pragma unroll
    for (int e = 0; e < PER; e++) {
      const uint32_t i = min(tid + 256u * e, dim - 1u);
      x[e] = act[sb + i]; w[e] = wt[wb + i]; r[e] = ADD ? act[rb + i] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < PER; e++) ss = tid + 256u * e < dim ? fmaf(x[e], x[e], ss) : ss;
  }
  if (tid < 256u) {
    ss = wave_add(ss);
    if ((tid & 63u) == 0) sums[tid >> 6] = ss;
  }
  __syncthreads();
  const float inv = 1.0f / sqrtf(((sums[0] + sums[1]) + (sums[2] + sums[3])) / (float)dim + eps);
  float m = 0.f;
#pragma unroll
  for (int e = 0; e < PER; e++) {
    x[e] = x[e] * inv * w[e];
    if (ADD) x[e] += r[e];
    m = fmaxf(m, fabsf(x[e]));
  }
  if (!WIDE) {
#pragma unroll
    for (int e = 0; e < PER; e++) if (tid + 256u * e < dim) out[db + tid + 256u * e] = x[e];
  } else if (in) {
    *(f4r_t*)(out + db + tid * 8u) = (f4r_t){x[0], x[1], x[2], x[3]};
    *(f4r_t*)(out + db + tid * 8u + 4) = (f4r_t){x[4], x[5], x[6], x[7]};
  }
  if constexpr (EMIT) {
    if (!in) m = 0.f;
    m = wave_max(m);
    if ((tid & 63u) == 0) tops[tid >> 6] = m;
    __syncthreads();
    m = tops[0];
#pragma unroll
    for (int w = 1; w < NT / 64; w++) m = fmaxf(m, tops[w]);
    const uint32_t e = (__float_as_uint(m) >> 23) & 0xFFu;
    float s = 1.f, si = 1.f;
    if (e >= 14u && e <= 254u) { s = __uint_as_float((267u - e) << 23); si = __uint_as_float((e - 13u) << 23); }
    if (tid == 0) { scale[2 * ri] = s; scale[2 * ri + 1] = si; }
    if (!in) return;
    // two planes: fp16(x s) and the fp16 remainder x s - fp16(x s), as the matmul's own conversion writes them
    uint32_t hi[4], lo[4];
#pragma unroll
    for (int p = 0; p < 4; p++) {
      const float u = x[p] * s, v = x[p + 4] * s;
      const __half uh = __float2half(u), vh = __float2half(v);
      hi[p] = (uint32_t)__half_as_ushort(uh) | (uint32_t)__half_as_ushort(vh) << 16;
      lo[p] = (uint32_t)__half_as_ushort(__float2half(u - __half2float(uh))) | (uint32_t)__half_as_ushort(__float2half(v - __half2float(vh))) << 16;
    }
    xf[act_piece(form, 0u, ri, tid, 0u)] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    xf[act_piece(form, 0u, ri, tid, 1u)] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
  }
}

// theta_i = pos * (1 / base^(2i/dim)).  The exponent and the reciprocal are float32 operations as
// in the shader; the power itself is evaluated in double and rounded once, which makes the
// frequency independent of the float32 pow implementation.
__device__ __forceinline__ void rope_cs(uint32_t i, uint32_t dim, uint32_t pos, float base, float* c, float* s) {
  const float e = (float)(2u * i) / (float)dim;
  const float p = (float)pow((double)base, (double)e);
  const float angle = (float)pos * (1.0f / p);
  *c = cosf(angle);
  *s = sinf(angle);
}

__global__ void __launch_bounds__(256)
k_rope(float* data, const uint32_t* __restrict__ ls, const uint32_t* __restrict__ ld, uint32_t n_tokens,
       uint32_t n_heads, uint32_t head_dim, uint32_t pos_offset, float base, uint64_t n_elems) {
  const uint32_t half = head_dim >> 1;
  const uint64_t tid = (uint64_t)blockIdx.x * 256u + threadIdx.x;
  if (tid >= (uint64_t)n_tokens * n_heads * half) return;
  const uint32_t token = (uint32_t)(tid / ((uint64_t)n_heads * half));
  const uint32_t rem = (uint32_t)(tid % ((uint64_t)n_heads * half));
  const uint32_t head = rem / half, d = rem % half;
  const uint64_t bs = (uint64_t)ls[token] + (uint64_t)head * head_dim, bd = (uint64_t)ld[token] + (uint64_t)head * head_dim;
  if (bs + head_dim > n_elems || bd + head_dim > n_elems) return;
  float c, s;
  rope_cs(d, head_dim, pos_offset + token, base, &c, &s);
  const float x0 = data[bs + d], x1 = data[bs + d + half];
  data[bd + d] = x0 * c - x1 * s;
  data[bd + d + half] = x0 * s + x1 * c;
}

// The tokens of a prompt chunk, of one sequence or of several that stand side by side: rotation of their Q and K heads in place and
// the append of their K and V rows to the caches, a workgroup per token.  The sines and cosines of a position (a power in double each)
// are worked out once for its heads instead of once for each: the launch is a pass over the rows (512 tokens of 32 + 2 x 8 heads of
// 128: three launches of 12.7, 5.2 and 5.5 us before).  Arithmetic of the stand-alone kernels.
//
// A thread takes W neighbouring pairs of a head, value d and d + dim / 2 of each (of V as well, which is only moved), APPEND_UNITS
// times at once: none of these loads waits for a store or for the sines.  W is 4 where every row starts on 16 bytes, else 1.
// 32 + 2 x 8 heads of 128: 24 tokens 8.4 us a pair at a time in a loop, 4.5 so; 512 tokens 11.3 and 8.7.
#define APPEND_SEQS 32u
#define APPEND_UNITS 4
// (q, k, v: of the first sequence of the launch, which may lie beyond 2^32)
struct AppendRows { uint64_t q, k, v; uint32_t q_step, q_heads, k_step, k_heads, v_step, dim, n_tok, head_step, pos0, rotate; float base;
                    uint32_t kc[APPEND_SEQS], vc[APPEND_SEQS]; };
template <int W>
__global__ void __launch_bounds__(256)
k_rope_append_rows(float* data, const AppendRows a, __half* kv16, uint64_t kv_start, uint64_t kv_count) {
  typedef float fw_t __attribute__((ext_vector_type(W)));
  typedef _Float16 hw_t __attribute__((ext_vector_type(W)));
  constexpr int U = APPEND_UNITS;
  extern __shared__ float turn[];                            // [dim / 2] cosines, then sines
  const uint32_t t = blockIdx.x, sq = blockIdx.y, tid = threadIdx.x, half = a.dim >> 1, per = half / W, pos = a.pos0 + t;
  const uint64_t row = (uint64_t)sq * a.n_tok + t;
  const uint32_t nq = a.rotate ? a.q_heads : 0u, units = (nq + 2u * a.k_heads) * per;
  // head i: the Q heads, those of K, those of V
  const auto from = [&](uint32_t i) -> float* {
    if (i < nq) return data + a.q + row * a.q_step + (uint64_t)i * a.dim;
    if (i < nq + a.k_heads) return data + a.k + row * a.k_step + (uint64_t)(i - nq) * a.dim;
    return data + a.v + row * a.v_step + (uint64_t)(i - nq - a.k_heads) * a.dim;
  };
  fw_t x0[U], x1[U];
  const auto ask = [&](uint32_t u0) {
#pragma unroll
    for (int j = 0; j < U; j++) {
      const uint32_t u = min(u0 + 256u * j + tid, units - 1u);
      const float* x = from(u / per) + (u % per) * W;
      x0[j] = *(const fw_t*)x; x1[j] = *(const fw_t*)(x + half);
    }
  };
  ask(0);
  if (a.rotate) {
    for (uint32_t d = tid; d < half; d += 256u) rope_cs(d, a.dim, pos, a.base, &turn[d], &turn[half + d]);
    __syncthreads();
  }
  const auto put = [&](uint64_t at, fw_t v) {                // into the cache: rounded to fp16 and mirrored, as the row copy does
    if (kv16 && at >= kv_start && at - kv_start < kv_count) {
      const hw_t h = __builtin_convertvector(v, hw_t);
      *(hw_t*)(kv16 + (at - kv_start)) = h;
      v = __builtin_convertvector(h, fw_t);
    }
    *(fw_t*)(data + at) = v;
  };
  for (uint32_t u0 = 0;;) {
#pragma unroll
    for (int j = 0; j < U; j++) {
      const uint32_t u = u0 + 256u * j + tid, i = u / per, d = (u % per) * W;
      if (u >= units) break;
      fw_t r0 = x0[j], r1 = x1[j];
      if (a.rotate && i < nq + a.k_heads) {
#pragma unroll
        for (int c = 0; c < W; c++) {
          const float cs = turn[d + c], sn = turn[half + d + c], p = x0[j][c], q = x1[j][c];
          r0[c] = p * cs - q * sn;
          r1[c] = p * sn + q * cs;
        }
        float* x = from(i) + d;
        *(fw_t*)x = r0; *(fw_t*)(x + half) = r1;
      }
      if (i >= nq) {
        const uint32_t h = i - nq, of_v = h >= a.k_heads;
        const uint64_t at = (uint64_t)(of_v ? a.vc[sq] : a.kc[sq]) + (uint64_t)(h - (of_v ? a.k_heads : 0u)) * a.head_step + (uint64_t)pos * a.dim + d;
        put(at, r0);
        put(at + half, r1);
      }
    }
    u0 += 256u * U;
    if (u0 >= units) break;
    ask(u0);
  }
}

// One workgroup per Q or K row: RMSNorm with eps = 1e-6 (fixed in the shader), weight per row from
// map_wt, then RoPE; rows written contiguously (Q rows, then K rows) from locs_qk_dst[0].
__global__ void __launch_bounds__(256)
k_qk_norm_rope(float* act, const float* wt, const uint32_t* __restrict__ lqs, const uint32_t* __restrict__ lqw,
               const uint32_t* __restrict__ lks, const uint32_t* __restrict__ lkw, const uint32_t* __restrict__ ldst,
               uint32_t q_rows, uint32_t q_dim, uint32_t k_rows, uint32_t k_dim, uint32_t pos, float base,
               uint64_t act_elems, uint64_t wt_elems) {
  __shared__ float sh[4];
  const uint32_t row = blockIdx.x, tid = threadIdx.x;
  const bool is_q = row < q_rows;
  const uint32_t lr = is_q ? row : row - q_rows;
  const uint32_t dim = is_q ? q_dim : k_dim, half = dim >> 1;
  if (half == 0) return;
  const uint64_t sb = is_q ? lqs[lr] : lks[lr], wb = is_q ? lqw[lr] : lkw[lr];
  const uint64_t db = (uint64_t)ldst[0] + (is_q ? (uint64_t)lr * q_dim : (uint64_t)q_rows * q_dim + (uint64_t)lr * k_dim);
  if (sb + dim > act_elems || db + dim > act_elems || wb + dim > wt_elems) return;
  float ss = 0.f;
  for (uint32_t i = tid; i < dim; i += 256u) { float x = act[sb + i]; ss = fmaf(x, x, ss); }
  ss = block_sum_256(ss, sh);
  const float inv = 1.0f / sqrtf(ss / (float)dim + 1e-6f);
  for (uint32_t i = tid; i < half; i += 256u) {
    const float y0 = act[sb + i] * inv * wt[wb + i];
    const float y1 = act[sb + i + half] * inv * wt[wb + i + half];
    float c, s;
    rope_cs(i, dim, pos, base, &c, &s);
    act[db + i] = y0 * c - y1 * s;
    act[db + i + half] = y0 * s + y1 * c;
  }
}

// spec = [src_row, dst_row] pairs; src = src_base[0] + src_row*row_size; dst = (dst_row+offset)*row_size.
// Destinations inside the map's fp16 KV range are rounded to fp16 and mirrored.
__global__ void __launch_bounds__(256)
k_row_copy(float* data, const uint32_t* __restrict__ spec, const uint32_t* __restrict__ src_base, uint32_t n_copies,
           uint32_t row_size, uint32_t dst_row_offset, uint64_t n_elems, __half* kv16, uint64_t kv_start,
           uint64_t kv_count) {
  const uint64_t tid = (uint64_t)blockIdx.x * 256u + threadIdx.x;
  const uint32_t ci = (uint32_t)(tid / row_size), ei = (uint32_t)(tid % row_size);
  if (ci >= n_copies) return;
  const uint64_t so = (uint64_t)src_base[0] + (uint64_t)spec[2 * ci] * row_size + ei;
  const uint64_t dof = ((uint64_t)spec[2 * ci + 1] + dst_row_offset) * row_size + ei;
  if (so >= n_elems || dof >= n_elems) return;
  float v = data[so];
  if (kv16 && dof >= kv_start && dof - kv_start < kv_count) {
    const __half h = __float2half(v);
    kv16[dof - kv_start] = h;
    v = __half2float(h);
  }
  data[dof] = v;
}

static int rmsnorm_impl(uint32_t map_act, uint32_t map_wt, uint32_t hs, uint32_t hw, uint32_t hr, uint32_t hd,
                        uint32_t n_rows, uint32_t dim, float eps, bool add) {
  Map* ma = get_f32_map(map_act);
  Map* mw = get_f32_map(map_wt);
  if (!ma || !mw) return ADAMAH_ERR_INVALID;
  if (n_rows == 0) return ADAMAH_OK;
  if (n_rows == 1 && dim > 0 && can_defer()) {
    // single row with operands known on the host: queue it, a neighbouring GEMV may absorb it
    PendOp p;
    if (res_scalar(hs, &p.a) && res_scalar(hw, &p.b) && res_scalar(hd, &p.c) && (!add || res_scalar(hr, &p.d)) &&
        in_range(p.a, dim, ma->n_elems) && in_range(p.c, dim, ma->n_elems) && in_range(p.b, dim, mw->n_elems) &&
        (!add || in_range(p.d, dim, ma->n_elems))) {
      p.kind = PK_RMSNORM; p.map_act = map_act; p.map_wt = map_wt; p.n = dim; p.op = add ? 1u : 0u; p.eps = eps;
      g.pend.push_back(p);
      return ADAMAH_OK;
    }
  }
  flush_pending();
  const uint32_t *ls = res_u32(hs, n_rows), *lw = res_u32(hw, n_rows), *ld = res_u32(hd, n_rows);
  const uint32_t* lr = add ? res_u32(hr, n_rows) : ls;
  if (!ls || !lw || !ld || !lr) return ADAMAH_ERR_INVALID;
  float* a = (float*)ma->buf;
  if (n_rows > 1 && dim > 0 && dim <= 8192 && tuning("ADAMAH_RMSNORM_ROWS", 1) != 0) {
    // rows in registers; when the results are the rows of a matrix [n_rows, dim], also in the form the
    // batched matmul reads
    const uint32_t* dh = res_host(hd, n_rows);
    bool emit = dh && dim >= 128 && (dim & 127u) == 0 && n_rows <= 4096 && tuning("ADAMAH_RMSNORM_EMIT", 1) != 0;
    for (uint32_t i = 1; emit && i < n_rows; i++) emit = (uint64_t)dh[i] == (uint64_t)dh[0] + (uint64_t)i * dim;
    // the kernel skips a row whose operands are out of range: only rows the host can vouch for are marked
    const uint32_t *sh = res_host(hs, n_rows), *wh = res_host(hw, n_rows), *rh = add ? res_host(hr, n_rows) : nullptr;
    emit = emit && sh && wh && (!add || rh);
    for (uint32_t i = 0; emit && i < n_rows; i++)
      emit = in_range(sh[i], dim, ma->n_elems) && in_range(dh[i], dim, ma->n_elems) && in_range(wh[i], dim, mw->n_elems) &&
             (!add || in_range(rh[i], dim, ma->n_elems));
    float* scale = nullptr;
    uint4* xf = nullptr;
    ActForm form = {};
    if (emit) emit = gemm_act_slots(n_rows, dim, &scale, &xf, &form);
    const float* w = (const float*)mw->buf;
    // evenly spaced rows (the usual case: rows of a matrix, one weight vector): their places go by value
    RowsByValue rv = {};
    {
      const uint32_t *s_h = res_host(hs, n_rows), *w_h = res_host(hw, n_rows), *d_h = res_host(hd, n_rows);
      const uint32_t* r_h = add ? res_host(hr, n_rows) : s_h;
      bool even = s_h && w_h && d_h && r_h && s_h[1] >= s_h[0] && w_h[1] >= w_h[0] && d_h[1] >= d_h[0] && r_h[1] >= r_h[0];
      if (even) {
        rv = {1u, s_h[0], s_h[1] - s_h[0], w_h[0], w_h[1] - w_h[0], d_h[0], d_h[1] - d_h[0], r_h[0], r_h[1] - r_h[0]};
        for (uint32_t i = 1; even && i < n_rows; i++)
          even = s_h[i] == s_h[0] + i * rv.ss && w_h[i] == w_h[0] + i * rv.ws && d_h[i] == d_h[0] + i * rv.ds &&
                 r_h[i] == r_h[0] + i * rv.rs;
      }
      if (!even) rv.on = 0u;
    }
#define RR(A, E, V, NT, PER) k_rmsnorm_rows<A, E, V, NT, PER><<<n_rows, NT, 0, g.stream>>>(a, w, dim | (rv.on << 31), eps, rv.s0, rv.ss, rv.w0, rv.ws, rv.d0, rv.ds, rv.r0, rv.rs, a, ls, lw, lr, ld, ma->n_elems, mw->n_elems, scale, xf, form)
#define RN(A, E) do { if (dim <= 2048) RR(A, E, true, 256, 8); else if (dim <= 4096) RR(A, E, true, 512, 8); else RR(A, E, true, 1024, 8); } while (0)
#define RO(A) do { if (dim <= 2048) RR(A, false, false, 256, 8); else if (dim <= 4096) RR(A, false, false, 256, 16); else RR(A, false, false, 256, 32); } while (0)
    if (dim & 7u) { if (add) RO(true); else RO(false); }
    else if (add) { if (emit) RN(true, true); else RN(true, false); }
    else { if (emit) RN(false, true); else RN(false, false); }
#undef RO
#undef RN
#undef RR
    count_launch();
    if (emit) gemm_act_mark(ma->buf, dh[0], n_rows, dim);
    return check_launch();
  }
  if (add)
    k_rmsnorm<true><<<n_rows, 256, 0, g.stream>>>(a, (const float*)mw->buf, a, ls, lw, lr, ld, dim, eps, ma->n_elems,
                                                  mw->n_elems);
  else
    k_rmsnorm<false><<<n_rows, 256, 0, g.stream>>>(a, (const float*)mw->buf, a, ls, lw, lr, ld, dim, eps, ma->n_elems,
                                                   mw->n_elems);
  count_launch();
  return check_launch();
}

// One token of many sequences in lockstep: the rotation of all their Q heads, the rotation of all their K heads and the
// append of the K and V rows to the caches (three ops, issued in that order) in one launch.  One workgroup per
// row: the Q rows, then the K rows, then the copies.  A copy whose source is a K row of the launch is done by that
// row's workgroup, which finds it in the copy list and stores the rotated row twice (in place, and to the cache with
// the cache's fp16 rounding); its own workgroup leaves at once.  The host has checked that every copy's source is
// either exactly one such K row (each at most once) or lies clear of both rotated ranges, and that all destinations
// lie in the fp16 KV range, which holds no source.  Arithmetic of the three stand-alone kernels.
__global__ void __launch_bounds__(256)
k_rope2_copy(float* data, uint32_t qa, uint32_t q_rows, uint32_t q_dim, uint32_t ka, uint32_t k_rows, uint32_t k_dim,
             uint32_t pos, float base, const uint32_t* __restrict__ spec, uint32_t src_base, uint32_t n_copies,
             uint32_t dst_row_offset, __half* kv16, uint64_t kv_start, uint64_t kv_count) {
  __shared__ uint32_t found;
  const uint32_t b = blockIdx.x, tid = threadIdx.x;
  auto put = [&](uint64_t dof, float v) {     // into the cache: rounded to fp16 and mirrored, as the row copy does
    if (kv16 && dof >= kv_start && dof - kv_start < kv_count) {
      const __half h = __float2half(v);
      kv16[dof - kv_start] = h;
      v = __half2float(h);
    }
    data[dof] = v;
  };
  if (b < q_rows + k_rows) {
    const bool is_q = b < q_rows;
    const uint32_t dim = is_q ? q_dim : k_dim, half = dim >> 1;
    const uint64_t row = is_q ? (uint64_t)qa + (uint64_t)b * q_dim : (uint64_t)ka + (uint64_t)(b - q_rows) * k_dim;
    uint32_t dst_row = 0xFFFFFFFFu;
    if (!is_q) {
      if (tid == 0) found = 0xFFFFFFFFu;
      __syncthreads();
      for (uint32_t ci = tid; ci < n_copies; ci += 256u)
        if ((uint64_t)src_base + (uint64_t)spec[2 * ci] * k_dim == row) found = spec[2 * ci + 1];   // at most one
      __syncthreads();
      dst_row = found;
    }
    for (uint32_t d = tid; d < half; d += 256u) {
      float c, s;
      rope_cs(d, dim, pos, base, &c, &s);
      const float x0 = data[row + d], x1 = data[row + d + half];
      const float r0 = x0 * c - x1 * s, r1 = x0 * s + x1 * c;
      data[row + d] = r0;
      data[row + d + half] = r1;
      if (dst_row != 0xFFFFFFFFu) {
        const uint64_t dof = ((uint64_t)dst_row + dst_row_offset) * k_dim;
        put(dof + d, r0);
        put(dof + d + half, r1);
      }
    }
    return;
  }
  const uint32_t ci = b - q_rows - k_rows;
  const uint64_t so = (uint64_t)src_base + (uint64_t)spec[2 * ci] * k_dim;
  if (so >= ka && so < (uint64_t)ka + (uint64_t)k_rows * k_dim) return;     // done by the K row's workgroup
  const uint64_t dof = ((uint64_t)spec[2 * ci + 1] + dst_row_offset) * k_dim;
  for (uint32_t e = tid; e < k_dim; e += 256u) put(dof + e, data[so + e]);
}

// A queued rotation (one token, more heads than a row run holds) or row copy (more copies than that) by itself.
static int launch_wide_alone(const PendOp& p, Map* m) {
  if (p.kind == PK_ROPE) {
    const uint32_t *ls = res_u32(p.h[0], 1), *ld = res_u32(p.h[1], 1);
    if (!ls || !ld) return ADAMAH_ERR_INVALID;
    const uint64_t pairs = (uint64_t)p.rpg * (p.k / 2);
    k_rope<<<cdiv(pairs, 256), 256, 0, g.stream>>>((float*)m->buf, ls, ld, 1, p.rpg, p.k, p.n, p.eps, m->n_elems);
  } else {
    const uint32_t *spec = res_u32(p.h[0], 2ull * p.rpg), *base = res_u32(p.h[1], 1);
    if (!spec || !base) return ADAMAH_ERR_INVALID;
    k_row_copy<<<cdiv((uint64_t)p.rpg * p.k, 256), 256, 0, g.stream>>>((float*)m->buf, spec, base, p.rpg, p.k, p.n, m->n_elems, m->kv16,
                                                                    m->kv_start, m->kv_count);
  }
  count_launch();
  return check_launch();
}

// q[i] is a wide rotation or row copy (op == 1).  Rotation of the Q heads, rotation of the K heads in place and the
// KV append behind them, all of one position: one launch; anything else: q[i] by itself.  Returns the entries used.
size_t launch_wide_rows(const std::vector<PendOp>& q, size_t i, int* rc) {
  Map* m = get_f32_map(q[i].map_act);
  if (!m) { *rc = ADAMAH_ERR_INVALID; return 1; }
  auto fold = [&]() -> bool {
    if (i + 2 >= q.size()) return false;
    const PendOp &pq = q[i], &pk = q[i + 1], &pc = q[i + 2];
    // (the K rows and the copies may be few enough for a row run of their own: 8 sequences of 32 + 8 heads then took three launches
    // of 5 us)
    if (pq.kind != PK_ROPE || pk.kind != PK_ROPE || pc.kind != PK_ROWCOPY ||
        pk.map_act != pq.map_act || pc.map_act != pq.map_act || pq.a != pq.c || pk.a != pk.c || pk.n != pq.n || pk.eps != pq.eps ||
        pc.k != pk.k || !m->kv16)
      return false;
    const uint64_t q0 = pq.a, q1 = q0 + (uint64_t)pq.rpg * pq.k, k0 = pk.a, k1 = k0 + (uint64_t)pk.rpg * pk.k;
    const uint64_t c0 = m->kv_start, c1 = c0 + m->kv_count;
    auto apart = [](uint64_t a0, uint64_t a1, uint64_t b0, uint64_t b1) { return a1 <= b0 || b1 <= a0; };
    if (!apart(q0, q1, k0, k1) || !apart(q0, q1, c0, c1) || !apart(k0, k1, c0, c1)) return false;
    const uint32_t *spec = res_host(pc.h[0], 2ull * pc.rpg), *base = res_host(pc.h[1], 1);
    if (!spec || !base || !res_u32(pc.h[0], 2ull * pc.rpg)) return false;
    std::vector<uint8_t> seen(pk.rpg, 0);
    for (uint32_t ci = 0; ci < pc.rpg; ci++) {
      const uint64_t so = (uint64_t)base[0] + (uint64_t)spec[2 * ci] * pc.k, s1 = so + pc.k;
      const uint64_t d0 = ((uint64_t)spec[2 * ci + 1] + pc.n) * pc.k, d1 = d0 + pc.k;
      if (d0 < c0 || d1 > c1 || s1 > m->n_elems) return false;
      if (so >= k0 && so < k1) {
        if ((so - k0) % pk.k) return false;
        const uint64_t j = (so - k0) / pk.k;
        if (seen[j]) return false;
        seen[j] = 1;
      } else if (!apart(so, s1, k0, k1) || !apart(so, s1, q0, q1) || !apart(so, s1, c0, c1)) return false;
    }
    k_rope2_copy<<<pq.rpg + pk.rpg + pc.rpg, 256, 0, g.stream>>>((float*)m->buf, pq.a, pq.rpg, pq.k, pk.a, pk.rpg, pk.k, pq.n, pq.eps,
                                                              res_u32(pc.h[0], 2ull * pc.rpg), base[0], pc.rpg, pc.n, m->kv16,
                                                              m->kv_start, m->kv_count);
    count_launch();
    *rc = check_launch();
    return true;
  };
  if (q[i].kind == PK_ROPE && fold()) return 3;
  *rc = launch_wide_alone(q[i], m);
  return 1;
}

}  // namespace adamah

using namespace adamah;

extern "C" {

int map_rmsnorm_dev(uint32_t map_id, uint32_t hs, uint32_t hw, uint32_t hd, uint32_t n_rows, uint32_t dim, float eps) {
  return rmsnorm_impl(map_id, map_id, hs, hw, 0, hd, n_rows, dim, eps, false);
}
int map_rmsnorm_x_dev(uint32_t map_act, uint32_t map_wt, uint32_t hs, uint32_t hw, uint32_t hd, uint32_t n_rows,
                      uint32_t dim, float eps) {
  return rmsnorm_impl(map_act, map_wt, hs, hw, 0, hd, n_rows, dim, eps, false);
}
int map_rmsnorm_add_dev(uint32_t map_id, uint32_t hs, uint32_t hw, uint32_t hr, uint32_t hd, uint32_t n_rows,
                        uint32_t dim, float eps) {
  return rmsnorm_impl(map_id, map_id, hs, hw, hr, hd, n_rows, dim, eps, true);
}

int map_rope_dev(uint32_t map_id, uint32_t hs, uint32_t hd, uint32_t n_tokens, uint32_t n_heads, uint32_t head_dim,
                 uint32_t pos_offset, float freq_base) {
  Map* m = get_f32_map(map_id);
  if (!m) return ADAMAH_ERR_INVALID;
  const uint64_t pairs = (uint64_t)n_tokens * n_heads * (head_dim / 2);
  if (pairs == 0) return ADAMAH_OK;
  if (n_tokens == 1 && can_defer()) {
    // one token with operands known on the host: queue it, it may share a launch with the KV append
    PendOp p;
    p.kind = PK_ROPE; p.map_act = map_id; p.rpg = n_heads; p.k = head_dim; p.n = pos_offset; p.eps = freq_base;
    if (res_scalar(hs, &p.a) && res_scalar(hd, &p.c)) {
      if (row_op_deferrable(p)) { g.pend.push_back(p); return ADAMAH_OK; }
      // more heads than a row run holds (one token of many sequences): queued as well, it may share a launch with
      // the rotation and the KV append next to it
      if (n_heads > ROW_RUN_MAX && (head_dim & 1u) == 0 && in_range(p.a, (uint64_t)n_heads * head_dim, m->n_elems) &&
          in_range(p.c, (uint64_t)n_heads * head_dim, m->n_elems) && tuning("ADAMAH_ROWS_WIDE", 1) != 0) {
        p.op = 1u; p.h[0] = hs; p.h[1] = hd;
        g.pend.push_back(p);
        return ADAMAH_OK;
      }
    }
  }
  flush_pending();
  const uint32_t *ls = res_u32(hs, n_tokens), *ld = res_u32(hd, n_tokens);
  if (!ls || !ld) return ADAMAH_ERR_INVALID;
  k_rope<<<cdiv(pairs, 256), 256, 0, g.stream>>>((float*)m->buf, ls, ld, n_tokens, n_heads, head_dim, pos_offset,
                                                  freq_base, m->n_elems);
  count_launch();
  return check_launch();
}

int map_qk_norm_rope_x_dev(uint32_t map_act, uint32_t map_wt, uint32_t hqs, uint32_t hqw, uint32_t hks, uint32_t hkw,
                           uint32_t hdst, uint32_t q_rows, uint32_t q_dim, uint32_t k_rows, uint32_t k_dim,
                           uint32_t pos_offset, float freq_base) {
  Map* ma = get_f32_map(map_act);
  Map* mw = get_f32_map(map_wt);
  if (!ma || !mw) return ADAMAH_ERR_INVALID;
  if (q_rows + k_rows == 0) return ADAMAH_OK;
  if (map_act == map_wt && can_defer()) {
    PendOp p;
    p.kind = PK_QKNR; p.map_act = map_act; p.map_wt = map_wt; p.rpg = q_rows; p.k = q_dim; p.op = k_rows; p.d = k_dim;
    p.n = pos_offset; p.eps = freq_base;
    p.h[0] = hqs; p.h[1] = hqw; p.h[2] = hks; p.h[3] = hkw; p.h[4] = hdst;
    if (row_op_deferrable(p)) { g.pend.push_back(p); return ADAMAH_OK; }
  }
  flush_pending();
  const uint32_t* one = res_u32(hdst, 1);
  const uint32_t *lqs = q_rows ? res_u32(hqs, q_rows) : one, *lqw = q_rows ? res_u32(hqw, q_rows) : one;
  const uint32_t *lks = k_rows ? res_u32(hks, k_rows) : one, *lkw = k_rows ? res_u32(hkw, k_rows) : one;
  if (!one || !lqs || !lqw || !lks || !lkw) return ADAMAH_ERR_INVALID;
  k_qk_norm_rope<<<q_rows + k_rows, 256, 0, g.stream>>>((float*)ma->buf, (const float*)mw->buf, lqs, lqw, lks, lkw, one,
                                                        q_rows, q_dim, k_rows, k_dim, pos_offset, freq_base,
                                                        ma->n_elems, mw->n_elems);
  count_launch();
  return check_launch();
}

int map_row_copy_offset_dev(uint32_t map_id, uint32_t hspec, uint32_t hbase, uint32_t dst_row_offset, uint32_t n_copies,
                            uint32_t row_size) {
  Map* m = get_f32_map(map_id);
  if (!m) return ADAMAH_ERR_INVALID;
  if (n_copies == 0 || row_size == 0) return ADAMAH_OK;
  if (can_defer()) {
    PendOp p;
    p.kind = PK_ROWCOPY; p.map_act = map_id; p.h[0] = hspec; p.h[1] = hbase; p.rpg = n_copies; p.k = row_size;
    p.n = dst_row_offset;
    if (row_op_deferrable(p)) { g.pend.push_back(p); return ADAMAH_OK; }
    if (n_copies > ROW_RUN_MAX && res_host(hspec, 2ull * n_copies) && res_host(hbase, 1) && tuning("ADAMAH_ROWS_WIDE", 1) != 0) {
      p.op = 1u;     // more copies than a row run holds: queued as well (see map_rope_dev); operands checked at launch
      g.pend.push_back(p);
      return ADAMAH_OK;
    }
  }
  flush_pending();
  const uint32_t *spec = res_u32(hspec, 2ull * n_copies), *base = res_u32(hbase, 1);
  if (!spec || !base) return ADAMAH_ERR_INVALID;
  k_row_copy<<<cdiv((uint64_t)n_copies * row_size, 256), 256, 0, g.stream>>>(
      (float*)m->buf, spec, base, n_copies, row_size, dst_row_offset, m->n_elems, m->kv16, m->kv_start, m->kv_count);
  count_launch();
  return check_launch();
}
int map_row_copy_dev(uint32_t map_id, uint32_t hspec, uint32_t hbase, uint32_t n_copies, uint32_t row_size) {
  return map_row_copy_offset_dev(map_id, hspec, hbase, 0, n_copies, row_size);
}

int adamah_hip_rope_append_rows_dev(uint32_t map_id, uint32_t q, uint32_t q_step, uint32_t q_heads, uint32_t k, uint32_t k_step,
                                    uint32_t k_heads, uint32_t v, uint32_t v_step, uint32_t head_dim, uint32_t n_tok, uint32_t n_seq,
                                    const uint32_t* k_cache, const uint32_t* v_cache, uint32_t head_step, uint32_t pos0, float freq_base,
                                    uint32_t rotate) {
  Map* m = get_f32_map(map_id);
  if (!m) return ADAMAH_ERR_INVALID;
  if (n_tok == 0 || n_seq == 0) return ADAMAH_OK;
  // What is read and what is written: rows of Q, K and V, and of each cache the rows of a head.  All of them lie in the map, a
  // token's heads within its row, and no two of them touch
  const uint64_t rows = (uint64_t)n_tok * n_seq, D = head_dim, last = rows - 1, qw = (uint64_t)q_heads * D, kw = (uint64_t)k_heads * D;
  if (!k_cache || !v_cache || D == 0 || (D & 1u) || D > 4096u || k_heads == 0 || n_tok > 0x7FFFFFFFu || k_step < kw || v_step < kw ||
      (rotate && (q_heads == 0 || q_step < qw)) || (k_heads > 1 && head_step < ((uint64_t)pos0 + n_tok) * D))
    return ADAMAH_ERR_INVALID;
  std::vector<std::pair<uint64_t, uint64_t>> used;
  if (rotate) used.push_back({q, q + last * q_step + qw});
  used.push_back({k, k + last * k_step + kw});
  used.push_back({v, v + last * v_step + kw});
  for (uint32_t s = 0; s < n_seq; s++)
    for (const uint32_t c : {k_cache[s], v_cache[s]})
      for (uint32_t h = 0; h < k_heads; h++) {
        const uint64_t at = c + (uint64_t)h * head_step + (uint64_t)pos0 * D;
        used.push_back({at, at + (uint64_t)n_tok * D});
      }
  for (const auto& u : used) if (u.second > m->n_elems) return ADAMAH_ERR_INVALID;
  std::sort(used.begin(), used.end());
  for (size_t i = 1; i < used.size(); i++) if (used[i].first < used[i - 1].second) return ADAMAH_ERR_INVALID;
  flush_pending();
  uint64_t starts = (uint64_t)k | v | k_step | v_step | (D >> 1) | (m->kv16 ? m->kv_start | m->kv_count : 0u) | (k_heads > 1 ? head_step : 0u) |
                    (rotate ? q | q_step : 0u);
  for (uint32_t s = 0; s < n_seq; s++) starts |= k_cache[s] | v_cache[s];
  for (uint32_t s0 = 0; s0 < n_seq; s0 += APPEND_SEQS) {
    const uint32_t part = std::min(n_seq - s0, APPEND_SEQS);
    const uint64_t row = (uint64_t)s0 * n_tok;
    AppendRows a = {q + row * q_step, k + row * k_step, v + row * v_step, q_step, q_heads, k_step, k_heads, v_step, head_dim,
                    n_tok, head_step, pos0, rotate, freq_base, {}, {}};
    for (uint32_t s = 0; s < part; s++) { a.kc[s] = k_cache[s0 + s]; a.vc[s] = v_cache[s0 + s]; }
#define APPEND(W) k_rope_append_rows<W><<<dim3(n_tok, part), 256, D * sizeof(float), g.stream>>>((float*)m->buf, a, m->kv16, m->kv_start, m->kv_count)
    if (starts & 3u) APPEND(1); else APPEND(4);
#undef APPEND
    count_launch();
  }
  return check_launch();
}

int adamah_qk_norm_rope_rows_dev(uint32_t map_act, uint32_t map_wt, const uint32_t* q_src_handles, uint32_t locs_q_wt,
                                 const uint32_t* k_src_handles, uint32_t locs_k_wt, const uint32_t* dst_handles,
                                 uint32_t m, uint32_t q_rows, uint32_t q_dim, uint32_t k_rows, uint32_t k_dim,
                                 uint32_t pos0, float freq_base) {
  if (m == 0) return ADAMAH_OK;
  if (!q_src_handles || !k_src_handles || !dst_handles) return ADAMAH_ERR_INVALID;
  int rc = ADAMAH_OK;
  Map* ma = get_f32_map(map_act);
  if (ma && map_act == map_wt && launch_qk_rows(ma, q_src_handles, locs_q_wt, k_src_handles, locs_k_wt, dst_handles, m, q_rows, q_dim, k_rows,
                                                k_dim, pos0, freq_base, &rc))
    return rc;
  for (uint32_t t = 0; t < m; t++) {
    const int r = map_qk_norm_rope_x_dev(map_act, map_wt, q_src_handles[t], locs_q_wt, k_src_handles[t], locs_k_wt,
                                         dst_handles[t], q_rows, q_dim, k_rows, k_dim, pos0 + t, freq_base);
    if (r != ADAMAH_OK) return r;
  }
  return ADAMAH_OK;
}

}  // extern "C"
