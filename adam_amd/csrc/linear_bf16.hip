// y = W . f(x) over bfloat16 weight maps, f a grouped RMSNorm (with weight and gate; of one row or of the sum of a row and
// a normed one) or nothing.
//
//   one row      k_gemv_bf16: f is computed by every workgroup while it stages x in LDS (float32), weights stream
//                through registers, float32 multiply-adds; store, add to the residual, gate / up pairs combined, or
//                store + best row of the workgroup (arg-max)
//   2..32 rows   bf16 matrix instructions straight from memory, K split over the waves of a workgroup: k_linear_few, a workgroup a
//                CU with the tokens in its registers, where those hold them; k_linear_skinny for shorter and longer rows
//   more rows    k_linear_tiled<BM, BN, ...>: bf16 matrix instructions over a ring of LDS tiles filled by direct-to-LDS loads
//   float32 operand map: the same tiles over three bfloat16 pieces of each row (k_split_rows); short rows: k_linear_f32, the
//                float32 matrix instruction over the widened weights
// Rows of more than one token pass through the operand map (bf16 or float32, rows k_stride apart, zero beyond k):
// k_operand_rows writes f(x) there, unless the producer already did.
#include "linear_common.h"
#include <algorithm>

namespace adamah {

#define LIN_MAX_GROUPS 1024u
#define LIN_MAX_K 32768u
#define NEG_MAX_F (-3.402823466e+38f)

int scratch_need(Scratch& s, size_t bytes) {
  if (bytes <= s.cap) return ADAMAH_OK;
  hipStreamSynchronize(g.stream);
  layout_changed();
  if (s.p) hipFree(s.p);
  s.p = nullptr; s.cap = 0;
  const size_t cap = std::max<size_t>(bytes, (size_t)1 << 20);
  if (hipMalloc((void**)&s.p, cap) != hipSuccess) { (void)hipGetLastError(); return ADAMAH_ERR_MEMORY; }
  s.cap = cap;
  return ADAMAH_OK;
}
void scratch_free(Scratch& s) {
  if (s.p) hipFree(s.p);
  s.p = nullptr; s.cap = 0;
}

// Sum over a workgroup of NW waves; sh: NW floats that no earlier sum still reads.
template <int NW>
__device__ __forceinline__ float block_sum(float v, float* sh) {
  v = wave_add(v);
  if ((threadIdx.x & 63u) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  v = 0.f;
#pragma unroll
  for (int w = 0; w < NW; w++) v += sh[w];
  return v;
}
// Root mean squares of the row's groups -> inv (with a barrier behind them).
template <int NT, class Val>
__device__ __forceinline__ void group_inverse(uint32_t k, uint32_t groups, float eps, float* inv, float* part, Val val) {
  constexpr uint32_t NW = NT / 64;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, gs = k / groups;
  if (groups >= NW) {
    for (uint32_t gi = wave; gi < groups; gi += NW) {
      float ss = 0.f;
      for (uint32_t i = lane; i < gs; i += 64u) { const float v = val(gi * gs + i); ss = fmaf(v, v, ss); }
      ss = wave_add(ss);
      if (lane == 0) inv[gi] = 1.0f / sqrtf(ss / (float)gs + eps);
    }
    __syncthreads();
  } else {                                    // fewer groups than waves: `sub` waves share a group
    const uint32_t sub = NW / groups, gi = wave / sub, sp = wave % sub;
    float ss = 0.f;
    if (gi < groups)
      for (uint32_t i = sp * 64u + lane; i < gs; i += sub * 64u) { const float v = val(gi * gs + i); ss = fmaf(v, v, ss); }
    ss = wave_add(ss);
    if (lane == 0) part[wave] = ss;
    __syncthreads();
    if (tid < groups) {
      float t = 0.f;
      for (uint32_t j = 0; j < sub; j++) t += part[tid * sub + j];
      inv[tid] = 1.0f / sqrtf(t / (float)gs + eps);
    }
    __syncthreads();
  }
}
// f(x) of one row by a workgroup of NT threads; put(i, value) for i in [0, k_stride).  first: this workgroup also stores
// what the spec wants kept.  put4(c, values): elements 4 c .. 4 c + 3.  inv: LDS, LIN_MAX_GROUPS floats, part: LDS, NT / 16
// floats.  WIDE: for rows of several floats a thread; without it the code is short and needs fewer registers, which is what
// counts where a thread has one (2048 rows of 64: 4.6 us, with it 5.4).  path: operand_path of the spec.  ahead(): called once,
// behind the row's first loads -- loads arrive in order, and what is asked for there (the first weights) must not hold the row up.
enum { ROW_ANY = 0, ROW_NORM = 1, ROW_BRANCH = 2, ROW_PLAIN = 3 };      // NORM, PLAIN: four elements a load; BRANCH: one
static uint32_t operand_path(const LinSpec& s, uint32_t nt) {
  if (s.branched) return s.k <= 8u * nt ? ROW_BRANCH : ROW_ANY;
  if (((s.src | s.src_stride | s.k | (s.kept ? s.keep | s.keep_stride : 0u)) & 3u) != 0u) return ROW_ANY;
  if (!s.groups) return ROW_PLAIN;
  const uint32_t gl = s.k / s.groups >> 2;                   // lanes (of four elements) a group has
  return s.k <= 16u * nt && (!s.gate_act || ((s.gate | s.gate_stride) & 3u) == 0u) && (!s.wt_len || ((s.wt | s.wt_len) & 3u) == 0u) &&
         (s.k / s.groups & 3u) == 0u && (s.groups == 1u || (gl & 63u) == 0u || (gl < 64u && (gl & (gl - 1u)) == 0u)) ? ROW_NORM : ROW_ANY;
}
// What a row is found by, apart from the spec: it is in registers when a wave starts, the spec's fields are a trip to memory (and
// loaded where they are used: a copy of the spec would load them all first).  mode: below; at: the weight's place, of a
// branched row the branch's weight's.
struct RowArgs { uint32_t src, k, kp, branch, at, mode, row, src_stride, branch_stride, gate_stride, res_stride, keep_stride; };
#define MODE_GROUPS(m) ((m) & 2047u)
#define MODE_BRANCHED(m) ((m) >> 11 & 3u)
#define MODE_GATED(m) ((m) >> 13 & 1u)
#define MODE_PATH(m) ((m) >> 14 & 3u)
#define MODE_WT(m) ((m) >> 16 & 1u)                  // there is a weight
#define MODE_WHOLE(m) ((m) >> 17 & 1u)               // as long as the row
#define MODE_GL(m) ((m) >> 18)                       // lanes (of four elements) a group has
static uint32_t operand_mode(const LinSpec& s, uint32_t nt) {
  return s.groups | s.branched << 11 | (s.gate_act ? 1u << 13 : 0u) | operand_path(s, nt) << 14 | (s.wt_len ? 1u << 16 : 0u) | (s.wt_len == s.k ? 1u << 17 : 0u) |
         (s.groups ? s.k / s.groups >> 2 : 64u) << 18;
}
template <int NT, bool WIDE, class Put, class Put4, class Ahead>
__device__ __forceinline__ void operand_row(const RowArgs& r, const LinSpec& s, float* act, bool first, float* inv, float* part, Put put, Put4 put4, Ahead ahead) {
  const uint32_t tid = threadIdx.x, mode = r.mode, path = MODE_PATH(mode), gl = MODE_GL(mode);
  const float* x = act + r.src + (uint64_t)r.row * r.src_stride;
  const auto keep = [&] { return act + s.keep + (uint64_t)r.row * r.keep_stride; };
  const auto kept = [&] { return first && s.kept; };
  const auto gate_act = [&] { return MODE_GATED(mode) ? s.gate_act : 0u; };
  const auto weight = [&] { return act + (MODE_BRANCHED(mode) ? s.wt : r.at); };
  if (WIDE && path == ROW_BRANCH) {
    // x + the branch's row behind a norm of its own, eight elements a thread, everything asked for at once (past the end: the
    // last one again, whose square counts for nothing)
    constexpr int R = 8;
    const float *b = act + r.branch + (uint64_t)r.row * r.branch_stride, *bw = act + r.at;
    float xv[R], bv[R], wv[R], nv[R];
#pragma unroll
    for (int j = 0; j < R; j++) {
      if ((uint32_t)j * NT >= r.k) break;
      const uint32_t i = min(tid + (uint32_t)j * NT, r.k - 1u);
      xv[j] = x[i]; bv[j] = b[i]; wv[j] = bw[i];
    }
    ahead();
    if (MODE_WT(mode)) {
      const float* wt = weight();
#pragma unroll
      for (int j = 0; j < R; j++) {
        if ((uint32_t)j * NT >= r.k) break;
        nv[j] = wt[min(tid + (uint32_t)j * NT, r.k - 1u)];
      }
    }
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < R; j++) {
      if ((uint32_t)j * NT >= r.k) break;
      ss = tid + (uint32_t)j * NT < r.k ? fmaf(bv[j], bv[j], ss) : ss;
    }
    const float ib = 1.0f / sqrtf(block_sum<NT / 64>(ss, part) / (float)r.k + s.eps);
    ss = 0.f;
#pragma unroll
    for (int j = 0; j < R; j++) {
      if ((uint32_t)j * NT >= r.k) break;
      xv[j] = fmaf(bv[j] * ib, s.wt_add + wv[j], xv[j]);
      ss = tid + (uint32_t)j * NT < r.k ? fmaf(xv[j], xv[j], ss) : ss;
    }
    const float ix = 1.0f / sqrtf(block_sum<NT / 64>(ss, part + NT / 64) / (float)r.k + s.eps);
    const bool keeps = kept();
#pragma unroll
    for (int j = 0; j < R; j++) {
      const uint32_t i = tid + (uint32_t)j * NT;
      if (i >= r.k) break;
      if (first && MODE_BRANCHED(mode) == 2u) act[s.res_out + (uint64_t)r.row * r.res_stride + i] = xv[j];
      float v = xv[j] * ix;
      if (MODE_WT(mode)) v *= s.wt_add + nv[j];
      if (keeps) keep()[i] = v;
      put(i, v);
    }
  } else if (MODE_BRANCHED(mode)) {
    ahead();
    // x + the branch's row behind a norm of its own: eight elements a thread stay in registers (a longer row is read again)
    constexpr int R = 8;
    const float *b = act + r.branch + (uint64_t)r.row * r.branch_stride, *bw = act + r.at;
    float* res = act + s.res_out + (uint64_t)r.row * r.res_stride;
    const float* wt = weight();
    const bool keeps = kept();
    float xv[R], bv[R], wv[R], nv[R], ss = 0.f;
#pragma unroll
    for (int j = 0; j < R; j++) {
      const uint32_t i = tid + (uint32_t)j * NT;
      const bool on = i < r.k;
      bv[j] = on ? b[i] : 0.f; xv[j] = on ? x[i] : 0.f; wv[j] = on ? bw[i] : 0.f; nv[j] = on && MODE_WT(mode) ? wt[i] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < R; j++) ss = fmaf(bv[j], bv[j], ss);
    for (uint32_t i = tid + (uint32_t)R * NT; i < r.k; i += NT) ss = fmaf(b[i], b[i], ss);
    const float ib = 1.0f / sqrtf(block_sum<NT / 64>(ss, part) / (float)r.k + s.eps);
    ss = 0.f;
#pragma unroll
    for (int j = 0; j < R; j++) {
      const uint32_t i = tid + (uint32_t)j * NT;
      xv[j] = fmaf(bv[j] * ib, s.wt_add + wv[j], xv[j]);
      if (i < r.k) ss = fmaf(xv[j], xv[j], ss);
    }
    const auto sum_at = [&](uint32_t i) { return fmaf(b[i] * ib, s.wt_add + bw[i], x[i]); };
    for (uint32_t i = tid + (uint32_t)R * NT; i < r.k; i += NT) { const float v = sum_at(i); ss = fmaf(v, v, ss); }
    const float ix = 1.0f / sqrtf(block_sum<NT / 64>(ss, part + NT / 64) / (float)r.k + s.eps);
    const auto done = [&](uint32_t i, float v, float w) {
      if (first && MODE_BRANCHED(mode) == 2u) res[i] = v;
      v *= ix;
      if (MODE_WT(mode)) v *= s.wt_add + w;
      if (keeps) keep()[i] = v;
      put(i, v);
    };
#pragma unroll
    for (int j = 0; j < R; j++) {
      const uint32_t i = tid + (uint32_t)j * NT;
      if (i < r.k) done(i, xv[j], nv[j]);
    }
    for (uint32_t i = tid + (uint32_t)R * NT; i < r.k; i += NT) done(i, sum_at(i), MODE_WT(mode) ? wt[i] : 0.f);
  } else if (WIDE && path == ROW_NORM) {
    // The row makes one trip: up to four times four elements a thread, everything asked for at once (twelve rows of 4096,
    // one float a load and each pass waiting for the one before: 15.8 us; so: 5.0).  A group is a power of two of
    // neighbouring lanes, or whole waves' worth, whose sums meet in LDS, or all of the row.
    constexpr int R = 4, NW = NT / 64;
    const uint32_t n4 = r.k >> 2, wave = tid >> 6;
    const float *gt = MODE_GATED(mode) ? act + s.gate + (uint64_t)r.row * r.gate_stride : act, *wt = weight();
    f4_t xv[R], gv[R], wv[R];
#pragma unroll
    for (int j = 0; j < R; j++) {
      const uint32_t c = min(tid + (uint32_t)j * NT, n4 - 1u);
      if ((uint32_t)j * NT >= n4) break;
      xv[j] = *(const f4_t*)(x + 4u * c);
      if (MODE_GATED(mode)) gv[j] = *(const f4_t*)(gt + 4u * c);
      if (MODE_WT(mode)) wv[j] = *(const f4_t*)(wt + (MODE_WHOLE(mode) ? 4u * c : 4u * c % s.wt_len));
    }
    ahead();
    float ss[R];
#pragma unroll
    for (int j = 0; j < R; j++) {
      const uint32_t c = tid + (uint32_t)j * NT;
      ss[j] = 0.f;
      if (c >= n4) continue;
      if (gate_act() == 3u)
#pragma unroll
        for (int e = 0; e < 4; e++) xv[j][e] *= silu_f(gv[j][e]);
#pragma unroll
      for (int e = 0; e < 4; e++) ss[j] = fmaf(xv[j][e], xv[j][e], ss[j]);
    }
    float scale[R];
    const float n = (float)(4u * gl);
    if (gl < 64u && MODE_GROUPS(mode) != 1u) {
#pragma unroll
      for (int j = 0; j < R; j++) {
        if ((uint32_t)j * NT >= n4) break;
        for (uint32_t o = gl >> 1; o > 0; o >>= 1) ss[j] += __shfl_xor(ss[j], (int)o, 64);
        scale[j] = 1.0f / sqrtf(ss[j] / n + s.eps);
      }
    } else {
      const uint32_t nb = (gl + 63u) >> 6;
#pragma unroll
      for (int j = 0; j < R; j++) {
        if ((uint32_t)j * NT >= n4) break;
        const float t = wave_add(ss[j]);
        if ((tid & 63u) == 0u) part[j * NW + wave] = t;
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < R; j++) {
        if ((uint32_t)j * NT >= n4) break;                   // (all lanes or none: they add up together)
        if (j > 0 && MODE_GROUPS(mode) == 1u) { scale[j] = scale[0]; continue; }
        // (read a partial sum a lane, added up one behind the other)
        const uint32_t lane = tid & 63u, b0 = ((uint32_t)j * NW + wave) / nb * nb;
        const uint32_t own = __float_as_uint(part[min(b0 + min(lane, nb - 1u), (uint32_t)(R * NW) - 1u)]);
        float t = 0.f;
#pragma unroll 8
        for (uint32_t b = 0; b < nb; b++) t += __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)own, (int)b));
        scale[j] = 1.0f / sqrtf(t / n + s.eps);
      }
    }
#pragma unroll
    for (int j = 0; j < R; j++) {
      const uint32_t c = tid + (uint32_t)j * NT;
      if (c >= n4) break;
      f4_t v = xv[j];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        v[e] *= scale[j];
        if (MODE_WT(mode)) v[e] *= s.wt_add + wv[j][e];
        if (gate_act() == 1u) v[e] *= sigmoid_f(gv[j][e]);
        else if (gate_act() == 2u) v[e] *= silu_f(gv[j][e]);
      }
      if (kept()) *(f4_t*)(keep() + 4u * c) = v;
      put4(c, v);
    }
  } else if (MODE_GROUPS(mode)) {
    ahead();
    const uint32_t gs = r.k / MODE_GROUPS(mode);
    const float *gt = act + s.gate + (uint64_t)r.row * r.gate_stride, *wt = weight();
    const bool keeps = kept();
    if (gate_act() == 3u) group_inverse<NT>(r.k, MODE_GROUPS(mode), s.eps, inv, part, [&](uint32_t i) { return x[i] * silu_f(gt[i]); });
    else group_inverse<NT>(r.k, MODE_GROUPS(mode), s.eps, inv, part, [&](uint32_t i) { return x[i]; });
    for (uint32_t i = tid; i < r.k; i += NT) {
      float v = x[i];
      if (gate_act() == 3u) v *= silu_f(gt[i]);
      v *= inv[i / gs];
      if (MODE_WT(mode)) v *= s.wt_add + wt[MODE_WHOLE(mode) ? i : i % s.wt_len];
      if (gate_act() == 1u) v *= sigmoid_f(gt[i]);
      else if (gate_act() == 2u) v *= silu_f(gt[i]);
      if (keeps) keep()[i] = v;
      put(i, v);
    }
  } else if (WIDE && path == ROW_PLAIN) {
    constexpr int R = 4;                                     // of the row; a longer one's rest behind ahead()
    const uint32_t n4 = r.k >> 2;
    f4_t v[R];
#pragma unroll
    for (int j = 0; j < R; j++) {
      if ((uint32_t)j * NT >= n4) break;
      v[j] = *(const f4_t*)(x + 4u * min(tid + (uint32_t)j * NT, n4 - 1u));
    }
    ahead();
    const auto done = [&](uint32_t c, f4_t v) {
      if (kept()) *(f4_t*)(keep() + 4u * c) = v;
      put4(c, v);
    };
#pragma unroll
    for (int j = 0; j < R; j++) {
      const uint32_t c = tid + (uint32_t)j * NT;
      if (c < n4) done(c, v[j]);
    }
#pragma unroll 4
    for (uint32_t c = tid + (uint32_t)R * NT; c < n4; c += NT) done(c, *(const f4_t*)(x + 4u * c));
  } else {
    ahead();
    const bool keeps = kept();
    for (uint32_t i = tid; i < r.k; i += NT) {
      if (keeps) keep()[i] = x[i];
      put(i, x[i]);
    }
  }
  for (uint32_t i = r.k + tid; i < r.kp; i += NT) put(i, 0.f);
}

template <class T, int NT, bool WIDE>
__global__ void __launch_bounds__(NT)
k_operand_rows(float* act, T* __restrict__ dst, const uint32_t* __restrict__ row_idx, uint32_t src, uint32_t src_stride, uint32_t k, uint32_t kp, uint32_t mode,
               uint32_t at, uint32_t branch, const LinSpec s) {
  __shared__ float inv[LIN_MAX_GROUPS];
  __shared__ float part[NT / 16];
  typedef T t4 __attribute__((ext_vector_type(4)));
  T* d = dst + (uint64_t)blockIdx.x * kp;
  const RowArgs r = {src, k, kp, branch, at, mode, row_idx ? row_idx[blockIdx.x] : blockIdx.x, src_stride, s.branch_stride, s.gate_stride, s.res_stride, s.keep_stride};
  operand_row<NT, WIDE>(r, s, act, true, inv, part, [&](uint32_t i, float v) { d[i] = (T)v; },
                        [&](uint32_t c, f4_t v) { *(t4*)(d + 4u * c) = (t4){(T)v[0], (T)v[1], (T)v[2], (T)v[3]}; }, [] {});
}
// Long rows, few of them: a row's latency is the launch's, so 1024 threads a row; many rows fill the CUs with 256 each, and
// rows of one float a thread have nothing to gain (300 rows of 64 on the wide form with 1024 threads: 5.7 us, so: 3.6; 12 rows
// of 100: 4.7 and 3.6).
// Rows with a branch have a form of their own, eight elements a thread: the threads that hold the row, and none of the wide
// form's registers (with the rule of the others, in us, a product of 16 columns behind them: 300 rows of 2048 20.8, so: 11.9;
// 2048 rows of 4096 43.6 and 34.4; 2 rows of 4096 12.0 and 10.5; 600 rows of 8192 41.4 and 31.8).
template <class T>
static void operand_rows(const LinSpec& s, float* act, T* dst, const uint32_t* row_idx, uint32_t rows) {
#define ROWS(NT, WIDE) k_operand_rows<T, NT, WIDE><<<rows, NT, 0, g.stream>>>(act, dst, row_idx, s.src, s.src_stride, s.k, s.k_stride, operand_mode(s, NT), \
                                                                              s.branched ? s.branch_wt : s.wt, s.branch, s)
  if (s.k <= 256u || (s.branched && s.k <= 2048u)) ROWS(256, false);
  else if (s.branched && s.k <= 4096u) ROWS(512, false);
  else if (s.branched) ROWS(1024, false);
  else if (s.k > 1024u && rows <= 2u * (uint32_t)g.n_cu) ROWS(1024, true);
  else ROWS(256, true);
#undef ROWS
  count_launch();
}

// ---- one row ------------------------------------------------------------------------------------------------------
// A wave takes R matrix rows at a time (two; for gate / up pairs row 32 b + j and its partner 16 further on) and walks
// along K, 512 columns a step, U steps in flight.  x in LDS as two planes (elements 0..3 / 4..7 of every eight), so that
// a lane's two 16-byte reads are conflict free.
// What bounds it is the weights' way in and, for the smaller matrices, what a workgroup does before it can use them: x and the
// first weights behind it are asked for from the leading arguments alone (in registers when a wave starts; the spec is a
// trip to memory, 0.5 us), sums of a norm stay in the vector unit.  us, weights cold, before and so: 2048 x 2048 5.0 and 4.1,
// 2048 x 4096 7.3 and 6.3, behind a norm 9.3 and 7.8, 4096 x 4096 behind a norm 11.8 and 9.4, 10304 x 2048 behind a branch
// 13.8 and 12.0, 4131 x 2048 (pairs, a tail) 10.4 and 8.0, 28672 x 4096 (pairs) 44.9 and 43.2, 4096 x 14336 25.4 and 24.0.
// A norm's sums keep the order that they had before (partial sums of the waves in turn; a branched row's columns by thread): four
// neighbours a load and the partial sums in pairs would take 0.2 us less, and behind a router that is another choice of experts.
enum { LEPI_STORE = 0, LEPI_ADD = 1, LEPI_PAIR = 2, LEPI_ARGMAX = 3 };
template <int EPI, int U, int R>
__global__ void __launch_bounds__(512)
k_gemv_bf16(const bf16_t* __restrict__ W, float* act, const uint32_t* __restrict__ row_idx, uint32_t kp, uint32_t n, uint32_t pairs, uint32_t src,
            uint32_t k_in, uint32_t mode, uint32_t branch, uint32_t at, const LinSpec s, float* best_val, uint32_t* best_idx) {
  static_assert(R == 2 || EPI == LEPI_STORE || EPI == LEPI_ADD, "one row");
  extern __shared__ __attribute__((aligned(16))) float xs[];
  __shared__ float inv[LIN_MAX_GROUPS];
  __shared__ float part[32];
  __shared__ float bv[8];
  __shared__ uint32_t bi[8];
  RowArgs ra = {src, k_in, kp, branch, at, mode, 0u, 0u, 0u, 0u, 0u, 0u};
  if (row_idx) {                                             // (an asm: not to be loaded, and waited for, where there is no list)
    ra.row = row_idx[0];
    ra.src_stride = s.src_stride; ra.branch_stride = s.branch_stride; ra.gate_stride = s.gate_stride; ra.res_stride = s.res_stride; ra.keep_stride = s.keep_stride;
    asm volatile("" : "+s"(ra.src_stride), "+s"(ra.branch_stride), "+s"(ra.gate_stride), "+s"(ra.res_stride), "+s"(ra.keep_stride));
  }
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, half = kp >> 1, n_tasks = R == 1 ? n : pairs + ((n - 2u * pairs + 1u) >> 1);
  // pairs: tasks of gate / up; the tail's rows come two a task behind them
  auto rows_of = [&](uint32_t task, uint32_t (&r)[R]) {
    if constexpr (R == 1) r[0] = task;
    else if (EPI == LEPI_PAIR && task < pairs) { r[0] = (task >> 4) * 32u + (task & 15u); r[1] = r[0] + 16u; }
    else { r[0] = task * 2u; r[1] = min(r[0] + 1u, n - 1u); }     // (2 pairs + 2 (task - pairs) for the tail)
  };
  uint4 p[R][U];
  auto fetch = [&](const uint32_t (&r)[R], uint32_t k0) {    // (past the row's end its last columns, which nothing uses)
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint32_t k = min(k0 + 512u * u, kp - 8u);
#pragma unroll
      for (int q = 0; q < R; q++) p[q][u] = *(const uint4*)(W + (uint64_t)r[q] * kp + k);
    }
  };
  // the first weights are on their way while x is staged, each further step's under the products of the one before
  uint32_t task = blockIdx.x * 8u + wave, k0 = lane * 8u, r[R];
  rows_of(min(task, n_tasks - 1u), r);
  operand_row<512, (U > 1)>(ra, s, act, blockIdx.x == 0u, inv, part,
                   [&](uint32_t i, float v) { xs[((i >> 2) & 1u) * half + (i >> 3) * 4u + (i & 3u)] = v; },
                   [&](uint32_t c, f4_t v) { *(f4_t*)(xs + (c & 1u) * half + (c >> 1) * 4u) = v; },
                   [&] { fetch(r, k0); __builtin_amdgcn_sched_barrier(0); });
  __syncthreads();
  float top = NEG_MAX_F, a[R] = {};
  uint32_t top_i = 0xFFFFFFFFu;
  while (task < n_tasks) {
    uint4 cur[R][U];
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int q = 0; q < R; q++) cur[q][u] = p[q][u];
    const bool last = k0 - lane * 8u + 512u * U >= kp;              // of these rows
    const uint32_t next = last ? task + gridDim.x * 8u : task, kn = last ? lane * 8u : k0 + 512u * U, c0 = r[0];
    if (next < n_tasks) {
      if (last) rows_of(next, r);
      fetch(r, kn);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint32_t k = k0 + 512u * u;
      if (k >= kp) break;
      const float4 lo = *(const float4*)(xs + (k >> 1)), hi = *(const float4*)(xs + half + (k >> 1));
#pragma unroll
      for (int q = 0; q < R; q++) {
        const uint4 w = cur[q][u];
        a[q] = fmaf(bf_lo(w.x), lo.x, a[q]); a[q] = fmaf(bf_hi(w.x), lo.y, a[q]); a[q] = fmaf(bf_lo(w.y), lo.z, a[q]); a[q] = fmaf(bf_hi(w.y), lo.w, a[q]);
        a[q] = fmaf(bf_lo(w.z), hi.x, a[q]); a[q] = fmaf(bf_hi(w.z), hi.y, a[q]); a[q] = fmaf(bf_lo(w.w), hi.z, a[q]); a[q] = fmaf(bf_hi(w.w), hi.w, a[q]);
      }
    }
    if (last) {
#pragma unroll
      for (int q = 0; q < R; q++) a[q] = wave_add(a[q]);
      if (EPI == LEPI_PAIR && task < pairs) {
        if (lane == 0) act[s.out + task] = silu_f(a[0]) * a[R - 1];
      } else {
        const uint32_t i = c0 + lane;
        float y = lane ? a[R - 1] : a[0];
        if (lane < (uint32_t)R && i < n) {
          if (s.biased) y += act[s.bias + i];
          float* d = EPI == LEPI_PAIR ? act + s.tail_out + (i - 2u * pairs) : act + s.out + i;
          *d = EPI == LEPI_ADD ? *d + y : y;
          if (EPI == LEPI_ARGMAX && !isnan(y) && y > top) { top = y; top_i = i; }
        }
      }
#pragma unroll
      for (int q = 0; q < R; q++) a[q] = 0.f;
    }
    task = next; k0 = kn;
  }
  if (EPI != LEPI_ARGMAX) return;
  const float v1 = __shfl(top, 1, 64);
  const uint32_t i1 = (uint32_t)__shfl((int)top_i, 1, 64);
  if (lane == 0) {
    if (v1 > top || (v1 == top && i1 < top_i)) { top = v1; top_i = i1; }
    bv[wave] = top; bi[wave] = top_i;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 8; w++) if (bv[w] > top || (bv[w] == top && bi[w] < top_i)) { top = bv[w]; top_i = bi[w]; }
    best_val[blockIdx.x] = top; best_idx[blockIdx.x] = top_i;
  }
}
// The one-row head over NR rows at a time (their operand, float32, ready at X): the weights go by once instead of once a row, 32768 x
// 4096 for 16 rows 697 us one by one.  Four matrix rows a wave, so that a value of x read from LDS meets four weights; a result's sums
// are the one-row kernel's, in its order.  32768 x 4096 for eight rows 95 us (55 at a large copy's rate): multiply-adds and memory in
// turn; 115 with loads, maxima and logits under conditions and the rows staged one load at a time.  Rows past the last are zeros;
// the logits at `out` are the row `kept`'s, if it is among them.
template <int NR>
__global__ void __launch_bounds__(512)
k_head_rows(const bf16_t* __restrict__ W, float* act, const LinSpec s, const float* __restrict__ X, uint32_t rows, uint32_t kept, uint32_t n_tasks,
            float* best_val, uint32_t* best_idx) {
  constexpr int U = 2;
  extern __shared__ __attribute__((aligned(16))) float xs[];  // [row][two planes: elements 0..3 / 4..7 of every eight]
  __shared__ float bv[8][NR];
  __shared__ uint32_t bi[8][NR];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, kp = s.k_stride, half = kp >> 1;
  uint4 p[4][U];
  auto fetch = [&](uint32_t task, uint32_t k0) {
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int u = 0; u < U; u++) {
        const uint32_t k = min(k0 + 512u * u, kp - 8u);       // (past the end: not used)
        p[j][u] = *(const uint4*)(W + (uint64_t)min(task * 4u + j, s.n - 1u) * kp + k);
      }
  };
  uint32_t task = blockIdx.x * 8u + wave, k0 = lane * 8u;
  fetch(min(task, n_tasks - 1u), k0);
  for (uint32_t c = threadIdx.x; c < (kp >> 2); c += 512u) {  // the rows' loads all at once
    f4_t v[NR];
#pragma unroll
    for (uint32_t r = 0; r < NR; r++) v[r] = *(const f4_t*)(X + (uint64_t)min(r, rows - 1u) * kp + 4u * c);
#pragma unroll
    for (uint32_t r = 0; r < NR; r++) *(f4_t*)(xs + r * kp + (c & 1u) * half + (c >> 1) * 4u) = r < rows ? v[r] : (f4_t){0, 0, 0, 0};
  }
  __syncthreads();
  float a[NR][4], top[NR];
  uint32_t top_i[NR];
#pragma unroll
  for (int r = 0; r < NR; r++) {
    top[r] = NEG_MAX_F; top_i[r] = 0xFFFFFFFFu;
#pragma unroll
    for (int j = 0; j < 4; j++) a[r][j] = 0.f;
  }
  while (task < n_tasks) {
    uint4 c[4][U];
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int u = 0; u < U; u++) c[j][u] = p[j][u];
    const bool last = k0 - lane * 8u + 512u * U >= kp;        // of these four rows
    const uint32_t next = last ? task + gridDim.x * 8u : task, kn = last ? lane * 8u : k0 + 512u * U;
    if (next < n_tasks) fetch(next, kn);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint32_t k = k0 + 512u * u;
      if (k >= kp) break;
      float w[4][8];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        w[j][0] = bf_lo(c[j][u].x); w[j][1] = bf_hi(c[j][u].x); w[j][2] = bf_lo(c[j][u].y); w[j][3] = bf_hi(c[j][u].y);
        w[j][4] = bf_lo(c[j][u].z); w[j][5] = bf_hi(c[j][u].z); w[j][6] = bf_lo(c[j][u].w); w[j][7] = bf_hi(c[j][u].w);
      }
#pragma unroll
      for (int r = 0; r < NR; r++) {
        const f4_t lo = *(const f4_t*)(xs + r * kp + (k >> 1)), hi = *(const f4_t*)(xs + r * kp + half + (k >> 1));
#pragma unroll
        for (int j = 0; j < 4; j++) {
#pragma unroll
          for (int e = 0; e < 4; e++) a[r][j] = fmaf(w[j][e], lo[e], a[r][j]);
#pragma unroll
          for (int e = 0; e < 4; e++) a[r][j] = fmaf(w[j][4 + e], hi[e], a[r][j]);
        }
      }
    }
    if (last) {
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const uint32_t n = task * 4u + j;
        const float bias = s.biased && n < s.n ? act[s.bias + n] : 0.f;
        float logit = 0.f;
#pragma unroll
        for (int r = 0; r < NR; r++) {
          float y = wave_add(a[r][j]);
          y = s.biased ? y + bias : y;
          a[r][j] = 0.f;
          logit = r == (int)kept ? y : logit;
          const bool above = n < s.n && y > top[r];           // (never a NaN)
          top[r] = above ? y : top[r]; top_i[r] = above ? n : top_i[r];
        }
        if (n < s.n && kept < (uint32_t)NR && lane == 0) act[s.out + n] = logit;
      }
    }
    task = next; k0 = kn;
  }
  if (lane == 0) {
#pragma unroll
    for (int r = 0; r < NR; r++) { bv[wave][r] = top[r]; bi[wave][r] = top_i[r]; }
  }
  __syncthreads();
  if (threadIdx.x < min(rows, (uint32_t)NR)) {
    const uint32_t r = threadIdx.x;
    float v = bv[0][r];
    uint32_t b = bi[0][r];
    for (int w = 1; w < 8; w++) if (bv[w][r] > v || (bv[w][r] == v && bi[w][r] < b)) { v = bv[w][r]; b = bi[w][r]; }
    best_val[r * gridDim.x + blockIdx.x] = v; best_idx[r * gridDim.x + blockIdx.x] = b;
  }
}
// best of n (value, index) pairs, a workgroup a row of them; ties to the lower index -> float(index) at dst_list[row] (or at dst)
__global__ void __launch_bounds__(256)
k_best_pair(const float* __restrict__ val, const uint32_t* __restrict__ idx, uint32_t n, float* dst, const uint32_t* __restrict__ dst_list) {
  val += (uint64_t)blockIdx.x * n; idx += (uint64_t)blockIdx.x * n;
  if (dst_list) dst += dst_list[blockIdx.x];
  __shared__ float sv[4];
  __shared__ uint32_t si[4];
  float v = NEG_MAX_F;
  uint32_t b = 0xFFFFFFFFu;
  for (uint32_t i = threadIdx.x; i < n; i += 256u)
    if (val[i] > v || (val[i] == v && idx[i] < b)) { v = val[i]; b = idx[i]; }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float tv = __shfl_xor(v, o, 64);
    const uint32_t ti = (uint32_t)__shfl_xor((int)b, o, 64);
    if (tv > v || (tv == v && ti < b)) { v = tv; b = ti; }
  }
  if ((threadIdx.x & 63u) == 0) { sv[threadIdx.x >> 6] = v; si[threadIdx.x >> 6] = b; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; w++) if (sv[w] > v || (sv[w] == v && si[w] < b)) { v = sv[w]; b = si[w]; }
    *dst = (float)(b == 0xFFFFFFFFu ? 0u : b);
  }
}
// arg-max of every row of a [rows, n] block.  A row has one workgroup, so its latency counts: sixteen floats a thread asked
// for at once (16 rows of 100000, one float at a time by 256 threads: 36 us; so: 5.1).
template <uint32_t NT>
__global__ void __launch_bounds__(NT)
k_best_row(const float* __restrict__ act, uint64_t src, uint32_t stride, uint32_t n, float* out, const uint32_t* __restrict__ dst) {
  __shared__ float sv[NT / 64u];
  __shared__ uint32_t si[NT / 64u];
  const float* x = act + src + (uint64_t)blockIdx.x * stride;
  float v = NEG_MAX_F;
  uint32_t b = 0xFFFFFFFFu, done = 0;
  if (((src | stride) & 3u) == 0u) {
    constexpr uint32_t U = 4;
    for (; done + 4u * U * NT <= n; done += 4u * U * NT) {
      f4_t t[U];
#pragma unroll
      for (uint32_t u = 0; u < U; u++) t[u] = *(const f4_t*)(x + done + 4u * (u * NT + threadIdx.x));
#pragma unroll
      for (uint32_t u = 0; u < U; u++)
#pragma unroll
        for (uint32_t e = 0; e < 4; e++) if (t[u][e] > v) { v = t[u][e]; b = done + 4u * (u * NT + threadIdx.x) + e; }
    }
  }
#pragma unroll 8
  for (uint32_t i = done + threadIdx.x; i < n; i += NT) { const float t = x[i]; if (t > v) { v = t; b = i; } }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float tv = __shfl_xor(v, o, 64);
    const uint32_t ti = (uint32_t)__shfl_xor((int)b, o, 64);
    if (tv > v || (tv == v && ti < b)) { v = tv; b = ti; }
  }
  if ((threadIdx.x & 63u) == 0) { sv[threadIdx.x >> 6] = v; si[threadIdx.x >> 6] = b; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t w = 1; w < NT / 64u; w++) if (sv[w] > v || (sv[w] == v && si[w] < b)) { v = sv[w]; b = si[w]; }
    out[dst[blockIdx.x]] = (float)(b == 0xFFFFFFFFu ? 0u : b);
  }
}

// ---- results of the matrix-instruction kernels --------------------------------------------------------------------
// Lane l of a 16 x 16 result holds matrix rows (outputs) 4 (l / 16) + 0..3 of token l % 16: one 16-byte (bfloat16:
// 8-byte) access where the rows' places allow it, four narrow ones at a ragged end.
__device__ __forceinline__ void put_out(const LinSpec& s, float* act, uint32_t row, uint32_t n0, f4_t v) {
  float* d = act + s.out + (uint64_t)row * s.out_stride + n0;
  if (((s.out | s.out_stride) & 3u) == 0u && (!s.biased || (s.bias & 3u) == 0u) && n0 + 4u <= s.n) {
    if (s.biased) v += *(const f4_t*)(act + s.bias + n0);
    if (s.epi == 1u) v += *(const f4_t*)d;
    *(f4_t*)d = v;
    return;
  }
  // (a loop for each form: with the form asked for at every value, float32 24 x 1001 x 60 took 4.44 us, so: 4.19)
  if (s.biased) {
#pragma unroll
    for (int i = 0; i < 4; i++) if (n0 + i < s.n) v[i] += act[s.bias + n0 + i];
  }
  if (s.epi == 1u) {
#pragma unroll
    for (int i = 0; i < 4; i++) if (n0 + i < s.n) d[i] += v[i];
  } else {
#pragma unroll
    for (int i = 0; i < 4; i++) if (n0 + i < s.n) d[i] = v[i];
  }
}
// gate rows n0 .. n0 + 3 and their up rows -> the activation's operand rows
template <class T>
__device__ __forceinline__ void put_pair(const LinSpec& s, T* opnd, uint32_t row, uint32_t n0, f4_t gt, f4_t up) {
  const uint32_t c = (n0 >> 5) * 16u + (n0 & 15u);
  typedef T t4 __attribute__((ext_vector_type(4)));
  T* d = opnd + s.out_opnd + (uint64_t)row * s.out_opnd_stride + c;
  t4 y;
#pragma unroll
  for (int i = 0; i < 4; i++) y[i] = (T)(silu_f(gt[i]) * up[i]);
  if (((s.out_opnd | s.out_opnd_stride) & 3u) == 0u && n0 + 4u <= s.n) { *(t4*)d = y; return; }
#pragma unroll
  for (int i = 0; i < 4; i++) if (n0 + i < s.n) d[i] = y[i];
}
// two neighbouring runs of 16 rows of an epi 2 product, from row n0 on: a pair, or two runs of the tail
template <class T>
__device__ __forceinline__ void put_pair_or_tail(const LinSpec& s, float* act, T* opnd, uint32_t row, uint32_t n0, f4_t a, f4_t b) {
  const uint32_t head = s.n - s.tail;
  if (n0 < head) { put_pair(s, opnd, row, n0, a, b); return; }
  float* d = act + s.tail_out + (uint64_t)row * s.tail_stride + (n0 - head);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    if (n0 + i < s.n) d[i] = a[i];
    if (n0 + 16u + i < s.n) d[16 + i] = b[i];
  }
}

// ---- 2 .. 32 rows -------------------------------------------------------------------------------------------------
// Bound by the weights' way in.  A workgroup owns 16 NB matrix rows; its NW waves take 64-column steps of K (a whole line of
// a row) in turn, two of them in flight, and add up through LDS.  12 rows, 4096 x 14336 (117 MB): 57 us with half the CUs
// at work, half lines and few loads in flight, 26.8 now (4.4 TB/s); 24 rows: 68 and 37.
template <int MT, int NB, int NW>
__global__ void __launch_bounds__(64 * NW)
k_linear_skinny(const bf16_t* __restrict__ W, const bf16_t* __restrict__ X, float* act, bf16_t* opnd, const LinSpec s, uint32_t rows) {
  __shared__ f4_t red[NW][NB * MT][64];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, c = lane & 15u, kg = lane >> 4, kp = s.k_stride;
  const uint32_t n0 = blockIdx.x * (16u * NB);
  const bf16_t *wr[NB], *xr[MT];
#pragma unroll
  for (int i = 0; i < NB; i++) wr[i] = W + (uint64_t)min(n0 + 16u * i + c, s.n - 1u) * kp + kg * 8u;
#pragma unroll
  for (int m = 0; m < MT; m++) xr[m] = X + (uint64_t)min(16u * m + c, rows - 1u) * kp + kg * 8u;
  f4_t acc[NB][MT];
#pragma unroll
  for (int i = 0; i < NB; i++)
#pragma unroll
    for (int m = 0; m < MT; m++) acc[i][m] = (f4_t){0, 0, 0, 0};
  uint32_t k = wave * 64u;
  const auto steps = [&](auto n) {
    constexpr int U = decltype(n)::value;
    bf8_t w[U][2][NB], x[U][2][MT];
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int i = 0; i < NB; i++) w[u][h][i] = *(const bf8_t*)(wr[i] + k + 64 * NW * u + 32 * h);
#pragma unroll
        for (int m = 0; m < MT; m++) x[u][h][m] = *(const bf8_t*)(xr[m] + k + 64 * NW * u + 32 * h);
      }
    __builtin_amdgcn_sched_barrier(0);                 // all asked for before the first is waited for
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
          for (int i = 0; i < NB; i++) acc[i][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u][h][i], x[u][h][m], acc[i][m], 0, 0, 0);
    k += 64u * NW * U;
  };
  while (k + 64u * NW < kp) steps(std::integral_constant<int, 2>{});
  if (k < kp) steps(std::integral_constant<int, 1>{});
#pragma unroll
  for (int i = 0; i < NB; i++)
#pragma unroll
    for (int m = 0; m < MT; m++) red[wave][i * MT + m][lane] = acc[i][m];
  __syncthreads();
  const auto sum = [&](uint32_t t) {
    f4_t v = red[0][t][lane];
#pragma unroll
    for (int w = 1; w < NW; w++) v += red[w][t][lane];
    return v;
  };
  if (s.epi == 2u) {
    if constexpr (NB == 2)
      if (wave < MT) {
        const f4_t gt = sum(wave), up = sum(MT + wave);
        const uint32_t row = 16u * wave + c;
        if (row < rows) put_pair_or_tail(s, act, opnd, row, n0 + 4u * kg, gt, up);
      }
  } else if (wave < NB * MT) {
    const f4_t v = sum(wave);
    const uint32_t row = 16u * (wave % MT) + c;
    if (row < rows) put_out(s, act, row, n0 + 16u * (wave / MT) + 4u * kg, v);
  }
}

// Four results of one token, units j0 .. j0 + 3 of a workgroup's own (below end): a unit is a matrix row, of an epi 2 product two of
// them, gate / up or two of the tail.
__device__ __forceinline__ void put_units(const LinSpec& s, float* act, uint32_t row, uint32_t j0, uint32_t end, f4_t v) {
  float* d = act + s.out + (uint64_t)row * s.out_stride + j0;
  if (s.biased) {
#pragma unroll
    for (int i = 0; i < 4; i++) if (j0 + i < end) v[i] += act[s.bias + j0 + i];
  }
  if (s.epi == 1u) {
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] += j0 + i < end ? d[i] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < 4; i++) if (j0 + i < end) d[i] = v[i];
}
typedef uint32_t words_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint32_t pair_row(uint32_t j) { return (j >> 4) * 32u + (j & 15u); }
__device__ __forceinline__ void put_units(const LinSpec& s, float* act, bf16_t* opnd, uint32_t row, uint32_t j0, uint32_t end, f4_t gt, f4_t up) {
  const uint32_t head = s.n - s.tail;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t r = pair_row(j0 + i);
    if (j0 + i >= end || r >= s.n) continue;
    if (r < head) { opnd[s.out_opnd + (uint64_t)row * s.out_opnd_stride + j0 + i] = (bf16_t)(silu_f(gt[i]) * up[i]); continue; }
    float* d = act + s.tail_out + (uint64_t)row * s.tail_stride + (r - head);
    d[0] = gt[i];
    if (r + 16u < s.n) d[16] = up[i];
  }
}

// Rows of 1152 .. 4096 columns.  Bound by the weights' way in.  One workgroup a CU, each an equal share of the units (the kernel above
// put 28672 rows into 896 workgroups, of which three fit a CU: the last 128 ran alone), in passes of 16 matrix rows.  A wave's S steps
// of K are the same in every pass, so its columns of the tokens stay in registers (they were read again for every 32 matrix rows:
// half as many bytes as the weights at 16 tokens, as many at 32), and a step's weights are asked for as soon as its own of the pass
// before (of two passes before where rows are short) have been used: 64 .. 128 KB of a CU in flight throughout, without a wait for
// all of them.  A pass leaves its sums over K in LDS; no barrier before there is no room for more.  What remains is the tokens' way
// in, 128 KB a CU for 16 of 4096 columns: 2 us at the rate of the L2s.
// The order of the sums over K is the other kernel's, to the bit (a router behind them turns another order into another expert): steps of
// K in turn by wave, the waves' sums in order.  ODD: a pass at most, where that kernel has sixteen waves: a wave here has two of them, their
// steps the even and the odd ones of its own.
// us, the kernel above and this one: 12 tokens, 28672 x 4096 (pairs) 54.3 and 41.5 (5.7 TB/s), 12576 x 4096 27.2 and 22, 32768 x 4096 58.2 and
// 48.3, 10304 x 2048 14.4 and 10.3, 2048 x 2048 5.5 and 4.7, 14336 x 2560 (pairs) 18.9 and 16.9; 32 tokens, the same: 68 and 47, 34.3 and
// 26.4, 71.5 and 54.4, 18.6 and 12.9, 7.7 and 6.9, 24.5 and 19.4.
template <int MT, int S, bool ODD>
__global__ void __launch_bounds__(512)
k_linear_few(const bf16_t* __restrict__ W, const bf16_t* __restrict__ X, float* act, bf16_t* opnd, uint32_t kp, uint32_t n, uint32_t rows,
             uint32_t units, uint32_t per, uint32_t pair, const LinSpec s) {
  constexpr int NW = 8, D = S <= 4 && !ODD ? 2 : 1, P = ODD ? 1 : 16 / MT, NS = ODD ? 2 : 1;
  __shared__ f4_t red[P][MT][NS * NW][64];
  const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), c = lane & 15u, kg = lane >> 4;
  const uint32_t begin = blockIdx.x * per, end = min(begin + per, units), passes = ((end - begin + 15u) >> 4) << pair;
  // step u of this wave: columns 64 (wave + 8 u) ..; some waves' last lies beyond the row's end: they read their first again, and `keep` makes zeros of it
  const bool over = 64u * (wave + NW * (S - 1)) >= kp;
  const uint32_t last = over ? 64u * wave : 64u * (wave + NW * (S - 1)), keep = over ? 0u : ~0u;
  const auto kept = [&](bf8_t v) { return __builtin_bit_cast(bf8_t, __builtin_bit_cast(words_t, v) & (words_t){keep, keep, keep, keep}); };
  const auto column = [&](int u) { return u == S - 1 ? last : 64u * (wave + NW * (uint32_t)u); };
  const auto row_of = [&](uint32_t p) {
    const uint32_t j = min(begin + 16u * (p >> pair) + c, end - 1u);
    return W + (uint64_t)min(pair ? pair_row(j) + 16u * (p & 1u) : j, n - 1u) * kp + kg * 8u;
  };
  bf8_t w[D][S][2], x[S][2][MT];
  const auto ask = [&](const bf16_t* r, int d, int u) {
#pragma unroll
    for (int h = 0; h < 2; h++) w[d][u][h] = *(const bf8_t*)(r + column(u) + 32 * h);
  };
  {
    const bf16_t *r = row_of(0), *xr[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) xr[m] = X + (uint64_t)min(16u * m + c, rows - 1u) * kp + kg * 8u;
#pragma unroll
    for (int u = 0; u < S; u++) {
      ask(r, 0, u);
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int m = 0; m < MT; m++) x[u][h][m] = *(const bf8_t*)(xr[m] + column(u) + 32 * h);
    }
    if (D == 2 && passes > 1u) {
      r = row_of(1);
#pragma unroll
      for (int u = 0; u < S; u++) ask(r, D - 1, u);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  uint32_t first = 0;
  const auto sums = [&](uint32_t to) {      // passes first .. to - 1 lie in LDS
    __syncthreads();
    const uint32_t tasks = ((to - first) >> pair) * MT;
    for (uint32_t t = wave; t < tasks; t += NW) {
      const uint32_t m = t % MT, p = (t / MT) << pair, row = 16u * m + c, j0 = begin + 16u * ((first + p) >> pair) + 4u * kg;
      const auto sum = [&](uint32_t q) {
        f4_t v = red[q][m][0][lane];
#pragma unroll
        for (int i = 1; i < NS * NW; i++) v += red[q][m][i][lane];
        return v;
      };
      const f4_t a = sum(p), b = pair ? sum(p + 1u) : a;
      if (row >= rows) continue;
      if (pair) put_units(s, act, opnd, row, j0, end, a, b);
      else put_units(s, act, row, j0, end, a);
    }
  };
  const auto pass = [&](uint32_t p, auto place, auto more) {
    constexpr int d = decltype(place)::value;
    if (p - first == (uint32_t)P) { sums(p); __syncthreads(); first = p; }
    const bf16_t* next = row_of(p + D);
    f4_t acc[NS][MT];
#pragma unroll
    for (int m = 0; m < MT; m++) acc[0][m] = acc[NS - 1][m] = (f4_t){0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < S; u++) {
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int m = 0; m < MT; m++) {
          if (u == S - 1) { w[d][u][h] = kept(w[d][u][h]); x[u][h][m] = kept(x[u][h][m]); }
          acc[u % NS][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[d][u][h], x[u][h][m], acc[u % NS][m], 0, 0, 0);
        }
      if (more) ask(next, d, u);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
      for (int q = 0; q < NS; q++) red[p - first][m][q * NW + wave][lane] = acc[q][m];
  };
  typedef std::integral_constant<int, 0> A;
  typedef std::integral_constant<int, D - 1> B;
  uint32_t p = 0;
  if (D == 2) {
    for (; p + 3u < passes; p += 2u) { pass(p, A{}, std::true_type{}); pass(p + 1u, B{}, std::true_type{}); }
    if (p + 2u < passes) { pass(p, A{}, std::true_type{}); pass(p + 1u, B{}, std::false_type{}); pass(p + 2u, A{}, std::false_type{}); }
    else { pass(p, A{}, std::false_type{}); if (p + 1u < passes) pass(p + 1u, B{}, std::false_type{}); }
  } else {
    for (; p + 1u < passes; p++) pass(p, A{}, std::true_type{});
    pass(p, A{}, std::false_type{});
  }
  sums(passes);
}

// ---- tiles --------------------------------------------------------------------------------------------------------
// Shares of K (part): workgroup plane z takes columns z k_per .. and leaves raw sums, rows of np, for k_linear_sum.
template <class T, int BM, int BN, int WM, int WN, int ST>
__global__ void __launch_bounds__(64 * WM * WN)
k_linear_tiled(const bf16_t* __restrict__ W, const bf16_t* __restrict__ X, float* act, T* opnd, const LinSpec s, uint32_t rows,
               uint32_t tiles_m, uint32_t tiles_n, uint32_t k_per, float* __restrict__ part, uint32_t np) {
  __shared__ __attribute__((aligned(16))) bf16_t la[ST * BN * 64], lb[ST * BM * 64];
  constexpr int NTN = BN / WN / 16, NTM = BM / WM / 16, PL = sizeof(T) == 4 ? 3 : 1;
  const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t c = lane & 15u, kg = lane >> 4, kp = s.k_stride, kx = PL * kp;
  // workgroups land on the eight dies in turn: give every die a run of neighbouring tiles
  const uint32_t total = tiles_m * tiles_n, per = (total + 7u) / 8u;
  const uint32_t id = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
  if (id >= total || (blockIdx.x >> 3) >= per) return;
  const uint32_t m0 = (id % tiles_m) * BM, n0 = (id / tiles_m) * BN, k0 = blockIdx.y * k_per;
  const uint32_t wn = (wave % WN) * (BN / WN), wm = (wave / WN) * (BM / WM);
  f4_t acc[NTN][NTM];
  tile_product<BM, BN, WM, WN, ST, PL>(
      acc, TileRows<BN, WM * WN>(wave, lane, [&](uint32_t r) { return W + (uint64_t)min(n0 + r, s.n - 1u) * kp; }),
      TileRows<BM, WM * WN>(wave, lane, [&](uint32_t r) { return X + (uint64_t)min(m0 + r, rows - 1u) * kx; }), kp, k0, min(kx, k0 + k_per),
      la, lb, wave, lane);
#pragma unroll
  for (int j = 0; j < NTM; j++) {
    const uint32_t row = m0 + wm + 16u * j + c;
    if (row >= rows) continue;
    if (part) {
      float* d = part + ((uint64_t)blockIdx.y * rows + row) * np;
#pragma unroll
      for (int i = 0; i < NTN; i++) {
        const uint32_t n = n0 + wn + 16u * i + 4u * kg;
        if (n < np) *(f4_t*)(d + n) = acc[i][j];
      }
    } else if (s.epi == 2u) {
#pragma unroll
      for (int i = 0; i < NTN; i += 2) put_pair_or_tail(s, act, opnd, row, n0 + wn + 16u * i + 4u * kg, acc[i][j], acc[i + 1][j]);
    } else {
#pragma unroll
      for (int i = 0; i < NTN; i++) put_out(s, act, row, n0 + wn + 16u * i + 4u * kg, acc[i][j]);
    }
  }
}
// The shares' sums, eight results (four and the four 16 on) a thread, np a multiple of 32.
template <class T>
__global__ void __launch_bounds__(256)
k_linear_sum(const LinSpec s, const float* __restrict__ part, float* act, T* opnd, uint32_t rows, uint32_t shares, uint32_t np) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x, per = np / 8u, row = i / per, q = i % per, n = (q >> 2) * 32u + (q & 3u) * 4u;
  if (row >= rows) return;
  f4_t a = {0, 0, 0, 0}, b = a;
  const float* p = part + (uint64_t)row * np + n;
  for (uint32_t z = 0; z < shares; z++, p += (uint64_t)rows * np) { a += *(const f4_t*)p; b += *(const f4_t*)(p + 16); }
  if (s.epi == 2u) put_pair_or_tail(s, act, opnd, row, n, a, b);
  else { put_out(s, act, row, n, a); put_out(s, act, row, n + 16u, b); }
}
// float32 operand rows as three bfloat16 rows whose sum they are exactly (8 significant bits each, so down to 2^-110 in size),
// the lowest first, as they are added up: the bfloat16 instruction's products of them are exact too, and at sixteen times the
// float32 instruction's rate three of them take a fifth of its time.  512 rows, 16384 x 2048: 322 -> 111 us (930 TFLOP/s of
// bfloat16 work), 2048 x 8192: 260 -> 76; 88 rows, 2048 x 2048: 57 -> 18.  Infinities and values that are no numbers stay in
// the highest piece; tile_product settles what an infinite weight makes of the others.
__global__ void __launch_bounds__(256)
k_split_rows(const float* __restrict__ x, bf16_t* __restrict__ dst, uint32_t kp, uint32_t rows) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x, per = kp / 4u, row = i / per, c = (i % per) * 4u;
  if (row >= rows) return;
  const float4 v = *(const float4*)(x + (uint64_t)row * kp + c);
  const float e[4] = {v.x, v.y, v.z, v.w};
  uint32_t p[3][4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const uint32_t u = __float_as_uint(e[j]);
    const float r = e[j] - __uint_as_float(u & 0xFFFF0000u), t = r - __uint_as_float(__float_as_uint(r) & 0xFFFF0000u);
    const bool number = (u & 0x7F800000u) != 0x7F800000u;
    p[0][j] = number ? __float_as_uint(t) >> 16 : 0u;
    p[1][j] = number ? __float_as_uint(r) >> 16 : 0u;
    p[2][j] = (u >> 16) | (!number && (u & 0x007FFFFFu) ? 0x40u : 0u);
  }
#pragma unroll
  for (int q = 0; q < 3; q++)
    *(uint2*)(dst + ((uint64_t)row * 3u + q) * kp + c) = make_uint2(p[q][0] | p[q][1] << 16, p[q][2] | p[q][3] << 16);
}

// ---- float32 operands ---------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
k_linear_f32(const bf16_t* __restrict__ W, const float* __restrict__ X, float* act, float* opnd, const LinSpec s, uint32_t rows) {
  __shared__ __attribute__((aligned(16))) float la[64][36], lb[64][36];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, c = lane & 15u, kg = lane >> 4, kp = s.k_stride;
  const uint32_t m0 = blockIdx.y * 64u, n0 = blockIdx.x * 64u, wn = (wave & 1u) * 32u, wm = (wave >> 1) * 32u;
  const uint32_t lr = tid >> 2, lc = (tid & 3u) * 8u;
  const bf16_t* wsrc = W + (uint64_t)min(n0 + lr, s.n - 1u) * kp + lc;
  const float* xsrc = X + (uint64_t)min(m0 + lr, rows - 1u) * kp + lc;
  f4_t acc[2][2];
  tile_product_f32(acc, wsrc, xsrc, kp, la, lb);
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const uint32_t row = m0 + wm + 16u * j + c;
    if (row >= rows) continue;
    if (s.epi == 2u) put_pair_or_tail(s, act, opnd, row, n0 + wn + 4u * kg, acc[0][j], acc[1][j]);
    else
#pragma unroll
      for (int i = 0; i < 2; i++) put_out(s, act, row, n0 + wn + 16u * i + 4u * kg, acc[i][j]);
  }
}

// ---- launch -------------------------------------------------------------------------------------------------------
static Scratch g_best, g_split, g_shares, g_rows;
void linear_release() { scratch_free(g_best); scratch_free(g_split); scratch_free(g_shares); scratch_free(g_rows); }

static bool span_ok(uint64_t off, uint64_t stride, uint64_t rows, uint64_t width, uint64_t n_elems) {
  return rows == 0 || in_range(off, (rows - 1) * stride + width, n_elems);
}

static int check_linear(Map* ma, Map* mo, Map* mw, const LinSpec& s, uint32_t rows, uint32_t src_rows) {
  if (!ma || !mw || mw->dtype != DTYPE_BF16 || rows == 0 || s.k == 0 || s.n == 0) return ADAMAH_ERR_INVALID;
  if (s.k_stride < s.k || (s.k_stride & 63u) || (s.w & 7u) || s.k_stride > LIN_MAX_K || s.epi > 2u) return ADAMAH_ERR_INVALID;
  if (!span_ok(s.w, s.k_stride, s.n, s.k_stride, mw->n_elems)) return ADAMAH_ERR_INVALID;
  if (s.groups > LIN_MAX_GROUPS || (s.groups && s.k % s.groups) || (s.gate_act && !s.groups) || (s.wt_len && !s.groups)) return ADAMAH_ERR_INVALID;
  if (!(rows > 1 && s.ready) && !span_ok(s.src, s.src_stride, src_rows, s.k, ma->n_elems)) return ADAMAH_ERR_INVALID;
  if (s.wt_len && !in_range(s.wt, s.wt_len, ma->n_elems)) return ADAMAH_ERR_INVALID;
  if (s.gate_act && !span_ok(s.gate, s.gate_stride, src_rows, s.k, ma->n_elems)) return ADAMAH_ERR_INVALID;
  if (s.tail > s.n || (s.tail && s.epi != 2u) || (s.epi == 2u && ((s.n - s.tail) & 31u)) || s.gate_act > 3u) return ADAMAH_ERR_INVALID;
  if (s.tail && !span_ok(s.tail_out, s.tail_stride, rows, s.tail, ma->n_elems)) return ADAMAH_ERR_INVALID;
  if (s.biased && (s.epi == 2u || !in_range(s.bias, s.n, ma->n_elems))) return ADAMAH_ERR_INVALID;
  if (!(rows > 1 && s.ready)) {
    if (s.branched > 2u || (s.branched && (s.groups != 1u || s.gate_act || (s.wt_len && s.wt_len != s.k)))) return ADAMAH_ERR_INVALID;
    if (s.branched && (!span_ok(s.branch, s.branch_stride, src_rows, s.k, ma->n_elems) || !in_range(s.branch_wt, s.k, ma->n_elems))) return ADAMAH_ERR_INVALID;
    if (s.branched == 2u) {                 // workgroups read src while one of them writes the sum
      if (!span_ok(s.res_out, s.res_stride, src_rows, s.k, ma->n_elems)) return ADAMAH_ERR_INVALID;
      for (const auto& r : {std::make_pair(s.src, s.src_stride), std::make_pair(s.branch, s.branch_stride)}) {
        const uint64_t e0 = s.res_out + (uint64_t)(src_rows - 1) * s.res_stride + s.k, e1 = r.first + (uint64_t)(src_rows - 1) * r.second + s.k;
        if (s.res_out < e1 && r.first < e0) return ADAMAH_ERR_INVALID;
      }
    }
    if (s.kept && !span_ok(s.keep, s.keep_stride, src_rows, s.k, ma->n_elems)) return ADAMAH_ERR_INVALID;
  }
  if (rows > 1) {
    if (!mo || (mo->dtype != DTYPE_BF16 && mo->dtype != DTYPE_F32) || (s.opnd & 7u)) return ADAMAH_ERR_INVALID;
    if (!span_ok(s.opnd, s.k_stride, rows, s.k_stride, mo->n_elems)) return ADAMAH_ERR_INVALID;
  }
  if (s.epi == 2u && rows > 1) return span_ok(s.out_opnd, s.out_opnd_stride, rows, (s.n - s.tail) / 2, mo->n_elems) ? ADAMAH_OK : ADAMAH_ERR_INVALID;
  return span_ok(s.out, s.out_stride, rows, s.epi == 2u ? (s.n - s.tail) / 2 : s.n, ma->n_elems) ? ADAMAH_OK : ADAMAH_ERR_INVALID;
}

// The tile and the shares of K that get through the rows soonest: rounds over the CUs times what a step of 64 columns takes
// there, measured on 40 .. 600 rows by 2048 .. 28672 x 2048 .. 14336: with one workgroup a CU, with two where two fit, and
// how much less of the first it is when hardly any CU has one; never faster than the matrix comes in.  Shares pay 4 us for
// the second launch and the way of the sums out and back (192 rows, 4096 x 14336: 70 us in one, 44 in four shares; 40 rows:
// 64 and 27; 40 rows, 12576 x 4096: 26 in one, 30 in two).  Over 540 shapes of 33 .. 2048 rows by 512 .. 28672 x 512 .. 14336,
// weights cold, the plan it picks takes 2.7 % longer than the best one in the mean (bfloat16; 32 % at most) and 2.4 % (float32
// in pieces; 39 %), and none longer than the two tiles that were all there was (0.47 and 0.37 of their time).
template <class T>
static int launch_tiles(const bf16_t* W, const bf16_t* X, float* act, T* op, const LinSpec& s, uint32_t rows) {
  struct Tile { uint32_t m, n; double one, idle, more, two; };          // more: hardly any CU has a second workgroup yet
  static const Tile tile[6] = {{256, 256, 1.70, 0.75, 0, 0}, {256, 128, 1.05, 0.72, 0, 0}, {128, 256, 1.05, 0.72, 0, 0},
                               {128, 128, 0.63, 0.70, 0, 0}, {64, 128, 0.49, 0.95, 0.80, 0.85}, {64, 64, 0.33, 0.75, 0.33, 0.58}};
  const uint32_t steps = (sizeof(T) == 4 ? 3u : 1u) * s.k_stride / 64u, np = (s.n + 31u) & ~31u;
  const uint64_t cu = (uint64_t)g.n_cu;
  const double out_us = (double)rows * np * 4.0 / 4.5e6, w_us = (double)s.n * s.k_stride * 2.0 / 4.2e6;
  double best = 1e30;
  uint32_t pick = 0, shares = 1;
  for (uint32_t t = 0; t < 6; t++) {
    const Tile& k = tile[t];
    const uint64_t tiles = (uint64_t)cdiv(rows, k.m) * cdiv(s.n, k.n), fit = k.two > 0 ? 2 * cu : cu;
    for (uint32_t sp = 1; sp <= 8 && (sp == 1 || (sp * 8 <= steps && tiles * sp <= fit)); sp++) {
      const uint64_t wgs = tiles * sp, left = wgs % fit;
      const double first = k.one * (wgs < cu ? k.idle + (1.0 - k.idle) * (double)wgs / (double)cu : 1.0);
      const double step = (double)(wgs / fit) * (k.two > 0 ? k.two : k.one) + (left == 0 ? 0.0 : left <= cu ? first : k.more + (k.two - k.more) * (double)(left - cu) / (double)cu);
      const double us = std::max(w_us, step * cdiv(steps, sp)) + (sp > 1 ? 4.0 + 2.0 * sp * out_us : 0.0);
      if (us < best) { best = us; pick = t; shares = sp; }
    }
  }
  uint32_t per = cdiv(steps, shares);
  shares = cdiv(steps, per);
  if (shares > 1 && scratch_need(g_shares, (size_t)shares * rows * np * sizeof(float)) != ADAMAH_OK) { shares = 1; per = steps; }
  float* part = shares > 1 ? (float*)g_shares.p : nullptr;
#define LT(BM, BN, WM, WN, ST) do { const uint32_t t = cdiv(rows, BM) * cdiv(s.n, BN); \
    k_linear_tiled<T, BM, BN, WM, WN, ST><<<dim3(cdiv(t, 8) * 8, shares), 64 * WM * WN, 0, g.stream>>>(W, X, act, op, s, rows, cdiv(rows, BM), cdiv(s.n, BN), \
                                                                                                      64 * per, part, np); } while (0)
  switch (pick) {
    case 0: LT(256, 256, 2, 4, 2); break;
    case 1: LT(256, 128, 4, 2, 3); break;
    case 2: LT(128, 256, 2, 4, 3); break;
    case 3: LT(128, 128, 2, 4, 4); break;
    case 4: LT(64, 128, 2, 2, 3); break;
    default: LT(64, 64, 2, 2, 4); break;
  }
#undef LT
  count_launch();
  if (part) {
    if (int r = check_launch()) return r;
    k_linear_sum<T><<<cdiv((uint64_t)rows * (np / 8), 256), 256, 0, g.stream>>>(s, part, act, op, rows, shares, np);
    count_launch();
  }
  return check_launch();
}

// A few workgroups more than CUs would each read and norm x first, on a CU that another one keeps busy: where x is normed and rows have 1024
// to 4096 columns, some waves take a second task instead, whose weights are asked for under the products of the first.  us, 264 to 288
// workgroups and 256 of them: behind a norm 1024 columns 6.1 and 5.6, 2048 8.3 and 7.95, 3072 11.0 and 9.9, 4096 11.95 and 11.65; behind a branch 6.3 and
// 5.8, 8.65 and 8.2, 11.5 and 10.5, 12.55 and 12.1; 2066 pairs of 2048, branched, 8.7 and 7.7.  Without a norm nothing waits (2048 columns 6.9 and 7.0); a
// short row's second task is a trip to memory that nothing hides (768 columns behind a norm 5.3 and 6.0); of a longer row, which a branch
// does not find in registers any more, a task is most of a wave's time (7168 columns behind a norm 17.7 and 18.2, behind a branch 22.6 and 23.6).
static uint32_t gemv_grid(const LinSpec& s, uint32_t n_tasks) {
  const uint32_t grid = cdiv(n_tasks, 8), cu = (uint32_t)g.n_cu;
  const bool once = (s.groups || s.branched) && s.k_stride >= 1024u && s.k_stride <= 4096u;
  return once && grid > cu && grid <= cu + cu / 8u ? cu : std::min(grid, 2u * cu);
}

// tasks of two rows (pairs of gate / up ahead of the tail's)
static uint32_t gemv_tasks(const LinSpec& s) { return s.epi == 2u ? (s.n - s.tail) / 2 + cdiv(s.tail, 2) : cdiv(s.n, 2); }

template <int EPI>
static void gemv_launch(Map* ma, Map* mw, const LinSpec& s, const uint32_t* row_idx) {
  const bf16_t* W = (const bf16_t*)mw->buf + s.w;
  const size_t lds = (size_t)s.k_stride * 4;
  const uint32_t mode = operand_mode(s, 512);
  const auto go = [&](auto* kernel, uint32_t n_tasks) {
    const uint32_t grid = gemv_grid(s, n_tasks);
    float* bv = (float*)g_best.p;
    if (lds > 60000) hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    kernel<<<grid, 512, lds, g.stream>>>(W, (float*)ma->buf, row_idx, s.k_stride, s.n, s.epi == 2u ? (s.n - s.tail) / 2 : 0u, s.src, s.k, mode, s.branch,
                                         s.branched ? s.branch_wt : s.wt, s, bv, bv ? (uint32_t*)(bv + grid) : nullptr);
    count_launch();
  };
  if (s.k_stride < 1024u) return go(k_gemv_bf16<EPI, 1, 2>, gemv_tasks(s));
  // A row a wave while that is a workgroup a CU at most: with two, half the CUs or less would have one (2048 x 2048 4.8 us, so 4.05;
  // 4096 x 4096 in two workgroups a CU 12.2, two rows a wave 9.8)
  if constexpr (EPI == LEPI_STORE || EPI == LEPI_ADD)
    if (s.n <= 8u * (uint32_t)g.n_cu) return s.k_stride > 2048u ? go(k_gemv_bf16<EPI, 8, 1>, s.n) : go(k_gemv_bf16<EPI, 4, 1>, s.n);
  go(k_gemv_bf16<EPI, 4, 2>, gemv_tasks(s));
}

int run_linear(Map* ma, Map* mo, Map* mw, const LinSpec& s, const uint32_t* row_idx, uint32_t rows) {
  float* act = (float*)ma->buf;
  if (rows == 1) {
    if (s.epi == 2u) gemv_launch<LEPI_PAIR>(ma, mw, s, row_idx);
    else if (s.epi == 1u) gemv_launch<LEPI_ADD>(ma, mw, s, row_idx);
    else gemv_launch<LEPI_STORE>(ma, mw, s, row_idx);
    return check_launch();
  }
  const bf16_t* W = (const bf16_t*)mw->buf + s.w;
  if (mo->dtype == DTYPE_F32) {
    float* op = (float*)mo->buf;
    if (!s.ready) operand_rows<float>(s, act, op + s.opnd, row_idx, rows);
    // Long rows in three bfloat16 pieces (the launch that splits them: 4 us; 88 rows of 512: 15.6 us on the float32
    // instruction, 11.2 in pieces; of 256: 8.3 and 8.2; of 128: 5.1 and 6.6).  k_split_rows counts four columns a thread in 32 bits.
    if (s.k_stride > 256u && (uint64_t)rows * s.k_stride < (1ull << 34) && scratch_need(g_split, (size_t)rows * 3 * s.k_stride * sizeof(bf16_t)) == ADAMAH_OK) {
      bf16_t* X = (bf16_t*)g_split.p;
      k_split_rows<<<cdiv((uint64_t)rows * s.k_stride / 4, 256), 256, 0, g.stream>>>(op + s.opnd, X, s.k_stride, rows);
      count_launch();
      if (int r = check_launch()) return r;
      return launch_tiles<float>(W, X, act, op, s, rows);
    }
    k_linear_f32<<<dim3(cdiv(s.n, 64), cdiv(rows, 64)), 256, 0, g.stream>>>(W, op + s.opnd, act, op, s, rows);
    count_launch();
    return check_launch();
  }
  bf16_t* op = (bf16_t*)mo->buf;
  const bf16_t* X = op + s.opnd;
  if (!s.ready) operand_rows<bf16_t>(s, act, op + s.opnd, row_idx, rows);
  if (rows > 32) return launch_tiles<bf16_t>(W, X, act, op, s, rows);
  const uint32_t pair = s.epi == 2u, units = pair ? cdiv(s.n, 32) * 16u : s.n, per = cdiv(units, g.n_cu), grid = cdiv(units, per);
  // Below 1152 columns a launch is over before its registers are worth filling, and of three steps the third is nearly empty (32 rows,
  // 3584 x 1088: 5.4 us as it is, 6.5 with this kernel; 8192 x 1024 under 16 rows 5.7, 9.7 with one step of four used); beyond 4096 the
  // tokens do not fit them.  In between a wave whose last step lies beyond the row's end reads its first columns again; where that is
  // more than a twentieth of the row, it costs more than it brings unless a CU has hardly a pass or more than two (16 rows, us, the kernel
  // below and this one: 4096 x 1216 4.5 and 5.1, 8192 x 2112 9.8 and 11.2, 4096 x 3648 9.2 and 10.6; but 1536 x 2112 6.0 and 5.8, 9216 x 2112 14.7 and
  // 12.4, 28671 x 2112 27.9 and 25.4; of pairs, whose CUs have twice the rows, 8192 x 2112 9.7 and 11.5, 512 x 2112 8.0 and 6.1).
  // One pass of nearly all its 16 matrix rows on every CU has nothing to stream behind: 16 waves in two lots of loads do it
  // as well or better (12 rows, 4096 x 4096: 9.4 and 10.4, of 32 rows 13.8 and 13.9; 13 matrix rows a CU, 3328 x 4096: 9.95 and 8.4, 14.1 and 13);
  // nor do two of them with one step of each in flight beat one workgroup of 32 a CU (8192 x 3072 12.2 and 13.9, 8192 x 4032 14.6 and 16.4).
  // The words are the same either way.
  const uint32_t room = 512u * cdiv(s.k_stride, 512), each = pair ? 2u * per : per;       // columns that the steps have room for; matrix rows a CU
  const bool whole = s.k_stride * 20u >= room * 19u;
  if (s.k_stride >= 1152u && s.k_stride <= 4096u &&
      (whole ? pair || s.k_stride <= 2048u || per <= 14u || (per > 16u && !(per > 28u && per <= 32u && s.k_stride > 2560u))
             : each <= 8u || each > (pair ? 64u : 34u))) {
    const auto go = [&](auto* one, auto* two) {
      (rows <= 16 ? one : two)<<<grid, 512, 0, g.stream>>>(W, X, act, op, s.k_stride, s.n, rows, units, per, pair, s);
    };
#define FEW(S) do { if (pair || per > 16u) go(k_linear_few<1, S, false>, k_linear_few<2, S, false>); else go(k_linear_few<1, S, true>, k_linear_few<2, S, true>); } while (0)
    switch (cdiv(s.k_stride, 512)) {
      case 3: FEW(3); break;
      case 4: FEW(4); break;
      case 5: FEW(5); break;
      case 6: FEW(6); break;
      case 7: FEW(7); break;
      default: FEW(8); break;
    }
#undef FEW
    count_launch();
    return check_launch();
  }
  // Workgroups of 16 matrix rows as long as no CU gets a second one (12 rows, 4096 x 4096: 9.6 us, of 32: 13.4)
#define LS(MT) do { if (s.epi != 2u && cdiv(s.n, 16) <= (uint32_t)g.n_cu) k_linear_skinny<MT, 1, 16><<<cdiv(s.n, 16), 1024, 0, g.stream>>>(W, X, act, op, s, rows); \
    else k_linear_skinny<MT, 2, 8><<<cdiv(s.n, 32), 512, 0, g.stream>>>(W, X, act, op, s, rows); } while (0)
  if (rows <= 16) LS(1); else LS(2);
#undef LS
  count_launch();
  return check_launch();
}

// Rows of a linear op named by a handle: every index must be known on the host, so that the largest can be checked.
static int row_list(uint32_t h_rows, uint32_t rows, const uint32_t** dev, uint32_t* src_rows) {
  *dev = nullptr; *src_rows = rows;
  if (!h_rows) return ADAMAH_OK;
  const uint32_t* hp = res_host(h_rows, rows);
  *dev = res_u32(h_rows, rows);
  if (!hp || !*dev) return ADAMAH_ERR_INVALID;
  *src_rows = *std::max_element(hp, hp + rows) + 1u;
  return ADAMAH_OK;
}

// k_merge_norm: dst += scale * sum over the two parts of rms(part) * weight
template <int NT>
__global__ void __launch_bounds__(NT)
k_merge_norm(const AdamahMergeSpec s, float* act) {
  __shared__ float sh[2][NT / 64];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const float* a = act + s.a + (uint64_t)blockIdx.x * s.stride;
  const float* b = act + s.b + (uint64_t)blockIdx.x * s.stride;
  float* d = act + s.dst + (uint64_t)blockIdx.x * s.dst_stride;
  float sa = 0.f, sb = 0.f;
#pragma unroll 4
  for (uint32_t i = tid; i < s.dim; i += NT) { sa = fmaf(a[i], a[i], sa); sb = fmaf(b[i], b[i], sb); }
  sa = wave_add(sa); sb = wave_add(sb);
  if (lane == 0) { sh[0][wave] = sa; sh[1][wave] = sb; }
  __syncthreads();
  sa = sb = 0.f;
#pragma unroll
  for (int w = 0; w < NT / 64; w++) { sa += sh[0][w]; sb += sh[1][w]; }
  const float ia = 1.0f / sqrtf(sa / (float)s.dim + s.eps), ib = 1.0f / sqrtf(sb / (float)s.dim + s.eps);
#pragma unroll 4
  for (uint32_t i = tid; i < s.dim; i += NT) d[i] = (s.store ? 0.f : d[i]) + s.scale * (a[i] * ia * act[s.wa + i] + b[i] * ib * act[s.wb + i]);
}

}  // namespace adamah

using namespace adamah;

extern "C" {

int adamah_linear_dev(uint32_t map_act, uint32_t map_opnd, uint32_t map_wt, uint32_t h_spec, uint32_t h_rows, uint32_t rows) { ADAMAH_API();
  Map *ma = get_f32_map(map_act), *mo = get_map(map_opnd), *mw = get_map(map_wt);
  const LinSpec* s = spec_of<LinSpec>(h_spec);
  const uint32_t* dev;
  uint32_t src_rows;
  if (!s) return ADAMAH_ERR_INVALID;
  if (int r = row_list(h_rows, rows, &dev, &src_rows)) return r;
  if (int r = check_linear(ma, mo, mw, *s, rows, src_rows)) return r;
  return run_linear(ma, mo, mw, *s, dev, rows);
}

int adamah_linear_argmax_dev(uint32_t map_act, uint32_t map_opnd, uint32_t map_wt, uint32_t h_spec, uint32_t h_dst, uint32_t rows) { ADAMAH_API();
  Map *ma = get_f32_map(map_act), *mo = get_map(map_opnd), *mw = get_map(map_wt);
  const LinSpec* s = spec_of<LinSpec>(h_spec);
  if (!s || s->epi != 0u) return ADAMAH_ERR_INVALID;
  if (int r = check_linear(ma, mo, mw, *s, rows, rows)) return r;
  const uint32_t* dst = res_host(h_dst, rows);
  if (!dst) return ADAMAH_ERR_INVALID;
  for (uint32_t i = 0; i < rows; i++) if (dst[i] >= ma->n_elems) return ADAMAH_ERR_INVALID;
  float* act = (float*)ma->buf;
  if (rows == 1) {
    const uint32_t grid = gemv_grid(*s, gemv_tasks(*s));
    if (int r = scratch_need(g_best, (size_t)grid * 8)) return r;
    gemv_launch<LEPI_ARGMAX>(ma, mw, *s, nullptr);
    k_best_pair<<<1, 256, 0, g.stream>>>((const float*)g_best.p, (const uint32_t*)g_best.p + grid, grid, act + dst[0], nullptr);
  } else {
    if (int r = run_linear(ma, mo, mw, *s, nullptr, rows)) return r;
    // (1024 threads only reduce more: rows of 50 in 4.1 us, with 256 in 3.0, of 1000 in 4.2 and 3.9; rows of 2000 in 4.5 and 5.1, of 4000 in 5.0 and 8.1)
    if (s->n > 1024u) k_best_row<1024><<<rows, 1024, 0, g.stream>>>(act, s->out, s->out_stride, s->n, act, res_u32(h_dst, rows));
    else k_best_row<256><<<rows, 256, 0, g.stream>>>(act, s->out, s->out_stride, s->n, act, res_u32(h_dst, rows));
  }
  count_launch();
  return check_launch();
}

// What adamah_linear_argmax_dev over one row gives, for each of the listed rows in turn
int adamah_hip_linear_argmax_rows_dev(uint32_t map_act, uint32_t map_opnd, uint32_t map_wt, uint32_t h_spec, uint32_t h_rows, uint32_t h_dst, uint32_t rows) { ADAMAH_API();
  Map *ma = get_f32_map(map_act), *mo = get_map(map_opnd), *mw = get_map(map_wt);
  const LinSpec* s = spec_of<LinSpec>(h_spec);
  const uint32_t* dev;
  uint32_t src_rows;
  if (!s || s->epi != 0u || rows == 0) return ADAMAH_ERR_INVALID;
  if (int r = row_list(h_rows, rows, &dev, &src_rows)) return r;
  if (int r = check_linear(ma, mo, mw, *s, 1, src_rows)) return r;
  const uint32_t *dst = res_host(h_dst, rows), *dst_dev = res_u32(h_dst, rows);
  if (!dst || !dst_dev) return ADAMAH_ERR_INVALID;
  for (uint32_t i = 0; i < rows; i++) if (dst[i] >= ma->n_elems) return ADAMAH_ERR_INVALID;
  float* act = (float*)ma->buf;
  // rows at a time: as many as 144 KB of LDS hold (a workgroup a CU), none of them for nothing
  const size_t row_bytes = (size_t)s->k_stride * 4;
  const uint32_t fit = (uint32_t)(((size_t)144 << 10) / row_bytes), nr = fit >= 8 && rows > 4 ? 8 : fit >= 4 && rows > 2 ? 4 : fit >= 2 && rows > 1 ? 2 : 1;
  if (rows == 1) {
    const uint32_t grid = gemv_grid(*s, gemv_tasks(*s));
    if (int r = scratch_need(g_best, (size_t)grid * 8)) return r;
    gemv_launch<LEPI_ARGMAX>(ma, mw, *s, dev);
    k_best_pair<<<1, 256, 0, g.stream>>>((const float*)g_best.p, (const uint32_t*)g_best.p + grid, grid, act + dst[0], nullptr);
    count_launch();
    return check_launch();
  }
  const uint32_t n_tasks = cdiv(s->n, 4), grid = std::min<uint32_t>(cdiv(n_tasks, 8), (uint32_t)g.n_cu);
  if (int r = scratch_need(g_best, (size_t)grid * rows * 8)) return r;
  if (int r = scratch_need(g_rows, rows * row_bytes)) return r;
  float* const X = (float*)g_rows.p;
  float* const bv = (float*)g_best.p;
  uint32_t* const bi = (uint32_t*)(bv + (size_t)grid * rows);
  operand_rows<float>(*s, act, X, dev, rows);
  const bf16_t* W = (const bf16_t*)mw->buf + s->w;
  for (uint32_t i = 0; i < rows; i += nr) {
    const uint32_t n = std::min(nr, rows - i), kept = i + n == rows ? n - 1u : 0xFFFFFFFFu;
#define HEAD(NR)                                                                                                    \
  do {                                                                                                              \
    hipFuncSetAttribute((const void*)k_head_rows<NR>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(NR * row_bytes)); \
    k_head_rows<NR><<<grid, 512, NR * row_bytes, g.stream>>>(W, act, *s, X + (size_t)i * s->k_stride, n, kept, n_tasks, bv + (size_t)i * grid, bi + (size_t)i * grid); \
  } while (0)
    if (nr == 8) HEAD(8); else if (nr == 4) HEAD(4); else if (nr == 2) HEAD(2); else HEAD(1);
#undef HEAD
    count_launch();
  }
  if (int r = check_launch()) return r;
  k_best_pair<<<rows, 256, 0, g.stream>>>(bv, bi, grid, act, dst_dev);
  count_launch();
  return check_launch();
}

int adamah_merge_norm_dev(uint32_t map_act, uint32_t h_spec, uint32_t rows) { ADAMAH_API();
  Map* ma = get_f32_map(map_act);
  const AdamahMergeSpec* s = spec_of<AdamahMergeSpec>(h_spec);
  if (!ma || !s || rows == 0 || s->dim == 0) return ADAMAH_ERR_INVALID;
  if (!span_ok(s->a, s->stride, rows, s->dim, ma->n_elems) || !span_ok(s->b, s->stride, rows, s->dim, ma->n_elems) ||
      !span_ok(s->dst, s->dst_stride, rows, s->dim, ma->n_elems) || !in_range(s->wa, s->dim, ma->n_elems) ||
      !in_range(s->wb, s->dim, ma->n_elems)) return ADAMAH_ERR_INVALID;
  if (rows < 64) k_merge_norm<1024><<<rows, 1024, 0, g.stream>>>(*s, (float*)ma->buf);
  else k_merge_norm<256><<<rows, 256, 0, g.stream>>>(*s, (float*)ma->buf);
  count_launch();
  return check_launch();
}

}  // extern "C"
