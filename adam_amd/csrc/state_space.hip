// State-space recurrence (Mamba-2): one decay per head and token, inputs, B and C behind a short convolution, B and C shared
// by the heads of a group.  S_t = a_t S_(t-1) + dt_t B_t x_t^T, y_t = S_t^T C_t + D x_t, a_t = exp(-exp(A_log) dt_t); state,
// step sizes, decays and every product with the state are float32.
//
// One token (decode): k_space_step.  A workgroup owns one head and 32 of its value columns, which are independent but for
// the convolved B and C that every workgroup of a group makes for itself, so no workgroup waits for another.
//
// A portion of a prompt: two launches.  k_space_prep, a workgroup per chunk of 16 tokens and group or head, writes what the
// chunks are made of: per group C [16, N], B^T [N, 16] and the products C_t . B_s; per head the convolved inputs and, with
// L_t the sum of the decays' logarithms up to token t of the chunk, exp(L_t - L_s) dt_s for s <= t, exp(L_t) and
// exp(L_last - L_s) dt_s.  k_space_scan, a workgroup per head and 16 value columns, walks over the chunks with the state in
// the accumulators of the float32 matrix instruction:
//   y_t = exp(L_t) S^T C_t + sum_{s <= t} (C_t . B_s) exp(L_t - L_s) dt_s x_s + D x_t
//   S  <- exp(L_last) S + sum_s B_s (exp(L_last - L_s) dt_s x_s)^T
// A decay is one number per head and token, so it multiplies results and the 16 input rows; the wide operands stay those of
// the group.  Every exponent is <= 0: no strength of decay overflows.
#include "recurrent_common.h"
#include <algorithm>

namespace adamah {

typedef AdamahStateSpaceSpec SSpec;
#define SSTEP 512u

// One token of one sequence per blockIdx.z; DN: state rows a thread holds (N <= 16 DN); TM >= taps.
template <int DN, int TM>
__global__ void __launch_bounds__(SSTEP)
k_space_step(const SSpec s, float* act, float* state, uint32_t seq0, uint32_t pos) {
  constexpr uint32_t NG = SSTEP / VC;
  __shared__ float bc[2][16 * DN], red[NG][VC], xs[VC];
  const uint32_t N = s.state, V = s.vdim, tid = threadIdx.x, h = blockIdx.x, v0 = blockIdx.y * VC, row = blockIdx.z;
  const uint32_t inner = s.heads * V, n_ch = inner + 2u * s.groups * N, rep = s.heads / s.groups, grp = h / rep;
  const float* xr = act + s.x + (uint64_t)row * s.x_stride;
  const float* x = xr + s.x_c;
  float* ring = state + (uint64_t)(seq0 + row) * s.seq_stride + s.conv_off;
  float* S = state + (uint64_t)(seq0 + row) * s.seq_stride + s.s_off + (uint64_t)h * N * V;
  const uint32_t bch = inner + grp * N, cch = inner + (s.groups + grp) * N, xch = h * V + v0;
  const uint32_t col = tid & (VC - 1u), dg = tid / VC, v = v0 + col;
  float st[DN];
#pragma unroll
  for (int i = 0; i < DN; i++) {
    const uint32_t d = dg + NG * i;
    st[i] = (pos != 0u && d < N && v < V) ? S[(uint64_t)d * V + v] : 0.f;
  }
  const float z = xr[s.x_dt + h] + act[s.dt_bias + h], a_log = act[s.a_log + h], skip = act[s.skip + h];
  for (uint32_t i = tid; i < 2u * N; i += SSTEP) {
    const bool is_c = i >= N;
    const uint32_t d = is_c ? i - N : i, ch = (is_c ? cch : bch) + d;
    bc[is_c ? 1 : 0][d] = conv_silu_ring<TM>(x, ring, n_ch, ch, pos, act + s.conv + (uint64_t)ch * s.taps, s.taps, act[s.conv_b + ch]);
  }
  const uint32_t last = SSTEP - 1u - tid;                     // the inputs: by the threads at the other end
  if (last < VC && v0 + last < V) {
    const uint32_t ch = xch + last;
    xs[last] = conv_silu_ring<TM>(x, ring, n_ch, ch, pos, act + s.conv + (uint64_t)ch * s.taps, s.taps, act[s.conv_b + ch]);
  }
  const float dt = softplus_f(z), keep = expf(-fminf(expf(a_log) * dt, NO_MEMORY));
  __syncthreads();
  const float xv = v < V ? xs[col] : 0.f, dx = dt * xv;
  float y = 0.f;
#pragma unroll
  for (int i = 0; i < DN; i++) {
    const uint32_t d = dg + NG * i;
    if (d < N && v < V) {
      const float t = fmaf(bc[0][d], dx, keep * st[i]);
      y = fmaf(t, bc[1][d], y);
      S[(uint64_t)d * V + v] = t;
    }
  }
  red[dg][col] = y;
  __syncthreads();
  if (dg == 0 && v < V) {
    y = 0.f;
#pragma unroll
    for (int i = 0; i < (int)NG; i++) y += red[i][col];
    act[s.out + (uint64_t)row * s.out_stride + h * V + v] = fmaf(skip, xv, y);
  }
  float* slot = ring + (uint64_t)(pos % s.taps) * n_ch;
  if (blockIdx.y == 0 && h % rep == 0)
    for (uint32_t d = tid; d < N; d += SSTEP) { slot[bch + d] = x[bch + d]; slot[cch + d] = x[cch + d]; }
  if (tid < VC && v0 + tid < V) slot[xch + tid] = x[xch + tid];
}

// ---- a portion ------------------------------------------------------------------------------------------------------
// Blocks of a (group, chunk): C [16][Np], B^T [Np][16], C . B [16][16]; of a (head, chunk): x [16][Vp], exp(L_t - L_s) dt_s
// [16][16], exp(L_t) [16], exp(L_last - L_s) dt_s [16].
struct SpaceDims { uint32_t Np, Vp, n_chunks; };
__host__ __device__ inline uint32_t group_floats(const SpaceDims& d) { return 32u * d.Np + 256u; }
__host__ __device__ inline uint32_t head_floats(const SpaceDims& d) { return 16u * d.Vp + 288u; }

template <int TM>
__global__ void __launch_bounds__(256)
k_space_prep(const SSpec s, const float* __restrict__ act, const float* __restrict__ state, float* __restrict__ scratch, SpaceDims sd,
             uint32_t m, uint32_t seq0, uint32_t pos) {
  extern __shared__ float lds[];
  const uint32_t N = s.state, V = s.vdim, tid = threadIdx.x, c0 = blockIdx.x * CH, inner = s.heads * V, n_ch = inner + 2u * s.groups * N;
  const float* x = act + s.x + s.x_c;
  const float* ring = state + (uint64_t)seq0 * s.seq_stride + s.conv_off;
  const auto conv = [&](uint32_t ch, auto put) {
    conv_silu_rows<TM>(x, s.x_stride, c0, m, ring, n_ch, ch, pos, act + s.conv + (uint64_t)ch * s.taps, s.taps, put, act[s.conv_b + ch]);
  };
  if (blockIdx.y < s.groups) {
    const uint32_t grp = blockIdx.y, P = N + 1u;
    float *bs = lds, *cs = lds + CH * P;
    float* oC = scratch + ((uint64_t)grp * sd.n_chunks + blockIdx.x) * group_floats(sd);
    float *oB = oC + 16u * sd.Np, *oD = oB + 16u * sd.Np;
    for (uint32_t i = tid; i < 2u * N; i += 256u) {
      const bool is_c = i >= N;
      const uint32_t d = is_c ? i - N : i;
      float* to = (is_c ? cs : bs) + d;
      conv(inner + ((is_c ? s.groups : 0u) + grp) * N + d, [&](int t, float v) { to[t * P] = v; });
    }
    __syncthreads();
    {
      const uint32_t t = tid >> 4, r = tid & 15u;
      float a = 0.f;
      if (r <= t) {
#pragma unroll 4
        for (uint32_t d = 0; d < N; d++) a = fmaf(cs[t * P + d], bs[r * P + d], a);
      }
      oD[place16(t, r)] = a;
    }
    for (uint32_t d = tid; d < sd.Np; d += 256u) {
      float c[CH], b[CH];
#pragma unroll
      for (int t = 0; t < (int)CH; t++) {
        c[t] = d < N ? cs[t * P + d] : 0.f;
        b[t] = d < N ? bs[t * P + d] : 0.f;
      }
      store_rows(oC, d, c);
      store_cols(oB, d, b);
    }
    return;
  }
  const uint32_t h = blockIdx.y - s.groups;
  float *dt = lds, *lg = lds + CH;
  float* oX = scratch + (uint64_t)s.groups * sd.n_chunks * group_floats(sd) + ((uint64_t)h * sd.n_chunks + blockIdx.x) * head_floats(sd);
  float *oM = oX + 16u * sd.Vp, *oE = oM + 256u, *oG = oE + 16u;
  if (tid < 64u) {                                            // tokens past the portion: no step, no decay
    const uint32_t t = tid & 15u;
    const bool in = c0 + t < m;
    const float d = in ? softplus_f(act[s.x + (uint64_t)(c0 + t) * s.x_stride + s.x_dt + h] + act[s.dt_bias + h]) : 0.f;
    if (tid < CH) { dt[t] = d; lg[t] = -fminf(expf(act[s.a_log + h]) * d, NO_MEMORY) * 1.44269504f; }
  }
  for (uint32_t i = tid; i < sd.Vp; i += 256u) {
    float y[CH] = {};
    if (i < V) conv(h * V + i, [&](int t, float v) { y[t] = v; });
    store_cols(oX, i, y);
  }
  __syncthreads();
  // Decays between two tokens from the logarithms between them: the difference of two long sums would keep the rounding of
  // everything ahead of both.
  const uint32_t t = tid >> 4, r = tid & 15u;
  float l = 0.f, e = 0.f;
#pragma unroll
  for (uint32_t i = 0; i < CH; i++) { l += i > r && i <= t ? lg[i] : 0.f; e += i <= r ? lg[i] : 0.f; }
  l = r <= t ? __builtin_amdgcn_exp2f(l) * dt[r] : 0.f;
  oM[place16(t, r)] = l;
  if (t == CH - 1u) { oE[r] = __builtin_amdgcn_exp2f(e); oG[r] = l; }
}

// Four waves share the state rows (NT tiles of 16 each); a tile's accumulator holds rows 4 g + i of lane group g, which
// is also how instruction i wants its right operand when the left one is read as four consecutive columns per lane.  Each leaves
// its rows' part of C S in LDS and its quarter of what the chunk's own part needs; a fifth wave adds up, multiplies and stores, a
// chunk behind: loads and stores share a counter, and a wave that does both waits for its stores (2048 tokens in 64 heads of 64 by
// 128, the waves taking turns with the outputs 104 us, so 85; scan_form says where they do all the same).  In every form one product
// behind the other by wave, the waves' parts as (0 + 1) + (2 + 3) times the decay, the chunk's own part behind that sum in order; C B
// times its decay is rounded before the skip is added.
template <int NT, int FORM> struct SpaceOps { f4_t c[NT], b[NT], g, u; std::conditional_t<FORM == SCAN_TURNS, f4_t, float> cb, m, e; float last; };
template <int NT, int FORM>
__device__ __forceinline__ void load_ops(SpaceOps<NT, FORM>& o, const float* gb, const float* hb, const SpaceDims& sd, uint32_t wave, uint32_t lane,
                                         uint32_t v0) {
  const float *pB = gb + 16u * sd.Np, *pD = pB + 16u * sd.Np, *pM = hb + 16u * sd.Vp, *pE = pM + 256u, *pG = pE + 16u;
#pragma unroll
  for (int j = 0; j < NT; j++) {
    const uint32_t at = (wave * NT + j) * 256u + lane * 4u;
    o.c[j] = *(const f4_t*)(gb + at);
    o.b[j] = *(const f4_t*)(pB + at);
  }
  o.g = *(const f4_t*)(pG + (lane >> 4) * 4u);
  o.u = *(const f4_t*)(hb + v0 * 16u + lane * 4u);
  if constexpr (FORM == SCAN_TURNS) {
    o.cb = *(const f4_t*)(pD + lane * 4u); o.m = *(const f4_t*)(pM + lane * 4u); o.e = *(const f4_t*)(pE + (lane >> 4) * 4u);
  } else {
    o.cb = pD[lane * 4u + wave]; o.m = pM[lane * 4u + wave]; o.e = pE[(lane >> 4) * 4u + wave];
  }
  o.last = pE[15];
}

template <int NT, int FORM>
__global__ void __launch_bounds__(SCAN_T(FORM), FORM == SCAN_TURNS ? 2 : 1)
k_space_scan(const SSpec s, const float* __restrict__ scratch, float* act, float* state, SpaceDims sd, uint32_t m, uint32_t seq0, uint32_t pos) {
  __shared__ f4_t pb[2][4][64];                              // [chunk & 1][wave][lane]
  __shared__ f4_t pc[2][3][64];                              // C B and skip, x, decay for the fifth wave, one of a lane's four by each wave
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6)), c = lane & 15u, kg = lane >> 4;
  const uint32_t h = blockIdx.x, v0 = blockIdx.y * 16u, N = s.state, V = s.vdim, v = v0 + c, rep = s.heads / s.groups, grp = h / rep;
  const uint32_t gs = group_floats(sd), hs = head_floats(sd), n = sd.n_chunks;
  state += (uint64_t)seq0 * s.seq_stride;
  float* out = act + s.out + h * V + v;
  const auto put = [&](uint32_t ci, f4_t cb, f4_t u, f4_t e) {         // the outputs of chunk ci
    const f4_t (*p)[64] = pb[ci & 1u];
    f4_t o = ((p[0][lane] + p[1][lane]) + (p[2][lane] + p[3][lane])) * e;
#pragma unroll
    for (int i = 0; i < 4; i++) o = __builtin_amdgcn_mfma_f32_16x16x4f32(cb[i], u[i], o, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t r = ci * CH + 4u * kg + i;
      if (r < m && v < V) out[(uint64_t)r * s.out_stride] = o[i];
    }
  };
  if (FORM != SCAN_TURNS && wave == 4u) {
    for (uint32_t ci = 0; ci < n; ci++) {
      __syncthreads();
      put(ci, pc[ci & 1u][0][lane], pc[ci & 1u][1][lane], pc[ci & 1u][2][lane]);
    }
  } else {
    const float* gb = scratch + (uint64_t)grp * n * gs;
    const float* hb = scratch + (uint64_t)s.groups * n * gs + (uint64_t)h * n * hs;
    float* S = state + s.s_off + (uint64_t)h * N * V;
    const float skip = act[s.skip + h];
    f4_t st[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) st[j] = (f4_t){0, 0, 0, 0};
    if (pos != 0u) {
#pragma unroll
      for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) st[j][i] = S[(uint64_t)min((wave * NT + j) * 16u + 4u * kg + i, N - 1u) * V + min(v, V - 1u)];
#pragma unroll
      for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) if ((wave * NT + j) * 16u + 4u * kg + i >= N || v >= V) st[j][i] = 0.f;
    }
    // The operands of the chunk two ahead, asked for on every path (past the end: the last one's again): under a condition
    // the wait at its end was for everything asked for (162 us for 94).
    const auto ask = [&](SpaceOps<NT, FORM>& o, uint32_t ci) {
      const uint64_t at = min(ci, n - 1u);
      load_ops<NT, FORM>(o, gb + at * gs, hb + at * hs, sd, wave, lane, v0);
      __builtin_amdgcn_sched_barrier(0);
    };
    const auto chunk = [&](const SpaceOps<NT, FORM>& cur, uint32_t ci) {
      const uint32_t x = ci & 1u;
      f4_t p = {0, 0, 0, 0};
#pragma unroll
      for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) p = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.c[j][i], st[j][i], p, 0, 0, 0);
#pragma unroll
      for (int j = 0; j < NT; j++) st[j] *= cur.last;
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) st[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.b[j][i], cur.g[i] * cur.u[i], st[j], 0, 0, 0);
      pb[x][wave][lane] = p;
      if constexpr (FORM == SCAN_TURNS) {
        __syncthreads();
        if (wave == (ci & 3u)) {
          f4_t cb = cur.cb * cur.m;
#pragma unroll
          for (int i = 0; i < 4; i++) cb[i] += c == 4u * kg + i ? skip : 0.f;
          put(ci, cb, cur.u, cur.e);
        }
      } else {
        ((float*)&pc[x][0][lane])[wave] = cur.cb * cur.m + (c == 4u * kg + wave ? skip : 0.f);
        ((float*)&pc[x][1][lane])[wave] = wave & 2u ? (wave & 1u ? cur.u[3] : cur.u[2]) : (wave & 1u ? cur.u[1] : cur.u[0]);
        ((float*)&pc[x][2][lane])[wave] = cur.e;
        __syncthreads();
      }
    };
    SpaceOps<NT, FORM> o0;
    ask(o0, 0);
    if constexpr (FORM == SCAN_FEW) {
      for (uint32_t ci = 0; ci < n; ci++) {
        if (ci) ask(o0, ci);
        chunk(o0, ci);
      }
    } else {
      // (a loop in one piece: with a way out behind each chunk the loads were moved down to where only the rest of the loop needs them)
      SpaceOps<NT, FORM> o1, o2;
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
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t d = (wave * NT + j) * 16u + 4u * kg + i;
        if (d < N && v < V) S[(uint64_t)d * V + v] = st[j][i];
      }
  }
  const uint32_t inner = s.heads * V, n_ch = inner + 2u * s.groups * N;      // the convolution's ring
  for (uint32_t r = m > s.taps ? m - s.taps : 0u; r < m; r++) {
    float* slot = state + s.conv_off + (uint64_t)((pos + r) % s.taps) * n_ch;
    const float* x = act + s.x + s.x_c + (uint64_t)r * s.x_stride;
    if (blockIdx.y == 0 && h % rep == 0)
      for (uint32_t d = tid; d < N; d += SCAN_T(FORM)) {
        const uint32_t b = inner + grp * N + d, cc = inner + (s.groups + grp) * N + d;
        slot[b] = x[b];
        slot[cc] = x[cc];
      }
    if (wave == 0u && kg == 0u && v < V) slot[h * V + v] = x[h * V + v];
  }
}

static Scratch g_space;
void state_space_release() { scratch_free(g_space); }

}  // namespace adamah

using namespace adamah;

extern "C" int adamah_state_space_dev(uint32_t map_act, uint32_t h_spec, uint32_t n_seq, uint32_t rows, uint32_t seq0, uint32_t pos) { ADAMAH_API();
  Map* ma = get_f32_map(map_act);
  const SSpec* s = spec_of<SSpec>(h_spec);
  if (!ma || !s || n_seq == 0 || rows == 0 || (n_seq > 1 && rows > 1)) return ADAMAH_ERR_INVALID;
  Map* ms = get_f32_map(s->state_map);
  const uint64_t N = s->state, V = s->vdim, H = s->heads, G = s->groups, n_tok = (uint64_t)n_seq * rows;
  if (!ms || N == 0 || N > 256 || V == 0 || V > 256 || H == 0 || G == 0 || H % G || s->taps == 0 || s->taps > MAX_TAPS) return ADAMAH_ERR_INVALID;
  const uint64_t n_ch = H * V + 2 * G * N;
  if (s->x_c + n_ch > s->x_stride || s->x_dt + H > s->x_stride || H + G > 65535) return ADAMAH_ERR_INVALID;
  if (!in_range(s->x, n_tok * s->x_stride, ma->n_elems) || !in_range(s->out, (n_tok - 1) * s->out_stride + H * V, ma->n_elems)) return ADAMAH_ERR_INVALID;
  if (!in_range(s->conv, n_ch * s->taps, ma->n_elems) || !in_range(s->conv_b, n_ch, ma->n_elems) || !in_range(s->dt_bias, H, ma->n_elems) ||
      !in_range(s->a_log, H, ma->n_elems) || !in_range(s->skip, H, ma->n_elems)) return ADAMAH_ERR_INVALID;
  if ((uint64_t)s->s_off + H * N * V > s->seq_stride || (uint64_t)s->conv_off + n_ch * s->taps > s->seq_stride ||
      !in_range((uint64_t)seq0 * s->seq_stride, (uint64_t)n_seq * s->seq_stride, ms->n_elems)) return ADAMAH_ERR_INVALID;
  float *act = (float*)ma->buf, *state = (float*)ms->buf;
  if (rows == 1) {
    const dim3 grid((uint32_t)H, cdiv(V, VC), n_seq);
#define STEP(DN, TM) k_space_step<DN, TM><<<grid, SSTEP, 0, g.stream>>>(*s, act, state, seq0, pos)
    if (s->taps <= 4) { if (N <= 64) STEP(4, 4); else if (N <= 128) STEP(8, 4); else STEP(16, 4); }
    else { if (N <= 64) STEP(4, MAX_TAPS); else if (N <= 128) STEP(8, MAX_TAPS); else STEP(16, MAX_TAPS); }
#undef STEP
    count_launch();
    return check_launch();
  }
  const SpaceDims sd = {(uint32_t)((N + 63) / 64 * 64), (uint32_t)((V + 15) / 16 * 16), cdiv(rows, CH)};
  if (int r = scratch_need(g_space, (G * sd.n_chunks * group_floats(sd) + H * sd.n_chunks * head_floats(sd)) * 4)) return r;
  float* sc = (float*)g_space.p;
  const dim3 pg(sd.n_chunks, (uint32_t)(G + H));
  const size_t lds = std::max<size_t>(2 * CH, (size_t)2 * CH * (N + 1)) * 4;
  if (s->taps <= 4) k_space_prep<4><<<pg, 256, lds, g.stream>>>(*s, act, state, sc, sd, rows, seq0, pos);
  else k_space_prep<MAX_TAPS><<<pg, 256, lds, g.stream>>>(*s, act, state, sc, sd, rows, seq0, pos);
  count_launch();
  if (int r = check_launch()) return r;
  const dim3 grid((uint32_t)H, cdiv(V, 16));
  const auto go = [&](auto tiles) {
    constexpr int NT = decltype(tiles)::value;
    const int form = scan_form((uint64_t)grid.x * grid.y, sd.n_chunks, NT, NT <= 2, true);
    if (form == SCAN_FEW) k_space_scan<NT, SCAN_FEW><<<grid, SCAN_T(SCAN_FEW), 0, g.stream>>>(*s, sc, act, state, sd, rows, seq0, pos);
    else if (form == SCAN_DEEP) k_space_scan<NT, SCAN_DEEP><<<grid, SCAN_T(SCAN_DEEP), 0, g.stream>>>(*s, sc, act, state, sd, rows, seq0, pos);
    else k_space_scan<NT, SCAN_TURNS><<<grid, SCAN_T(SCAN_TURNS), 0, g.stream>>>(*s, sc, act, state, sd, rows, seq0, pos);
  };
  switch (sd.Np / 64u) {
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 3: go(std::integral_constant<int, 3>{}); break;
    default: go(std::integral_constant<int, 4>{}); break;
  }
  count_launch();
  return check_launch();
}
