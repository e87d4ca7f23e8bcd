// Mixture of gated experts over rows whose router logits are known (AdamahExpertsSpec).  Scores, choice and weights are
// float32.
//
// One row: two launches.  Every workgroup chooses the experts for itself (a row of logits is small: each candidate counts
// those that beat it), so nothing has to wait for a launch that only chooses.  k_experts_in: gate and up rows of the chosen
// experts, two matrix rows a wave; k_experts_out: a row of the result is one dot product over the shared expert's activations
// and the chosen experts', each run times its expert's weight; the row itself times the weights of those that
// give it back is added at the end.
//
// More rows: k_experts_choose (a wave per row), k_experts_list (a workgroup per expert: its rows in order), then the two
// products over tiles of one expert's rows each: k_experts_tiled or k_experts_many (bfloat16 operands), k_experts_f32.  The rows of an
// expert are picked up where they lie; activations and results are laid down so that k_experts_sum can add up a row's in a
// fixed order: what a row gets does not depend on which other rows there are.
#include "linear_common.h"
#include <algorithm>

namespace adamah {

typedef AdamahExpertsSpec XSpec;
#define MAX_CHOICES 1024u
#define MAX_TOP 64u
#define MAX_STEP 32768u      // activations of one row
#define XSTEP 512u

// ---- one row --------------------------------------------------------------------------------------------------------
struct Choice { uint32_t id[MAX_TOP]; float wt[MAX_TOP]; uint32_t n; float back; };
struct Chosen : Choice { float score[MAX_CHOICES], by[MAX_CHOICES]; };
// The chosen experts with matrices, best first, and their weights; n of them; back: what the row itself is multiplied by.
// Up to 64 candidates every wave chooses among by itself, one a lane, and all write the same words: no barrier (a wave may read
// them at once), and what it needs (choose_ask) can be asked for ahead of everything else.
struct Asked { float z, c; };
__device__ __forceinline__ Asked choose_ask(const XSpec& s, const float* act) {
  const uint32_t i = min(threadIdx.x & 63u, s.experts + s.identity - 1u);
  return {act[s.logits + i], act[s.correction + i]};
}
__device__ __forceinline__ void choose_row(const XSpec& s, const float* act, const Asked& q, Chosen& ch) {
  const uint32_t tid = threadIdx.x, lane = tid & 63u, n = s.experts + s.identity;
  const float *z = act + s.logits, *corr = act + s.correction;
  if (n <= 64u) {
    const float mx = wave_max(q.z), e = lane < n ? expf(q.z - mx) : 0.f, p = e * (1.0f / wave_add(e)), me = p + q.c;
    uint32_t rank = 0;
#pragma unroll 8
    for (uint32_t j = 0; j < n; j++) {
      const float by = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(me), (int)j));
      rank += by > me || (by == me && j < lane) ? 1u : 0u;
    }
    const int to = (int)((lane < n ? rank : lane) * 4u);     // lane r gets the candidate of rank r (nothing: 0)
    const uint32_t id = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)(lane + 1u)) - 1u;
    const float w = __uint_as_float((uint32_t)__builtin_amdgcn_ds_permute(to, (int)__float_as_uint(p)));
    const bool real = lane < s.top && id < s.experts;
    const uint64_t mask = __ballot(real);
    const float back = wave_add(lane < s.top && !real ? w : 0.f);
    const uint32_t at = __popcll(mask & ((1ull << lane) - 1ull));
    if (real) { ch.id[at] = id; ch.wt[at] = w; }
    if (lane == 0) { ch.n = __popcll(mask); ch.back = back; }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    return;
  }
  float mx = -3.4e38f, sum = 0.f;
  for (uint32_t i = lane; i < n; i += 64u) mx = fmaxf(mx, z[i]);
  mx = wave_max(mx);
  for (uint32_t i = lane; i < n; i += 64u) sum += expf(z[i] - mx);
  const float inv = 1.0f / wave_add(sum);
  for (uint32_t i = tid; i < n; i += XSTEP) { const float p = expf(z[i] - mx) * inv; ch.score[i] = p; ch.by[i] = p + corr[i]; }
  if (tid < MAX_TOP) { ch.id[tid] = 0xFFFFFFFFu; ch.wt[tid] = 0.f; }
  __syncthreads();
  for (uint32_t i = tid; i < n; i += XSTEP) {
    const float me = ch.by[i];
    uint32_t rank = 0;
#pragma unroll 8
    for (uint32_t j = 0; j < n; j++) rank += ch.by[j] > me || (ch.by[j] == me && j < i) ? 1u : 0u;
    if (rank < s.top) { ch.id[rank] = i; ch.wt[rank] = ch.score[i]; }
  }
  __syncthreads();
  if (tid < 64u) {
    const uint32_t e = ch.id[lane];
    const float w = ch.wt[lane];
    const bool real = e < s.experts;
    const uint64_t mask = __ballot(real);
    const float back = wave_add(real ? 0.f : w);
    const uint32_t at = __popcll(mask & ((1ull << lane) - 1ull));
    if (real) { ch.id[at] = e; ch.wt[at] = w; }              // (one wave: every lane has read its own before)
    if (lane == 0) { ch.n = __popcll(mask); ch.back = back; }
  }
  __syncthreads();
}

__device__ __forceinline__ void fma8(float& a, const uint4& w, const float4& lo, const float4& hi) {
  a = fmaf(bf_lo(w.x), lo.x, a); a = fmaf(bf_hi(w.x), lo.y, a); a = fmaf(bf_lo(w.y), lo.z, a); a = fmaf(bf_hi(w.y), lo.w, a);
  a = fmaf(bf_lo(w.z), hi.x, a); a = fmaf(bf_hi(w.z), hi.y, a); a = fmaf(bf_lo(w.w), hi.z, a); a = fmaf(bf_hi(w.w), hi.w, a);
}

// x in LDS as two planes (elements 0..3 / 4..7 of every eight), so that a lane's two 16-byte reads are conflict free.
#define PLANE(i, half) ((((i) >> 2) & 1u) * (half) + ((i) >> 3) * 4u + ((i) & 3u))

// `left` runs of two buffers, both asked for already: each is asked for again behind its use while there are more
#define RUNS_OF_TWO(left, run, fetch)                          \
  do {                                                         \
    for (; left > 3u; left -= 2u) { run(0); fetch(0); run(1); fetch(1); } \
    if (left == 3u) { run(0); fetch(0); run(1); run(0); }      \
    else if (left == 2u) { run(0); run(1); }                   \
    else if (left == 1u) run(0);                               \
  } while (0)
// The first run of columns is asked for before x is staged, as soon as the choice is known; not two at a time (6 x 1024 pairs of rows
// of 2048, 50 MB: 15.2 us, so 13.5).
template <int U>
__global__ void __launch_bounds__(XSTEP)
k_experts_in(const bf16_t* __restrict__ W, float* act, Choice* choice, const XSpec s) {
  extern __shared__ __attribute__((aligned(16))) float xs[];
  __shared__ Chosen ch;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, kp = s.k_stride, half = kp >> 1, F = (s.ff + 15u) & ~15u;
  const Asked q = choose_ask(s, act);
  // (no load under a condition, here and below: each would wait for the one before; short rows have two values a thread)
  constexpr uint32_t R = U == 1 ? 2 : 4;
  float v[R];
#pragma unroll
  for (uint32_t u = 0; u < R; u++) v[u] = act[s.x + min(threadIdx.x + u * XSTEP, s.width - 1u)];
  choose_row(s, act, q, ch);
  const uint32_t n_tasks = ch.n * F;
  uint32_t task = blockIdx.x * (XSTEP / 64u) + wave, k0 = lane * 8u;
  uint4 g[U], h[U];
  const auto fetch = [&] {
    const uint32_t j = task / F, t = task - j * F;
    const bf16_t* wg = W + s.gate_up + (uint64_t)ch.id[j] * s.gate_up_step + (uint64_t)((t >> 4) * 32u + (t & 15u)) * kp;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint32_t k = min(k0 + 512u * u, kp - 8u);
      g[u] = *(const uint4*)(wg + k); h[u] = *(const uint4*)(wg + (uint64_t)16u * kp + k);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  if (task < n_tasks) fetch();
#pragma unroll
  for (uint32_t u = 0; u < R; u++) {
    const uint32_t i = threadIdx.x + u * XSTEP;
    if (i < kp) xs[PLANE(i, half)] = i < s.width ? v[u] : 0.f;
  }
  for (uint32_t i = threadIdx.x + R * XSTEP; i < kp; i += XSTEP) xs[PLANE(i, half)] = i < s.width ? act[s.x + i] : 0.f;
  __syncthreads();
  float a = 0.f, b = 0.f;
  while (task < n_tasks) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint32_t k = k0 + 512u * u;
      if (k >= kp) break;
      const float4 lo = *(const float4*)(xs + (k >> 1)), hi = *(const float4*)(xs + half + (k >> 1));
      fma8(a, g[u], lo, hi); fma8(b, h[u], lo, hi);
    }
    const uint32_t done = task;
    const bool last = k0 - lane * 8u + 512u * U >= kp;
    if (last) { k0 = lane * 8u; task += gridDim.x * (XSTEP / 64u); } else k0 += 512u * U;
    if (task < n_tasks) fetch();
    if (last) {
      a = wave_add(a); b = wave_add(b);
      const uint32_t j = done / F;
      if (lane == 0) act[s.act + j * s.ff_stride + done - j * F] = silu_f(a) * b;
      a = b = 0.f;
    }
  }
  if (blockIdx.x == 0u && threadIdx.x < MAX_TOP) {           // for the launch behind this one
    choice->id[threadIdx.x] = ch.id[threadIdx.x]; choice->wt[threadIdx.x] = ch.wt[threadIdx.x];
    if (threadIdx.x == 0u) { choice->n = ch.n; choice->back = ch.back; }
  }
}

// A row of the result a wave: the chosen experts' columns, then the shared expert's.  LDS holds the activations times their experts'
// weights, by place in the choice (whatever its length), the shared expert's behind all places.  Activations and the choice are asked for
// together; so are the shared expert's first columns where which ones a lane has does not hang on the choice, ahead of all others.  Two
// runs of U times 512 columns in flight besides.
// What bounds it is the weights' way in and what stands ahead of it (2048 rows of 6 x 1024 and 2048 columns, 33.5 MB, 6.9 us at a
// large copy's rate: 14.2 us with two rows a wave, half the CUs at work and nothing ahead of the choice, 12.5 so).
template <int U>
__global__ void __launch_bounds__(XSTEP)
k_experts_out(const bf16_t* __restrict__ W, float* act, const Choice* __restrict__ choice, const XSpec s, uint32_t magic) {
  extern __shared__ __attribute__((aligned(16))) float xs[];
  __shared__ Choice ch;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, fs = s.ff_stride, stride = gridDim.x * (XSTEP / 64u);
  const uint32_t sk = s.shared_ff ? s.shared_ff_stride : 0u, places = min(s.top, s.experts) * fs, held = places + sk, half = held >> 1;
  const uint32_t row0 = blockIdx.x * (XSTEP / 64u) + wave;
  const uint32_t id = choice->id[lane], n_ch = choice->n;    // (a word a lane: MAX_TOP of them)
  const float wt = choice->wt[lane], back = choice->back;
  const float gate = act[s.logits + s.experts + s.identity - (s.shared_ff ? 0u : 1u)];
  // Sixteen values a thread (of a short row two) asked for at once and no load under a condition
  constexpr uint32_t R = U == 1 ? 2 : 16;
  const auto value = [&](uint32_t i0) {
    const uint32_t i = min(i0, held - 1u), j = __umulhi(i, magic);
    return act[i < places ? s.act + j * fs + min(i - j * fs, s.ff - 1u) : s.shared_act + min(i - places, s.shared_ff - 1u)];
  };
  float v[R];
#pragma unroll
  for (uint32_t u = 0; u < R; u++) v[u] = value(threadIdx.x + u * XSTEP);
  // runs of a row: `chosen` of them up to column `edge`, the others behind it; the first of these is at hand for the wave's first row
  const bool early = (fs & 511u) == 0u && sk >= 512u * U;
  uint4 p[2][U], e[U];
  if (early)
#pragma unroll
    for (int u = 0; u < U; u++) e[u] = *(const uint4*)(W + s.shared_down + (uint64_t)min(row0, s.width - 1u) * sk + lane * 8u + 512u * u);
  __builtin_amdgcn_sched_barrier(0);
  ch.id[lane] = id; ch.wt[lane] = wt;                        // (every wave the same words, for itself)
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  const auto runs_of = [](uint32_t columns) { return (columns + 512u * U - 1u) / (512u * U); };
  const uint32_t body = n_ch * fs, end = body + sk, edge = early ? body : end, chosen = runs_of(edge), all = chosen + runs_of(end - edge);
  const auto base = [&](uint32_t run) { return (run < chosen ? run * (512u * U) : edge + (run - chosen) * (512u * U)) + lane * 8u; };
  const auto limit = [&](uint32_t run) { return run < chosen ? edge : end; };
  const auto skip = [&](uint32_t row, uint32_t run) { return early && row == row0 && run == chosen; };
  uint32_t from = row0, fr = skip(row0, 0u) ? 1u : 0u;       // the run to be asked for
  const auto wrap = [&](uint32_t& row, uint32_t& run) { if (run >= all) { run = 0u; row += stride; } };
  wrap(from, fr);
  const auto fetch = [&](int x) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint32_t k = min(base(fr) + 512u * u, limit(fr) - 8u), j = min(__umulhi(k, magic), (uint32_t)MAX_TOP - 1u);
      const uint64_t at = k < body ? s.down + (uint64_t)ch.id[j] * s.down_step + (uint64_t)from * fs + (k - j * fs)
                                   : s.shared_down + (uint64_t)from * sk + (k - body);
      p[x][u] = *(const uint4*)(W + at);
    }
    fr++;
    if (skip(from, fr)) fr++;
    wrap(from, fr);
    __builtin_amdgcn_sched_barrier(0);
  };
  uint32_t left = row0 < s.width ? ((s.width - 1u - row0) / stride + 1u) * all - (early ? 1u : 0u) : 0u;
  if (left > 0u) fetch(0);
  if (left > 1u) fetch(1);
  const float sg = sigmoid_f(gate);
  const auto put = [&](uint32_t i, float x) {
    const uint32_t j = min(__umulhi(i, magic), (uint32_t)MAX_TOP - 1u);
    if (i < held) xs[PLANE(i, half)] = i < places ? (i - j * fs < s.ff ? x * ch.wt[j] : 0.f) : i - places < s.shared_ff ? x * sg : 0.f;
  };
#pragma unroll
  for (uint32_t u = 0; u < R; u++) put(threadIdx.x + u * XSTEP, v[u]);
  for (uint32_t i = threadIdx.x + R * XSTEP; i < held; i += XSTEP) put(i, value(i));
  __syncthreads();
  float a = 0.f;
  uint32_t row = row0, r = 0u;
  const auto add = [&](const uint4 (&w)[U]) {                // run r of the row
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint32_t k = base(r) + 512u * u, i = k < body ? k : k - body + places;
      if (k >= limit(r)) break;
      const float4 lo = *(const float4*)(xs + (i >> 1)), hi = *(const float4*)(xs + half + (i >> 1));
      fma8(a, w[u], lo, hi);
    }
    r++;
  };
  const auto done = [&] {
    if (r < all) return;
    a = wave_add(a);
    if (lane == 0) {
      const float y = fmaf(back, act[s.x + row], a);
      float* d = act + s.out + row;
      *d = s.epi ? *d + y : y;
    }
    a = 0.f; r = 0u; row += stride;
  };
  const auto at_hand = [&] { if (skip(row, r)) add(e); };
  if (all == 0u) {                                           // nothing chosen has a matrix, and nothing is shared
    while (row < s.width) done();
    return;
  }
  if (row < s.width) { at_hand(); done(); }
  const auto run = [&](int x) { add(p[x]); at_hand(); done(); };
  RUNS_OF_TWO(left, run, fetch);
}

// ---- more rows ------------------------------------------------------------------------------------------------------
// Entry row * top + j of `ids` / `wts`: the j-th expert of a row, best first, and its weight.
template <int NV>
__global__ void __launch_bounds__(256)
k_experts_choose(const XSpec s, const float* __restrict__ act, uint32_t* __restrict__ ids, float* __restrict__ wts, uint32_t rows) {
  const uint32_t lane = threadIdx.x & 63u, row = blockIdx.x * 4u + (threadIdx.x >> 6), n = s.experts + s.identity;
  if (row >= rows) return;
  const float* z = act + s.logits + (uint64_t)row * s.logits_stride;
  float p[NV], by[NV], mx = -3.4e38f, sum = 0.f;
#pragma unroll
  for (int i = 0; i < NV; i++) { const uint32_t e = lane + 64u * i; p[i] = e < n ? z[e] : -3.4e38f; mx = fmaxf(mx, p[i]); }
  mx = wave_max(mx);
#pragma unroll
  for (int i = 0; i < NV; i++) { p[i] = lane + 64u * i < n ? expf(p[i] - mx) : 0.f; sum += p[i]; }
  const float inv = 1.0f / wave_add(sum);
#pragma unroll
  for (int i = 0; i < NV; i++) { const uint32_t e = lane + 64u * i; p[i] *= inv; by[i] = e < n ? p[i] + act[s.correction + e] : -3.4e38f; }
  uint32_t gone = 0;                                        // bit i: candidate lane + 64 i has been taken
  for (uint32_t j = 0; j < s.top; j++) {
    float top = -3.4e38f, w = 0.f;
    uint32_t at = 0xFFFFFFFFu;
#pragma unroll
    for (int i = 0; i < NV; i++) {
      const uint32_t e = lane + 64u * i;
      if (e < n && !(gone >> i & 1u) && (at == 0xFFFFFFFFu || by[i] > top)) { top = by[i]; at = e; w = p[i]; }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float t2 = __shfl_xor(top, o, 64), w2 = __shfl_xor(w, o, 64);
      const uint32_t a2 = (uint32_t)__shfl_xor((int)at, o, 64);
      if (a2 != 0xFFFFFFFFu && (at == 0xFFFFFFFFu || t2 > top || (t2 == top && a2 < at))) { top = t2; at = a2; w = w2; }
    }
    if ((at & 63u) == lane) gone |= 1u << (at >> 6);
    if (lane == 0) { ids[(uint64_t)row * s.top + j] = at; wts[(uint64_t)row * s.top + j] = w; }
  }
}

// A workgroup per expert: the entries that chose it, in order, at list + e * rows; cnt[e]: how many.  A wave takes a run of entries, 64 neighbours a load,
// and counts and places them by the lanes that hold the expert; the first KEPT loads are asked for at once and kept for the second walk.  Bound by latency:
// 12288 entries in 32 lists 5.1 us (13.1 with a run of neighbours a thread); as many loads and waves as the entries need and no more, 48 entries 1.8 us (3.8 with 16 of
// either), 960 2.6 (4.3), 3584 3.0 (4.4).
template <uint32_t WAVES, uint32_t KEPT>
__global__ void __launch_bounds__(64 * WAVES)
k_experts_list(const uint32_t* __restrict__ ids, uint32_t* __restrict__ list, uint32_t* __restrict__ cnt, uint32_t rows, uint32_t top) {
  __shared__ uint32_t part[WAVES];
  const uint32_t e = blockIdx.x, lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), total = rows * top;
  const uint32_t run = (total + WAVES * 64u - 1u) / (WAVES * 64u), lo = wave * run * 64u;      // (of 64 entries)
  const auto id_at = [&](uint32_t j) { return ids[min(lo + 64u * j + lane, total - 1u)]; };
  const auto mine = [&](uint32_t j, uint32_t id) { return (uint64_t)__ballot(id == e && lo + 64u * j + lane < total); };      // which lanes' entries chose it
  uint64_t kept[KEPT];
  {
    uint32_t id[KEPT];
#pragma unroll
    for (uint32_t j = 0; j < KEPT; j++) id[j] = id_at(j);
#pragma unroll
    for (uint32_t j = 0; j < KEPT; j++) kept[j] = j < run ? mine(j, id[j]) : 0u;
  }
  uint32_t n = 0;
#pragma unroll
  for (uint32_t j = 0; j < KEPT; j++) n += __popcll(kept[j]);
#pragma unroll 8
  for (uint32_t j = KEPT; j < run; j++) n += __popcll(mine(j, id_at(j)));
  if (lane == 0u) part[wave] = n;
  __syncthreads();
  uint32_t at = 0;
  for (uint32_t w = 0; w < wave; w++) at += part[w];
  if (wave == WAVES - 1u && lane == 0u) cnt[e] = min(at + n, rows);             // (a row takes an expert once)
  const auto place = [&](uint32_t j, uint64_t m) {
    const uint32_t to = at + __popcll(m & ((1ull << lane) - 1ull));
    if ((m >> lane & 1ull) && to < rows) list[(uint64_t)e * rows + to] = lo + 64u * j + lane;
    at += __popcll(m);
  };
#pragma unroll
  for (uint32_t j = 0; j < KEPT; j++) place(j, kept[j]);
#pragma unroll 8
  for (uint32_t j = KEPT; j < run; j++) place(j, mine(j, id_at(j)));
}

// Which tile a workgroup has: tiles are numbered expert by expert, within one by matrix rows and then by tokens, so that
// neighbours share the matrix rows; workgroups land on the eight dies in turn, and every die gets a run of neighbours.
// Every wave finds it for itself from the experts' counts.
struct Tile { uint32_t e, count, first, m, n; };     // expert, its rows, its first activation row, tile of tokens / matrix rows
// What stands ahead of a tile is its launch's time once more a round, so sums and running sums stay in the vector unit and counts are loaded once.
__device__ __forceinline__ uint32_t running_sum(uint32_t v) {      // of this lane and those before it
#define RUN_STEP(ctrl, rows) v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, rows, 0xF, false)
  RUN_STEP(0x111, 0xF); RUN_STEP(0x112, 0xF); RUN_STEP(0x114, 0xF); RUN_STEP(0x118, 0xF);     // 1, 2, 4, 8 lanes back in a row of 16
  RUN_STEP(0x142, 0xA); RUN_STEP(0x143, 0xC);                                                 // the row before's last lane, the lower half's
#undef RUN_STEP
  return v;
}
__device__ __forceinline__ uint32_t lane_of(uint32_t v, int l) { return (uint32_t)__builtin_amdgcn_readlane((int)v, l); }
// counts of the first 64 experts, a lane each
__device__ __forceinline__ uint32_t first_counts(const uint32_t* __restrict__ cnt, uint32_t experts) {
  const uint32_t lane = threadIdx.x & 63u, c = cnt[min(lane, experts - 1u)];
  return lane < experts ? c : 0u;
}
// tiles of bm rows over all experts
__device__ __forceinline__ uint32_t count_tiles(const uint32_t* __restrict__ cnt, uint32_t experts, uint32_t c0, uint32_t bm) {
  uint32_t n = (c0 + bm - 1u) / bm;
  for (uint32_t e = 64u + (threadIdx.x & 63u); e < experts; e += 64u) n += (cnt[e] + bm - 1u) / bm;
  return lane_of(running_sum(n), 63);
}
__device__ __forceinline__ bool pick_tile(const uint32_t* __restrict__ cnt, uint32_t experts, uint32_t c0, uint32_t bm, uint32_t total, uint32_t tiles_n, Tile& t) {
  const uint32_t lane = threadIdx.x & 63u;
  total *= tiles_n;
  const uint32_t per = (total + 7u) / 8u, id = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per || id >= total) return false;
  uint32_t tiles = 0, rows = 0;                              // ahead of this run of 64 experts
  for (uint32_t b = 0; b < experts; b += 64u) {
    const uint32_t c = b == 0u ? c0 : b + lane < experts ? cnt[b + lane] : 0u, mine = (c + bm - 1u) / bm * tiles_n;
    const uint32_t ts = running_sum(mine), rs = running_sum(c);
    const uint64_t here = __ballot(tiles + ts > id);
    if (here) {
      const int l = __ffsll((unsigned long long)here) - 1;
      const uint32_t tm = lane_of(mine, l) / tiles_n, at = id - (tiles + lane_of(ts - mine, l));
      t.e = b + (uint32_t)l; t.count = lane_of(c, l); t.first = rows + lane_of(rs - c, l);
      t.m = at % tm; t.n = at / tm;
      return true;
    }
    tiles += lane_of(ts, 63); rows += lane_of(rs, 63);
  }
  return false;
}
// results: first product -> the operand rows of the activations, second -> a row of `parts` per entry
template <class T>
__device__ __forceinline__ void put_activation(const XSpec& s, T* opnd, uint32_t arow, uint32_t n0, f4_t gt, f4_t up) {
  const uint32_t c = (n0 >> 5) * 16u + (n0 & 15u), F = (s.ff + 15u) & ~15u;
  typedef T t4 __attribute__((ext_vector_type(4)));
  t4 y;
#pragma unroll
  for (int i = 0; i < 4; i++) y[i] = (T)(silu_f(gt[i]) * up[i]);
  if (c < F) *(t4*)(opnd + s.act_opnd + (uint64_t)arow * s.ff_stride + c) = y;       // (F: whole runs of 16; rows start on 8 elements)
}
__device__ __forceinline__ void put_part(const XSpec& s, float* parts, uint32_t entry, uint32_t n0, f4_t v) {
  float* d = parts + (uint64_t)entry * s.width + n0;
  if ((s.width & 3u) == 0u) { if (n0 < s.width) *(f4_t*)d = v; return; }
#pragma unroll
  for (int i = 0; i < 4; i++) if (n0 + i < s.width) d[i] = v[i];
}

// la: ST BN 64 elements, lb: STX BM 64; ONCE: weights that hardly any other tile reads
template <int BM, int BN, int WM, int WN, int ST, int STX, bool ONCE, bool IN>
__device__ __forceinline__ void experts_tile(const bf16_t* __restrict__ W, bf16_t* opnd, float* __restrict__ parts, const XSpec& s, const uint32_t* __restrict__ list,
                                             const uint32_t* __restrict__ cnt, uint32_t c0, uint32_t total, uint32_t rows, uint32_t tiles_n, bf16_t* la, bf16_t* lb) {
  constexpr int NTN = BN / WN / 16, NTM = BM / WM / 16;
  const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t c = lane & 15u, kg = lane >> 4, kp = IN ? s.k_stride : s.ff_stride, n = IN ? 2u * ((s.ff + 15u) & ~15u) : s.width;
  Tile t;
  if (!pick_tile(cnt, s.experts, c0, BM, total, tiles_n, t)) return;
  const uint32_t m0 = t.m * BM, n0 = t.n * BN, wn = (wave % WN) * (BN / WN), wm = (wave / WN) * (BM / WM);
  const bf16_t* We = W + (IN ? s.gate_up + (uint64_t)t.e * s.gate_up_step : s.down + (uint64_t)t.e * s.down_step);
  const uint32_t* le = list + (uint64_t)t.e * rows;
  f4_t acc[NTN][NTM];
  tile_product<BM, BN, WM, WN, ST, 1, STX, ONCE>(acc, TileRows<BN, WM * WN, ONCE>(wave, lane, [&](uint32_t r) { return We + (uint64_t)min(n0 + r, n - 1u) * kp; }),
                                                 TileRows<BM, WM * WN>(wave, lane, [&](uint32_t r) {
                                                   const uint32_t i = min(m0 + r, t.count - 1u);
                                                   return opnd + (IN ? s.opnd + (uint64_t)(le[i] / s.top) * kp : s.act_opnd + (uint64_t)(t.first + i) * kp);
                                                 }), kp, 0u, kp, la, lb, wave, lane, m0 + wm < t.count);
#pragma unroll
  for (int j = 0; j < NTM; j++) {
    const uint32_t i = m0 + wm + 16u * j + c;
    if (i >= t.count) continue;
    if (IN) {
#pragma unroll
      for (int q = 0; q < NTN; q += 2) put_activation(s, opnd, t.first + i, n0 + wn + 16u * q + 4u * kg, acc[q][j], acc[q + 1][j]);
    } else {
      const uint32_t entry = le[i];
#pragma unroll
      for (int q = 0; q < NTN; q++) put_part(s, parts, entry, n0 + wn + 16u * q + 4u * kg, acc[q][j]);
    }
  }
}

// few rows an expert
template <bool IN>
__global__ void __launch_bounds__(256)
k_experts_tiled(const bf16_t* __restrict__ W, bf16_t* opnd, float* __restrict__ parts, const XSpec s, const uint32_t* __restrict__ list,
                const uint32_t* __restrict__ cnt, uint32_t rows, uint32_t tiles_n) {
  __shared__ __attribute__((aligned(16))) bf16_t la[4 * 64 * 64], lb[4 * 64 * 64];
  const uint32_t c0 = first_counts(cnt, s.experts);
  experts_tile<64, 64, 2, 2, 4, 4, false, IN>(W, opnd, parts, s, list, cnt, c0, count_tiles(cnt, s.experts, c0, 64u), rows, tiles_n, la, lb);
}
// More: tiles of 128, 192 or 256 rows by 256 matrix rows, a workgroup a CU.  A launch takes as many rounds of tiles as a CU gets, whatever the last one
// holds, and that hangs on the experts' counts, which only the device knows: every workgroup finds by them the size that costs least.  The results do not
// hang on it.  A round takes what stands around a tile's steps and those steps, which are longer the more CUs have a tile, and less than in proportion to the rows
// (weights and tokens on their way into LDS bound them; a third buffer for the weights, which come from memory: 2048 rows, 6 of 34 experts 1024 wide in 2048, both
// products 208 us with two, 196 so).  Over 16 shapes of 3 .. 128 experts, 1 .. 64 steps and 8 .. 600 rows an expert, weights from memory, both products take 0.6 %
// longer than in the best sizes (64 rows among them) in the mean, 12 % at most (16 experts 1024 wide in 2048, 64 rows: 70 us and 62).
#define MANY_SIZES 3u
struct Chip { uint32_t cus, magic; float inv; };                                  // tiles / cus = umulhi(tiles, magic)
__host__ __device__ __forceinline__ float many_us(uint32_t size, uint32_t tiles, uint32_t steps, const Chip& c) {      // of `tiles` tiles of 128 + 64 size rows
  const float around = 9.f + (float)size, alone = size == 0u ? 0.6f : size == 1u ? 0.75f : 0.85f, full = size == 0u ? 0.47f : size == 1u ? 0.7f : 1.f;
  const uint32_t rounds = (uint32_t)((uint64_t)(tiles + c.cus - 1u) * c.magic >> 32);
  return (float)rounds * (around + (float)steps * (alone + full * (rounds > 1u ? 1.f : (float)tiles * c.inv)));
}
// Weights that one tile alone reads do not stay in the L2, where the tokens are, if every CU has a tile (32 experts 1024 wide in 2048, 50 rows each: 67 us and
// so 60 in tiles of 128, 69 and 61 in tiles of 256; 8 of them, 128 rows, a CU in four at work: 38 and 40; 64 of 4 steps, 95 rows: 16.5 and 18.2).
struct Many { uint32_t size; bool once; };
__host__ __device__ __forceinline__ Many many_pick(const uint32_t (&tiles_m)[MANY_SIZES], uint32_t experts_with_rows, uint32_t tiles_n, uint32_t steps, const Chip& c) {
  const float u0 = many_us(0u, tiles_m[0] * tiles_n, steps, c), u1 = many_us(1u, tiles_m[1] * tiles_n, steps, c), u2 = many_us(2u, tiles_m[2] * tiles_n, steps, c);
  const uint32_t i = u0 <= u1 && u0 <= u2 ? 0u : u1 <= u2 ? 1u : 2u, t = i == 0u ? tiles_m[0] : i == 1u ? tiles_m[1] : tiles_m[2];
  return {i, t == experts_with_rows && t * tiles_n >= c.cus && steps >= 8u};
}
template <bool IN>
__global__ void __launch_bounds__(512)
k_experts_many(const bf16_t* __restrict__ W, bf16_t* opnd, float* __restrict__ parts, const XSpec s, const uint32_t* __restrict__ list,
               const uint32_t* __restrict__ cnt, uint32_t rows, uint32_t tiles_n, const Chip chip) {
  __shared__ __attribute__((aligned(16))) bf16_t lds[(3 * 256 + 2 * 256) * 64];
  const uint32_t c0 = first_counts(cnt, s.experts);
  uint32_t t[MANY_SIZES] = {(c0 + 127u) / 128u, (c0 + 191u) / 192u, (c0 + 255u) / 256u}, some = __popcll(__ballot(c0 != 0u));
  for (uint32_t b = 64u; b < s.experts; b += 64u) {
    const uint32_t e = b + (threadIdx.x & 63u), c = e < s.experts ? cnt[e] : 0u;
    t[0] += (c + 127u) / 128u; t[1] += (c + 191u) / 192u; t[2] += (c + 255u) / 256u;
    some += __popcll(__ballot(c != 0u));
  }
#pragma unroll
  for (uint32_t i = 0; i < MANY_SIZES; i++) t[i] = lane_of(running_sum(t[i]), 63);
  const Many m = many_pick(t, some, tiles_n, (IN ? s.k_stride : s.ff_stride) >> 6, chip);
  bf16_t* const lb = lds + 3 * 256 * 64;
#define MANY_TILE(BM, STX, ONCE) experts_tile<BM, 256, 2, 4, 3, STX, ONCE, IN>(W, opnd, parts, s, list, cnt, c0, t[BM / 64 - 2], rows, tiles_n, lds, lb)
  if (m.size == 0u) { if (m.once) MANY_TILE(128, 3, true); else MANY_TILE(128, 3, false); }
  else if (m.size == 1u) { if (m.once) MANY_TILE(192, 2, true); else MANY_TILE(192, 2, false); }
  else { if (m.once) MANY_TILE(256, 2, true); else MANY_TILE(256, 2, false); }
#undef MANY_TILE
}

template <bool IN>
__global__ void __launch_bounds__(256)
k_experts_f32(const bf16_t* __restrict__ W, float* opnd, float* __restrict__ parts, const XSpec s, const uint32_t* __restrict__ list,
              const uint32_t* __restrict__ cnt, uint32_t rows, uint32_t tiles_n) {
  __shared__ __attribute__((aligned(16))) float la[64][36], lb[64][36];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, c = lane & 15u, kg = lane >> 4;
  const uint32_t kp = IN ? s.k_stride : s.ff_stride, n = IN ? 2u * ((s.ff + 15u) & ~15u) : s.width;
  Tile t;
  const uint32_t c0 = first_counts(cnt, s.experts);
  if (!pick_tile(cnt, s.experts, c0, 64u, count_tiles(cnt, s.experts, c0, 64u), tiles_n, t)) return;
  const uint32_t m0 = t.m * 64u, n0 = t.n * 64u, wn = (wave & 1u) * 32u, wm = (wave >> 1) * 32u, lr = tid >> 2, lc = (tid & 3u) * 8u;
  const bf16_t* We = W + (IN ? s.gate_up + (uint64_t)t.e * s.gate_up_step : s.down + (uint64_t)t.e * s.down_step);
  const uint32_t* le = list + (uint64_t)t.e * rows;
  const uint32_t xi = min(m0 + lr, t.count - 1u);
  f4_t acc[2][2];
  tile_product_f32(acc, We + (uint64_t)min(n0 + lr, n - 1u) * kp + lc,
                   opnd + (IN ? s.opnd + (uint64_t)(le[xi] / s.top) * kp : s.act_opnd + (uint64_t)(t.first + xi) * kp) + lc, kp, la, lb);
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const uint32_t i = m0 + wm + 16u * j + c;
    if (i >= t.count) continue;
    if (IN) put_activation(s, opnd, t.first + i, n0 + wn + 4u * kg, acc[0][j], acc[1][j]);
    else {
      const uint32_t entry = le[i];
#pragma unroll
      for (int q = 0; q < 2; q++) put_part(s, parts, entry, n0 + wn + 16u * q + 4u * kg, acc[q][j]);
    }
  }
}

// A row's results, its own times the weights of the experts that give it back, and the shared expert's.
__global__ void __launch_bounds__(256)
k_experts_sum(const XSpec s, float* act, const float* __restrict__ parts, const uint32_t* __restrict__ ids, const float* __restrict__ wts,
              uint32_t shared, uint32_t shared_stride) {
  __shared__ float w[MAX_TOP];
  __shared__ uint32_t real[MAX_TOP];
  const uint32_t row = blockIdx.x, tid = threadIdx.x;
  if (tid < s.top) { w[tid] = wts[(uint64_t)row * s.top + tid]; real[tid] = ids[(uint64_t)row * s.top + tid] < s.experts ? 1u : 0u; }
  __syncthreads();
  float back = 0.f;
  for (uint32_t j = 0; j < s.top; j++) back += real[j] ? 0.f : w[j];
  const float sg = s.shared_ff ? sigmoid_f(act[s.logits + (uint64_t)row * s.logits_stride + s.experts + s.identity]) : 0.f;
  const float *x = act + s.x + (uint64_t)row * s.x_stride, *sh = act + shared + (uint64_t)row * shared_stride;
  const float* p = parts + (uint64_t)row * s.top * s.width;
  float* d = act + s.out + (uint64_t)row * s.out_stride;
  // Four columns a thread and no load under a condition (an entry that gives the row back has no result: what lies there is read and
  // left out): 2048 rows of 2048, 6 of 34: 45 us with a float a load and a branch for each, so: 25; 10 rows 26 and 6.
  if (((s.width | s.x | s.x_stride | shared | shared_stride | s.out | s.out_stride) & 3u) == 0u) {
    for (uint32_t i = tid * 4u; i < s.width; i += 1024u) {
      const f4_t xv = *(const f4_t*)(x + i), hv = *(const f4_t*)(sh + i);
      f4_t y = {back * xv[0], back * xv[1], back * xv[2], back * xv[3]};
      for (uint32_t j0 = 0; j0 < s.top; j0 += 6u) {
        f4_t v[6];
#pragma unroll
        for (uint32_t u = 0; u < 6u; u++) v[u] = *(const f4_t*)(p + (uint64_t)min(j0 + u, s.top - 1u) * s.width + i);
#pragma unroll
        for (uint32_t u = 0; u < 6u; u++) {
          const uint32_t j = min(j0 + u, s.top - 1u);
          const bool on = j0 + u < s.top && real[j];
          const float wj = w[j];
#pragma unroll
          for (int e = 0; e < 4; e++) y[e] = on ? fmaf(wj, v[u][e], y[e]) : y[e];
        }
      }
      if (s.shared_ff)
#pragma unroll
        for (int e = 0; e < 4; e++) y[e] = fmaf(sg, hv[e], y[e]);
      if (s.epi) { const f4_t o = *(const f4_t*)(d + i); y = (f4_t){o[0] + y[0], o[1] + y[1], o[2] + y[2], o[3] + y[3]}; }
      *(f4_t*)(d + i) = y;
    }
    return;
  }
  for (uint32_t i = tid; i < s.width; i += 256u) {
    float y = back * x[i];
#pragma unroll 4
    for (uint32_t j = 0; j < s.top; j++) if (real[j]) y = fmaf(w[j], p[(uint64_t)j * s.width + i], y);
    if (s.shared_ff) y = fmaf(sg, sh[i], y);
    d[i] = s.epi ? d[i] + y : y;
  }
}

static Scratch g_experts;
void experts_release() { scratch_free(g_experts); }

static Chip chip() {
  const uint32_t n = (uint32_t)g.n_cu;
  return {n, (uint32_t)((0x100000000ull + n - 1u) / n), 1.f / (float)n};
}
// Whether k_experts_many is the quicker one over matrices of n rows of kp columns, by the experts' average (the device alone knows their counts).
// k_experts_tiled has four tiles of 64 x 64 to one of 256 columns, so that few rows still fill the chip, but twice the bytes a product on their way into LDS.
// Weights from memory, both products, us in tiles of 64 and in the best of the others: 8 experts 1024 wide in 2048, 50 rows each 40 and 52, 128 rows 55
// and 61, 200 rows 66 and 58; 32 of them, 40 rows 91 and 89, 64 rows 113 and 93; 8 experts 256 wide in 512, 97 rows 12 and 23, 600 rows 27 and 29; 64 experts
// 1408 wide in 2048, 33 rows 226 and 214, 64 rows 305 and 240; 128 experts 128 wide in 512, 50 rows 30 and 27.
static bool many_rows_pay(uint32_t experts, uint32_t identity, uint64_t entries, uint32_t kp, uint32_t n) {
  const float to = (float)std::min<uint64_t>(experts, entries), avg = (float)entries * (float)experts / (float)(experts + identity) / to;
  const Chip c = chip();
  const uint32_t steps = kp >> 6;
  const auto tiles = [&](float bm) { return avg > 0.7f * bm ? to * (avg / bm + 0.5f) : to; };      // (half of an expert's last one is empty)
  const float few = tiles(64.f) * (float)cdiv(n, 64) * c.inv;                // a CU's
  float many = 1e30f;
  for (uint32_t i = 0; i < MANY_SIZES; i++)
    many = std::min(many, many_us(i, (uint32_t)std::min(1.6e7f, tiles(128.f + 64.f * (float)i) * (float)cdiv(n, 256)), steps, c));
  return many < 3.f + 0.25f * (float)steps * std::max(1.f, few) + 2.f * few;
}

template <bool IN>
static void experts_product(Map* mo, Map* mw, const XSpec& s, float* parts, const uint32_t* list, const uint32_t* cnt, uint32_t rows) {
  const bf16_t* W = (const bf16_t*)mw->buf;
  const uint64_t entries = (uint64_t)rows * s.top;
  const uint32_t n = IN ? 2u * ((s.ff + 15u) & ~15u) : s.width;
  const auto grid = [&](uint32_t bm, uint32_t tiles_n) {       // no more tiles than this, whatever the rows choose
    return cdiv((entries / bm + std::min<uint64_t>(s.experts, entries)) * tiles_n, 8) * 8u;
  };
  if (mo->dtype == DTYPE_F32)
    k_experts_f32<IN><<<grid(64, cdiv(n, 64)), 256, 0, g.stream>>>(W, (float*)mo->buf, parts, s, list, cnt, rows, cdiv(n, 64));
  else if (many_rows_pay(s.experts, s.identity, entries, IN ? s.k_stride : s.ff_stride, n))
    k_experts_many<IN><<<grid(128, cdiv(n, 256)), 512, 0, g.stream>>>(W, (bf16_t*)mo->buf, parts, s, list, cnt, rows, cdiv(n, 256), chip());
  else
    k_experts_tiled<IN><<<grid(64, cdiv(n, 64)), 256, 0, g.stream>>>(W, (bf16_t*)mo->buf, parts, s, list, cnt, rows, cdiv(n, 64));
  count_launch();
}

}  // namespace adamah

using namespace adamah;

extern "C" int adamah_hip_experts_plan(const uint32_t* counts, uint32_t experts, uint32_t identity, uint64_t entries, uint32_t k, uint32_t n, uint32_t* tile, uint32_t* once) {
  if (g.n_cu <= 0 || !counts || experts == 0u || entries == 0u || k == 0u || (k & 63u) || n == 0u || !tile || !once) return ADAMAH_ERR_INVALID;
  *tile = 64u; *once = 0u;
  if (!many_rows_pay(experts, identity, entries, k, n)) return ADAMAH_OK;
  uint32_t t[MANY_SIZES] = {0, 0, 0}, some = 0;
  for (uint32_t e = 0; e < experts; e++) {
    for (uint32_t i = 0; i < MANY_SIZES; i++) t[i] += cdiv(counts[e], 128u + 64u * i);
    some += counts[e] ? 1u : 0u;
  }
  const Many m = many_pick(t, some, cdiv(n, 256), k >> 6, chip());
  *tile = 128u + 64u * m.size; *once = m.once ? 1u : 0u;
  return ADAMAH_OK;
}

extern "C" int adamah_experts_dev(uint32_t map_act, uint32_t map_opnd, uint32_t map_wt, uint32_t h_spec, uint32_t h_shared, uint32_t rows) { ADAMAH_API();
  Map *ma = get_f32_map(map_act), *mo = get_map(map_opnd), *mw = get_map(map_wt);
  const XSpec* s = spec_of<XSpec>(h_spec);
  if (!ma || !mw || mw->dtype != DTYPE_BF16 || !s || rows == 0) return ADAMAH_ERR_INVALID;
  const uint64_t E = s->experts, n = E + s->identity, F16 = (s->ff + 15u) / 16u * 16u, fs = s->ff_stride, wd = s->width;
  const uint64_t n_log = n + (s->shared_ff ? 1 : 0), entries = (uint64_t)rows * s->top;
  if (E == 0 || n > MAX_CHOICES || s->top == 0 || s->top > MAX_TOP || s->top > n || s->ff == 0 || fs < F16 || (fs & 63u) || wd == 0) return ADAMAH_ERR_INVALID;
  if (s->k_stride < wd || (s->k_stride & 63u) || s->k_stride > MAX_STEP || ((s->gate_up | s->gate_up_step | s->down | s->down_step) & 7u)) return ADAMAH_ERR_INVALID;
  if (s->gate_up_step < 2 * F16 * s->k_stride || s->down_step < wd * fs || entries > 0x7FFFFFFFull || s->epi > 1u) return ADAMAH_ERR_INVALID;
  const auto rows_ok = [&](uint64_t off, uint64_t stride, uint64_t width) { return in_range(off, (rows - 1) * stride + width, ma->n_elems); };
  if (!in_range(s->gate_up, (E - 1) * s->gate_up_step + 2 * F16 * s->k_stride, mw->n_elems) ||
      !in_range(s->down, (E - 1) * s->down_step + wd * fs, mw->n_elems)) return ADAMAH_ERR_INVALID;
  if (!rows_ok(s->logits, s->logits_stride, n_log) || !in_range(s->correction, n, ma->n_elems) || !rows_ok(s->x, s->x_stride, wd) ||
      !rows_ok(s->out, s->out_stride, wd)) return ADAMAH_ERR_INVALID;
  float* act = (float*)ma->buf;
  const bf16_t* W = (const bf16_t*)mw->buf;
  if (rows == 1) {
    const uint64_t most = std::min<uint64_t>(s->top, E), held = most * fs + (s->shared_ff ? s->shared_ff_stride : 0);
    if (held > MAX_STEP || !in_range(s->act, most * fs, ma->n_elems)) return ADAMAH_ERR_INVALID;
    if (s->shared_ff && (s->shared_ff_stride < s->shared_ff || (s->shared_ff_stride & 63u) || (s->shared_down & 7u) ||
                         !in_range(s->shared_down, wd * s->shared_ff_stride, mw->n_elems) || !in_range(s->shared_act, s->shared_ff, ma->n_elems))) return ADAMAH_ERR_INVALID;
    if (int r = scratch_need(g_experts, sizeof(Choice))) return r;
    Choice* choice = (Choice*)g_experts.p;
    const uint32_t cu2 = 2u * (uint32_t)g.n_cu, in_grid = std::min<uint32_t>(cdiv(most * F16, XSTEP / 64), cu2), in_lds = s->k_stride * 4u;
    const uint32_t out_grid = std::min<uint32_t>(cdiv(wd, XSTEP / 64), cu2), out_lds = (uint32_t)held * 4u;
    const uint32_t magic = (uint32_t)((0x100000000ull + fs - 1) / fs);       // i / fs = umulhi(i, magic) for i <= MAX_STEP
#define LDS_FOR(K, B) if ((B) > 48000) hipFuncSetAttribute((const void*)(K), hipFuncAttributeMaxDynamicSharedMemorySize, (int)(B))
    if (s->k_stride >= 1024u) { LDS_FOR(k_experts_in<4>, in_lds); k_experts_in<4><<<in_grid, XSTEP, in_lds, g.stream>>>(W, act, choice, *s); }
    else k_experts_in<1><<<in_grid, XSTEP, in_lds, g.stream>>>(W, act, choice, *s);
    count_launch();
    if (int r = check_launch()) return r;
    if (held >= 1024u) { LDS_FOR(k_experts_out<4>, out_lds); k_experts_out<4><<<out_grid, XSTEP, out_lds, g.stream>>>(W, act, choice, *s, magic); }
    else k_experts_out<1><<<out_grid, XSTEP, out_lds, g.stream>>>(W, act, choice, *s, magic);
#undef LDS_FOR
    count_launch();
    return check_launch();
  }
  if (!mo || (mo->dtype != DTYPE_BF16 && mo->dtype != DTYPE_F32) || ((s->opnd | s->act_opnd) & 7u)) return ADAMAH_ERR_INVALID;
  if (!in_range(s->opnd, (uint64_t)rows * s->k_stride, mo->n_elems) || !in_range(s->act_opnd, entries * fs, mo->n_elems)) return ADAMAH_ERR_INVALID;
  uint32_t shared = s->x, shared_stride = s->x_stride;
  if (s->shared_ff) {
    const AdamahLinearSpec* sh = spec_of<AdamahLinearSpec>(h_shared);
    if (!sh || sh->n != wd || sh->epi) return ADAMAH_ERR_INVALID;
    if (int r = adamah_linear_dev(map_act, map_opnd, map_wt, h_shared, 0, rows)) return r;      // (checks its own ranges)
    shared = sh->out; shared_stride = sh->out_stride;
  }
  // scratch: results per entry, choices, weights, the experts' lists and counts
  if (int r = scratch_need(g_experts, (entries * wd + 2 * entries + E * rows + E) * 4)) return r;
  float* parts = (float*)g_experts.p;
  uint32_t* ids = (uint32_t*)(parts + entries * wd);
  float* wts = (float*)(ids + entries);
  uint32_t *list = (uint32_t*)(wts + entries), *cnt = list + E * rows;
#define CHOOSE(NV) k_experts_choose<NV><<<cdiv(rows, 4), 256, 0, g.stream>>>(*s, act, ids, wts, rows)
  if (n <= 64) CHOOSE(1); else if (n <= 128) CHOOSE(2); else if (n <= 256) CHOOSE(4); else CHOOSE(16);
#undef CHOOSE
  count_launch();
  if (int r = check_launch()) return r;
#define LIST(W, K) k_experts_list<W, K><<<(uint32_t)E, 64 * W, 0, g.stream>>>(ids, list, cnt, rows, s->top)
  if (entries <= 1024u) LIST(4, 4); else if (entries <= 4096u) LIST(16, 4); else LIST(16, 16);
#undef LIST
  count_launch();
  if (int r = check_launch()) return r;
  experts_product<true>(mo, mw, *s, parts, list, cnt, rows);
  if (int r = check_launch()) return r;
  experts_product<false>(mo, mw, *s, parts, list, cnt, rows);
  if (int r = check_launch()) return r;
  k_experts_sum<<<rows, 256, 0, g.stream>>>(*s, act, parts, ids, wts, shared, shared_stride);
  count_launch();
  return check_launch();
}
