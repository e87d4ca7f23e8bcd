// Batched (M > 1) quantised matmul  C[M, N] = A[M, K] . W[N, K]^T  for Q4_0 weights on the fp16
// matrix cores: prefill chunks and batched decode.
//
// Reference: shaders/src/f32/map_matmul_t_xq4.comp:33-73 (one thread per output, scalar K loop;
// dispatch adamah.c:8693-8803).  With more than one activation row the weights are reused, so this
// is the one place on the path where the work is a dense contraction and belongs on MFMA.
//
// v_mfma_f32_16x16x32_f16:  D[i][j] += sum_k A[i][k] B[k][j];  lane l supplies A[l % 16][8g..8g+7] and
// B[8g..8g+7][l % 16] with g = l / 16, and receives D[4g..4g+3][l % 16].  Here i runs over 16 activation rows,
// j over 16 weight rows, and the 32 k of one instruction are ONE 32-weight block: lane (row, g) loads block g of
// the step's four blocks of its weight row as one 16-byte word group, a 4 x 4 transpose of words between the four
// lanes of a row (gfx950 row-swap instructions) leaves it with word g of every block, and the nibbles become
// fp16 (q - 8) exactly.  Each block's products are summed by the matrix core from zero and the block's fp16
// scale is applied to that sum in float32 (one fused multiply-add per output and block), so the weights need no
// rounding at all.  The activations of the tile are converted once per matmul to two fp16 planes (x s = xh + xl,
// s a power of two per row so that no row can overflow; divided out of the float32 result), in the element order
// the unpacking produces; two instructions per block (xh, xl), every product exact.
//
// Tiled form: workgroup = NW waves, each with R tiles of 16 weight rows = 16 NW R weight rows x 16 MT activation
// rows; one step = 128 weights of K (four blocks).
// Narrow form (more than 64 activation rows of fewer than 2048 columns): 32 activation rows x 128 weight rows a workgroup.
// Ring form (more than 64 activation rows): eight waves of 64 weight rows over 64, 96 or 128 activation rows, on 32x32x16
// instructions, weights, scales and activations straight to a ring of LDS stages.
// Either over shares of K, which k_gemm_splitk_sum adds up; gemm_plan says which.
// Few rows (2 .. 64): k_gemm_q4_rows, k_gemm_q4_f16_rows16.  The waves of a workgroup share R tiles of 16 weight rows and take
// every NWV-th step of K each, so that small matrices still spread over the whole chip; their partial tiles are summed
// through LDS in a fixed order.  At most 64 rows are converted to operand tiles (ActForm), more to rows.
#include "gemv_common.h"
#include "lds_ring.h"
#include "tile_store.h"
#include <algorithm>

namespace adamah {

typedef _Float16 h2q_t __attribute__((ext_vector_type(2)));
typedef _Float16 h4q_t __attribute__((ext_vector_type(4)));
typedef float f4q_t __attribute__((ext_vector_type(4)));
typedef float f4qu_t __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u2q_t __attribute__((ext_vector_type(2)));
typedef uint32_t u4q_t __attribute__((ext_vector_type(4)));
typedef _Float16 h8q_t __attribute__((ext_vector_type(8)));

// Two-term activations.  A product w * x of the reference is a float32 product of float32 values; one fp16
// rounding of an operand (2^-12 relative) is harmless in a single projection but adds up over the ~200
// projections of a forward pass (a 512-token chunk ended 1.3e-3 .. 6e-3 away from the token-by-token hidden
// state).  The activations are therefore fed as exact sums of two fp16 numbers,
//   x * s  = xh + xl          xh = fp16(x s), xl = fp16(x s - xh)                (22 significant bits),
// and the weights as the integers (q - 8) with the block scale applied afterwards in float32.  Q8_0 weights (the LM
// head of a lockstep batch, the last projection of a pass) keep one fp16 term for each operand.
__device__ __forceinline__ void split_pair(float a, float b, uint32_t* hi, uint32_t* lo) {
  const _Float16 ah = (_Float16)a, bh = (_Float16)b;
  const h2q_t h = {ah, bh}, l = {(_Float16)(a - (float)ah), (_Float16)(b - (float)bh)};
  *hi = __builtin_bit_cast(uint32_t, h);
  *lo = __builtin_bit_cast(uint32_t, l);
}
// eight consecutive activations (already scaled) -> the 16-byte pieces of both planes, pairs in the order the
// nibble unpacking produces: (0,4)(1,5)(2,6)(3,7)
__device__ __forceinline__ void split_word(const float* v, uint4* hi, uint4* lo) {
  split_pair(v[0], v[4], &hi->x, &lo->x);
  split_pair(v[1], v[5], &hi->y, &lo->y);
  split_pair(v[2], v[6], &hi->z, &lo->z);
  split_pair(v[3], v[7], &hi->w, &lo->w);
}

// The activations are converted once per matmul (or by the kernel that produced them) to the two fp16
// planes the matrix cores consume: rows scaled by their power of two, elements of every 8-word in the
// order (0,4)(1,5)(2,6)(3,7), in the places that `form` gives them (rows of both planes, or operand tiles).  One workgroup per
// row; also stores (s, 1/s).
__global__ void __launch_bounds__(256)
k_act_f16(const float* act, const uint32_t* __restrict__ la, uint32_t M, uint32_t K, float* scale, uint4* x, ActForm form) {
  __shared__ float red[4];
  const uint32_t row = blockIdx.x, op = blockIdx.y, tid = threadIdx.x;
  const float* src = act + (uint64_t)la[op] + (uint64_t)row * K;
  float m = 0.f;
  for (uint32_t i = tid; i < K; i += 256u) m = fmaxf(m, fabsf(src[i]));
  m = wave_max(m);
  if ((tid & 63u) == 0) red[tid >> 6] = m;
  __syncthreads();
  m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const uint32_t e = (__float_as_uint(m) >> 23) & 0xFFu;
  float s = 1.f, inv = 1.f;
  if (e >= 14u && e <= 254u) { s = __uint_as_float((267u - e) << 23); inv = __uint_as_float((e - 13u) << 23); }
  if (tid == 0) {
    scale[2 * ((uint64_t)op * M + row)] = s;
    scale[2 * ((uint64_t)op * M + row) + 1] = inv;
  }
  for (uint32_t w = tid; w < (K >> 3); w += 256u) {
    const f4qu_t v0 = *(const f4qu_t*)(src + w * 8u), v1 = *(const f4qu_t*)(src + w * 8u + 4u);
    const float v[8] = {v0.x * s, v0.y * s, v0.z * s, v0.w * s, v1.x * s, v1.y * s, v1.z * s, v1.w * s};
    uint4 hi, lo;
    split_word(v, &hi, &lo);
    x[act_piece(form, op, row, w, 0u)] = hi;
    x[act_piece(form, op, row, w, 1u)] = lo;
  }
}

// nibbles of one 32-bit word -> the four fp16 pairs (q - 8) exactly: (1024 + n) - 1032 and (64 + n) - 72
struct DeqK { uint32_t magic_lo, magic_hi, nib_lo, nib_hi; h2q_t off_lo, off_hi; };
__device__ __forceinline__ void deq_ints(uint32_t w, const DeqK& c, h2q_t* t) {
  const uint32_t w8 = w >> 8;
  t[0] = __builtin_bit_cast(h2q_t, (w & c.nib_lo) | c.magic_lo) + c.off_lo;
  t[1] = __builtin_bit_cast(h2q_t, (w & c.nib_hi) | c.magic_hi) + c.off_hi;
  t[2] = __builtin_bit_cast(h2q_t, (w8 & c.nib_lo) | c.magic_lo) + c.off_lo;
  t[3] = __builtin_bit_cast(h2q_t, (w8 & c.nib_hi) | c.magic_hi) + c.off_hi;
}
// one word of a block -> the operand fragment (q - 8), exact in fp16, eight weights in the order deq_ints makes
__device__ __forceinline__ u4q_t deq_word(uint32_t w, const DeqK& c) {
  h2q_t t[4];
  deq_ints(w, c, t);
  return (u4q_t){__builtin_bit_cast(uint32_t, t[0]), __builtin_bit_cast(uint32_t, t[1]), __builtin_bit_cast(uint32_t, t[2]),
                 __builtin_bit_cast(uint32_t, t[3])};
}
// Lanes l, l + 16, l + 32, l + 48 hold the four 32-weight blocks of one step of a weight row, four words each.
// One matrix instruction is to cover ONE block (so that the block's scale can be applied to its result), i.e.
// lane group g has to supply word g of that block: a 4 x 4 transpose of words between the four lanes, done with
// the row-swap instructions of gfx950 (v_permlane32_swap: upper half of the first register <-> lower half of the
// second; v_permlane16_swap: odd 16-lane rows of the first <-> even rows of the second).  Afterwards word b of
// the result is word g of block b.
typedef uint32_t u2s_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u4q_t transpose_blocks(u4q_t q) {
  const u2s_t a = __builtin_amdgcn_permlane32_swap(q.x, q.z, false, false);
  const u2s_t b = __builtin_amdgcn_permlane32_swap(q.y, q.w, false, false);
  const u2s_t c = __builtin_amdgcn_permlane16_swap(a.x, b.x, false, false);
  const u2s_t d = __builtin_amdgcn_permlane16_swap(a.y, b.y, false, false);
  return (u4q_t){c.x, c.y, d.x, d.y};
}
// the scales of the four blocks (lane group g holds block g's): all four to every lane, as float
__device__ __forceinline__ f4q_t gather_scales(_Float16 d) {
  const uint32_t v = (uint32_t)__builtin_bit_cast(uint16_t, d);
  const u2s_t a = __builtin_amdgcn_permlane32_swap(v, v, false, false);        // {d0 d1 d0 d1}, {d2 d3 d2 d3} by lane group
  const u2s_t lo = __builtin_amdgcn_permlane16_swap(a.x, a.x, false, false);   // {d0 d0 d0 d0}, {d1 d1 d1 d1}
  const u2s_t hi = __builtin_amdgcn_permlane16_swap(a.y, a.y, false, false);   // {d2 ...}, {d3 ...}
  auto f = [](uint32_t b) { return (float)__builtin_bit_cast(_Float16, (uint16_t)b); };
  return (f4q_t){f(lo.x), f(lo.y), f(hi.x), f(hi.y)};
}
// the same as four halves
__device__ __forceinline__ h4q_t gather_scales16(uint32_t d) {
  const u2s_t a = __builtin_amdgcn_permlane32_swap(d, d, false, false);
  const u2s_t lo = __builtin_amdgcn_permlane16_swap(a.x, a.x, false, false), hi = __builtin_amdgcn_permlane16_swap(a.y, a.y, false, false);
  return __builtin_bit_cast(h4q_t, (u2q_t){lo.x | lo.y << 16, hi.x | hi.y << 16});
}
#define DEQK_INIT(c)                                                                           \
  DeqK c = {0x64006400u, 0x54005400u, 0x000F000Fu, 0x00F000F0u,                                \
            {(_Float16)-1032.f, (_Float16)-1032.f}, {(_Float16)-72.f, (_Float16)-72.f}};       \
  asm volatile("" : "+v"(c.magic_lo)); /* opaque: lets instruction selection use the three-operand and-or */ \
  asm volatile("" : "+v"(c.magic_hi));                                                         \
  asm volatile("" : "+s"(c.nib_lo));                                                           \
  asm volatile("" : "+s"(c.nib_hi))
#define MFMA_F16(a, b, c) __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8q_t, a), __builtin_bit_cast(h8q_t, b), c, 0, 0, 0)

// Workgroup = NW waves, each with R tiles of 16 weight rows = 16 NW R weight rows x 16 MT activation rows.
// A pair of activation fragments (both planes) read from LDS feeds 2 R matrix instructions; the weights of a
// wave's R tiles are unpacked in its registers, block by block as the K loop needs them.  One step = 128 weights
// of K; the next step's weight words and activation pieces are loaded into registers while the matrix cores work
// on the current one.  The activation tile is staged by every workgroup, so wide workgroups (eight waves) move
// fewer bytes per flop: 28672x4096 at M = 512 went 434 -> 344 us with 256 instead of 128 weight rows per workgroup.
// TILES: the activations come as operand tiles (at most 64 rows), else as rows.
template <int MT, int R, int NW, bool TILES>
__global__ void __launch_bounds__(64 * NW)
k_gemm_q4_f16_tiled(const uint8_t* __restrict__ W, const __half* __restrict__ d16, const u4q_t* __restrict__ x, ActForm form, uint32_t K, uint32_t N, uint32_t M, uint32_t b_val, uint32_t c_val, uint32_t by_val, float* out,
                     const uint32_t* __restrict__ lb, const uint32_t* __restrict__ lc, const float* __restrict__ scale,
                     GemmSegs segs, uint32_t ksplit, uint32_t kper, float* __restrict__ part) {
  // (the first 14 dwords of the arguments are in registers when a wave starts; by_val bit 0 / 1: the weights' / the
  // result's element offset of op 0 is b_val / c_val -- known on the host -- instead of a load from lb / lc, which
  // the first weight loads would have to wait for)
  // ksplit > 1 (one op): blockIdx.z is a share of K -- kper blocks, a multiple of 4 -- and the tile's raw sums go to
  // part[share][row][n] for k_gemm_splitk_sum; wide tiles then still give every CU a workgroup on a narrow matrix.
  constexpr uint32_t BM = 16u * MT, ROWB = 272u;
  __shared__ __attribute__((aligned(16))) uint8_t xs[2u * BM * ROWB];   // first plane, then second plane
  uint8_t* const xs2 = xs + BM * ROWB;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t r16 = lane & 15u, g = lane >> 4;
  constexpr uint32_t NT = 64u * NW, NP = 256u * MT / NT;       // threads; 16-byte pieces per thread, plane and step
  const uint32_t n0 = blockIdx.x * (16u * NW * R) + wave * (16u * R), m0 = blockIdx.y * BM;
  const uint32_t op = ksplit > 1u ? 0u : blockIdx.z, kz = ksplit > 1u ? blockIdx.z : 0u;
  const uint64_t c_off = (by_val & 2u) ? (uint64_t)c_val : (uint64_t)lc[op], gbase = ((by_val & 1u) ? (uint64_t)b_val : (uint64_t)lb[op]) >> 5;
  const uint32_t nblk = K >> 5;                                // blocks per row
  const uint32_t kb_lo = kz * kper, kb_hi = min(nblk, kb_lo + kper);   // this workgroup's blocks of K
  uint32_t nrow[R];
#pragma unroll
  for (int r = 0; r < R; r++) nrow[r] = min(n0 + r * 16u + r16, N - 1u);   // rows past N: clamped, not stored

  f4q_t acc[R][MT];
#pragma unroll
  for (int r = 0; r < R; r++)
#pragma unroll
    for (int t = 0; t < MT; t++) acc[r][t] = (f4q_t){0.f, 0.f, 0.f, 0.f};
  DEQK_INIT(dk);

  // staging: the tile's 16 pieces per row, plane and step; thread -> (row, piece) pairs, NP per thread, in the order they lie in
  // (of operand tiles a row's neighbouring pieces are a request to the L1 each: 64 x 28672 x 4096 68.3 us by rows, 66.2 so)
  const auto srow = [](uint32_t w) { return TILES ? (w >> 8) * 16u + (w & 15u) : w >> 4; };
  const auto spiece = [](uint32_t w) { return TILES ? (w >> 4) & 15u : w & 15u; };
  uint64_t xoff[NP], xloff[TILES ? NP : 1];
  constexpr uint32_t per_blk = TILES ? 64u : 4u;             // pieces from a block of a row to the next one
  const u4q_t* const xl = x + form.lo;
#pragma unroll
  for (uint32_t u = 0; u < NP; u++) {
    const uint32_t w = tid + u * NT, row = min(m0 + srow(w), M - 1u);   // rows past M: clamped, not stored
    xoff[u] = TILES ? act_piece(form, op, row, spiece(w), 0u) : ((uint64_t)op * M + row) * form.kw + spiece(w);
    if (TILES) xloff[u] = act_piece(form, op, row, spiece(w), 1u);
  }
  u4q_t xn[NP], xln[NP], qn[R];
  _Float16 dn[R];
  // always executed; the step past K re-reads the last one and is not used
#define GEMM_FETCH(kb_raw)                                                        \
  do {                                                                            \
    const uint32_t kb_ = min((kb_raw), kb_hi - 4u);                               \
    _Pragma("unroll") for (int r = 0; r < R; r++) {                               \
      const uint64_t gi = gbase + (uint64_t)nrow[r] * nblk + kb_ + g;             \
      qn[r] = *(const u4q_t*)(W + (gi << 4));                                     \
      dn[r] = __builtin_bit_cast(_Float16, d16[gi]);                              \
    }                                                                             \
    _Pragma("unroll") for (uint32_t u = 0; u < NP; u++) {                         \
      xn[u] = x[xoff[u] + kb_ * per_blk];                                            \
      xln[u] = TILES ? x[xloff[u] + kb_ * per_blk] : xl[xoff[u] + kb_ * per_blk];                                            \
    }                                                                             \
  } while (0)
  GEMM_FETCH(kb_lo);

  for (uint32_t kb0 = kb_lo; kb0 < kb_hi; kb0 += 4u) {
#pragma unroll
    for (uint32_t u = 0; u < NP; u++) {
      const uint32_t w = tid + u * NT;
      *(u4q_t*)(xs + srow(w) * ROWB + spiece(w) * 16u) = xn[u];
      *(u4q_t*)(xs2 + srow(w) * ROWB + spiece(w) * 16u) = xln[u];
    }
    u4q_t q[R];
    f4q_t ds[R];
#pragma unroll
    for (int r = 0; r < R; r++) { q[r] = transpose_blocks(qn[r]); ds[r] = gather_scales(dn[r]); }
    __syncthreads();
    GEMM_FETCH(kb0 + 4u);
#pragma unroll
    for (int b = 0; b < 4; b++) {      // one 32-weight block of the step at a time
      u4q_t wq[R];
#pragma unroll
      for (int r = 0; r < R; r++) wq[r] = deq_word(b == 0 ? q[r].x : b == 1 ? q[r].y : b == 2 ? q[r].z : q[r].w, dk);
      // TG activation tiles at a time: their first-plane instructions, then the second-plane ones (each depends on
      // one issued TG * R instructions earlier), then the scaling of the block results
      constexpr int TG = R >= 4 ? 2 : MT >= 4 ? 4 : MT;
#pragma unroll
      for (int t0 = 0; t0 < MT; t0 += TG) {
        u4q_t ah[TG], al[TG];
        f4q_t blk[TG][R];
#pragma unroll
        for (int t = 0; t < TG; t++) {
          const uint32_t xo = ((t0 + t) * 16u + r16) * ROWB + b * 64u + g * 16u;
          ah[t] = *(const u4q_t*)(xs + xo); al[t] = *(const u4q_t*)(xs2 + xo);
        }
#pragma unroll
        for (int t = 0; t < TG; t++)
#pragma unroll
          for (int r = 0; r < R; r++) blk[t][r] = MFMA_F16(ah[t], wq[r], ((f4q_t){0.f, 0.f, 0.f, 0.f}));
#pragma unroll
        for (int t = 0; t < TG; t++)
#pragma unroll
          for (int r = 0; r < R; r++) blk[t][r] = MFMA_F16(al[t], wq[r], blk[t][r]);
#pragma unroll
        for (int t = 0; t < TG; t++)
#pragma unroll
          for (int r = 0; r < R; r++) {
            const float d = ds[r][b];
#pragma unroll
            for (int i = 0; i < 4; i++) acc[r][t0 + t][i] = fmaf(blk[t][r][i], d, acc[r][t0 + t][i]);
          }
      }
    }
    __syncthreads();
  }
  // lane (r16, g) holds D[4g + i][r16]: activation rows m0 + 16 t + 4g + i, weight row n0 + 16 r + r16
  const auto row = [&](int t, int i) { return m0 + t * 16u + 4u * g + i; };
  if (ksplit <= 1u) {      // (raw sums of a share of K: scale and placement are k_gemm_splitk_sum's)
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float inv = scale[2 * ((uint64_t)op * M + min(row(t, i), M - 1u)) + 1];
#pragma unroll
        for (int r = 0; r < R; r++) acc[r][t][i] *= inv;
      }
  }
  uint32_t n[R];
#pragma unroll
  for (int r = 0; r < R; r++) n[r] = n0 + r * 16u + r16;
  store_columns<MT, 4, R, false>([&](int t, int i, int r) { return acc[r][t][i]; }, row, n, M, N, kz, c_off, out, ksplit > 1u ? part : nullptr, segs);
}
#undef GEMM_FETCH

// The shares of K of a split launch of the kernel above, summed in the order of the shares, scaled by the row's factor
// and stored where the unsplit launch would have stored them (one op).  Four results per thread.
// Bound by memory: every share's four and the row to be added to are asked for at once (Z: the number of shares, 0: any), results go out
// 16 bytes a lane.  One share behind the other and four bytes a lane: five shares of 512 x 6144 18.0 us, so 12.8; 1877 tokens through the
// Llama 8B shape 79.8 -> 78.3 ms.
template <int Z>
__global__ void __launch_bounds__(256)
k_gemm_splitk_sum(const float* __restrict__ part, uint32_t ksplit, uint32_t M, uint32_t N, float* out, uint32_t c_val,
                  uint32_t by_val, const uint32_t* __restrict__ lc, const float* __restrict__ scale, GemmSegs segs) {
  const uint64_t total = (uint64_t)M * N, i0 = ((uint64_t)blockIdx.x * 256u + threadIdx.x) * 4u;
  if (i0 >= total) return;
  const uint64_t c_off = (by_val & 2u) ? (uint64_t)c_val : (uint64_t)lc[0];
  float v[4];
  if ((N & 3u) == 0u) {                   // the four are one row's
    f4q_t a[Z ? Z : 1];
#pragma unroll
    for (int z = 0; z < (Z ? Z : 1); z++) a[z] = *(const f4q_t*)(part + z * total + i0);
    const uint32_t row = total >> 32 ? (uint32_t)(i0 / N) : (uint32_t)i0 / N, n = (uint32_t)(i0 - (uint64_t)row * N);
    const uint64_t c = c_off + i0, r = segs.res + i0, d = segs.dst + i0;
    // (a result that is also what is added must be stored first)
    const bool lines = !segs.count && ((c_off | (segs.add ? segs.res | segs.dst : 0u)) & 3u) == 0u && !(segs.add && segs.res < c_off + total && c_off < segs.res + total);
    f4q_t old = {0.f, 0.f, 0.f, 0.f};
    if (lines && segs.add) old = *(const f4q_t*)(out + r);
    const float inv = scale[2 * (uint64_t)row + 1];
#pragma unroll
    for (int z = 1; z < Z; z++) a[0] += a[z];
    if (!Z)
      for (uint32_t z = 1; z < ksplit; z += 8u) {
        f4q_t b[8];
#pragma unroll
        for (uint32_t j = 0; j < 8; j++) b[j] = *(const f4q_t*)(part + min(z + j, ksplit - 1u) * total + i0);
#pragma unroll
        for (uint32_t j = 0; j < 8; j++) if (z + j < ksplit) a[0] += b[j];
      }
    if (lines) {
      const f4q_t y = {a[0][0] * inv, a[0][1] * inv, a[0][2] * inv, a[0][3] * inv};
      *(f4q_t*)(out + c) = y;
      if (segs.add) *(f4q_t*)(out + d) = old + y;
      return;
    }
    if (segs.count) {
      const ColumnPlace p = column_place(n, N, 0u, out, segs), p3 = column_place(n + 3u, N, 0u, out, segs);
      float* const to = p.col + (uint64_t)row * p.step;
      if (p3.col == p.col + 3 && p3.step == p.step && ((to - out) & 3) == 0) { *(f4q_t*)to = (f4q_t){a[0][0] * inv, a[0][1] * inv, a[0][2] * inv, a[0][3] * inv}; return; }
    }
    v[0] = a[0][0]; v[1] = a[0][1]; v[2] = a[0][2]; v[3] = a[0][3];
  } else {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      float a = i0 + e < total ? part[i0 + e] : 0.f;
      for (uint32_t z = 1; z < ksplit; z++) a += i0 + e < total ? part[z * total + i0 + e] : 0.f;
      v[e] = a;
    }
  }
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const uint64_t i = i0 + e;
    if (i >= total) break;
    const uint32_t row = (uint32_t)(i / N), n = (uint32_t)(i % N);
    const float y = v[e] * scale[2 * (uint64_t)row + 1];
    const ColumnPlace p = column_place(n, N, c_off, out, segs);
    p.col[(uint64_t)row * p.step] = y;
    if (!segs.count && segs.add) out[segs.dst + (uint64_t)row * N + n] = out[segs.res + (uint64_t)row * N + n] + y;   // the add behind it
  }
}

// ---- more than 64 activation rows ------------------------------------------------------------------------------------
// Eight waves of 64 weight rows each, side by side, over 32 MA activation rows: a wave has 2 x MA results of 32 x 32.  A step
// is 64 columns (two blocks); its packed weights (16 KB), their scales (2 KB) and both planes of the activations (8 KB per 32
// rows) go straight to LDS, a ring of four stages (MA = 2) or three (MA = 3, 4).  512 x 28672 x 4096: 317 -> 248 us = 485
// TFLOP/s.  96 rows a workgroup put 224 of the 256 CUs to work where 128 put 168 (384 x 28672 x 4096: 216 us and 197, not in
// proportion: with more CUs at work the clock falls, the products' power: 2.56 GHz with 32 workgroups, 2.0 with 224, 1.86 with 256,
// launches one by one).  What bounds it is the vector work beside the matrix instructions (a multiply-add per result and block, the
// unpacking): they share a wave's issue, so what counts is that no instruction of either kind waits for another.  LDS reads without bank conflicts: 266 -> 246 us.
// v_mfma_f32_32x32x16_f16: lane l supplies row l % 32, k = 8 (l / 32) .. + 7 of either operand and receives rows
// 8 (r / 4) + 4 (l / 32) + r % 4 of column l % 32 -- here the columns are weight rows, so a block's scale is one number per
// lane.  S16 (rows of whole runs of 256 columns that begin on 16 bytes of scales): the scales of four steps come in one 16-byte piece a row.
// A step's own four bytes of every row each took a line from the L2, 40 % of the requests (7.6 of 18.9 million for 512 x 28672 x 4096; now
// a quarter of that).  4096 x 14336 under 341 rows 116 -> 110 us, 4096 x 4096 under 512 56.5 -> 55; 1877 tokens through the Llama 8B
// shape 79.9 -> 79.2 ms.
// An instruction covers half a block; two permutes bring a block's words to the half of the wave that owns them.
typedef float f16q_t __attribute__((ext_vector_type(16)));
#define RING_W 16384u
#define RING_S 2048u
#define RING_S16 8192u
#define MFMA32_F16(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8q_t, a), __builtin_bit_cast(h8q_t, b), c, 0, 0, 0)

template <int MA, bool S16>
__global__ void __launch_bounds__(512)
k_gemm_q4_ring(const uint8_t* __restrict__ W, const __half* __restrict__ d16, const u4q_t* __restrict__ xh, const u4q_t* __restrict__ xl,
               uint32_t K, uint32_t N, uint32_t M, uint32_t gbase, uint32_t c_val, uint32_t by_val, uint32_t pairs_per, float* out,
               float* __restrict__ part, const uint32_t* __restrict__ lc, const float* __restrict__ scale, GemmSegs segs) {
  constexpr uint32_t BM = 32u * MA, BN = 512u, XOFF = RING_W + (S16 ? 0u : RING_S), RING_STAGE = XOFF + MA * 8192u;
  constexpr int SL = S16 ? 2 : 3, LOADS = SL + MA, RING_ST = MA == 2 ? 4 : 3;      // loads of a wave and stage: 2 of weights, 1 of scales (S16: its own), MA of activations
  static_assert(MA >= 2 && MA <= 4, "stages and schedule");
  __shared__ __attribute__((aligned(16))) uint8_t ring[RING_ST * RING_STAGE + (S16 ? 2u * RING_S16 : 0u)];
  constexpr uint32_t SOFF = RING_ST * RING_STAGE;            // S16: scales of four steps, two buffers
  const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t r32 = lane & 31u, h = lane >> 5;
  // Workgroups land on the eight dies in turn.  by_val & 4: a die takes a run of tiles, those of one run of weight rows next to each
  // other, so that its L2 has the weights once (256 x 32000 x 2048, 63 runs of weight rows: 106 us as they come, so: 84).
  uint32_t tn = blockIdx.x, tm = blockIdx.y;
  if (by_val & 4u) {
    const uint32_t rows = (M + BM - 1u) / BM, total = (N + BN - 1u) / BN * rows, id = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (id >= total) return;
    tn = id / rows; tm = id % rows;
  }
  const uint32_t n0 = tn * BN, m0 = tm * BM, kz = blockIdx.z;
  const uint32_t nblk = K >> 5, pairs = K >> 6, p_lo = kz * pairs_per, p_hi = min(pairs, p_lo + pairs_per);
  const uint32_t steps = p_hi - p_lo;

  // piece j of an activation row lies at j ^ slot(row): no two rows that are read together meet in a bank
  const auto slot = [](uint32_t row) { return (row & 7u) ^ ((row >> 4) & 1u); };
  // a load is a base for the wave and an offset for the lane
  uint32_t wo[2], so, xo[MA];
#pragma unroll
  for (uint32_t u = 0; u < 2; u++)                           // 32 rows of 32 bytes an instruction; LDS: [row][32]
    wo[u] = (min(n0 + (wave * 2u + u) * 32u + (lane >> 1), N - 1u) * nblk + (lane & 1u)) << 4;
  so = min(n0 + wave * 64u + lane, N - 1u) * nblk * 2u;      // 64 rows of 4 bytes; LDS: [row][4]
#pragma unroll
  for (uint32_t u = 0; u < MA; u++) {                        // 8 rows of 128 bytes; LDS: [plane][row][8 pieces, swizzled]
    const uint32_t row = ((wave * MA + u) * 8u) % BM + (lane >> 3);
    xo[u] = (min(m0 + row, M - 1u) * (K >> 3) + ((lane & 7u) ^ slot(row))) << 4;
  }
  const uint32_t base = lds_byte(ring);
  // load i of this wave for step s of this share; steps past its end re-read its last one (the count in flight stays)
  const auto load = [&](int i, uint32_t s, uint32_t into) {
    const uint32_t at = base + into * RING_STAGE;
    const uint64_t pair = min(p_lo + s, p_hi - 1u);
    if (i < 2) load_to_lds(W + (((uint64_t)gbase + pair * 2u) << 4), wo[i], at + (wave * 2u + i) * 1024u);
    else if (!S16 && i == 2) load4_to_lds(d16 + gbase + pair * 2u, so, at + RING_W + wave * 256u);
    else {
      const uint32_t j = wave * MA + (i - SL);
      load_to_lds((j >= 4u * MA ? xl : xh) + pair * 8u, xo[i - SL], at + XOFF + j * 1024u);
    }
  };

  // S16: the scales of the four steps that step s is the first of (64 rows of 16 bytes; LDS: [row][16])
  // (skipped inside the asm: a branch of the compiler's would part the loop's one block)
  const auto load_scales = [&](uint32_t s, bool skip) {
    const uint32_t run = (p_lo + s) >> 2;
    load_to_lds_unless(skip, d16 + gbase + run * 8u, so, base + SOFF + (run & 1u) * RING_S16 + wave * 1024u);
  };

  f16q_t acc[2][MA], blk[2], zero;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    zero[i] = 0.f; blk[1][i] = 0.f;
#pragma unroll
    for (int w = 0; w < 2; w++)
#pragma unroll
      for (int t = 0; t < MA; t++) acc[w][t][i] = 0.f;
  }
  DEQK_INIT(dk);
  u4q_t q[2], raw[2], wf[2][2][2], fr[2][2];              // wf [block][tile][half], fr [plane][half]
  h2q_t ds[2];
  float d[2][2], dn[2][2], dlast = 0.f;                      // [tile][block]
  const uint32_t wrow = (wave * 64u + r32) * 32u + h * 16u, srow = RING_W + (wave * 64u + r32) * 4u;
  const uint32_t xrow = XOFF + r32 * 128u;
  const auto read_w = [&](const uint8_t* st, int w, uint32_t s) {      // step s
    raw[w] = *(const u4q_t*)(st + wrow + w * 1024u);
    const uint32_t at = p_lo + s;
    if (S16) ds[w] = *(const h2q_t*)(ring + SOFF + (at >> 2 & 1u) * RING_S16 + (wave * 64u + r32) * 16u + w * 512u + (at & 3u) * 4u);
    else ds[w] = *(const h2q_t*)(st + srow + w * 128u);
  };
  const auto take_w = [&](int w) {
    const u2s_t a = __builtin_amdgcn_permlane32_swap(raw[w].x, raw[w].y, false, false), b = __builtin_amdgcn_permlane32_swap(raw[w].z, raw[w].w, false, false);
    q[w] = (u4q_t){a.x, b.x, a.y, b.y};                      // block 0's halves, block 1's halves
    dn[w][0] = (float)ds[w].x; dn[w][1] = (float)ds[w].y;
    asm volatile("" : "+v"(dn[w][0]), "+v"(dn[w][1]));      // (as floats: else every multiply-add widens its own)
  };
  const auto unpack = [&](int b, int w, int e) { wf[b][w][e] = deq_word(b ? (e ? q[w].w : q[w].z) : (e ? q[w].y : q[w].x), dk); };
  const auto read_x = [&](const uint8_t* st, int b, int t, int plane, int e) {
    fr[plane][e] = *(const u4q_t*)(st + xrow + plane * (MA * 4096u) + t * 4096u + (((4u * b + 2u * e + h) ^ slot(r32)) << 4));
  };
#pragma unroll
  for (int s = 0; s < RING_ST - 1; s++) {
    if (S16) load_scales(s, (s != 0 && ((p_lo + s) & 3u) != 0u) || (uint32_t)s >= steps);
#pragma unroll
    for (int i = 0; i < LOADS; i++) load(i, s, s);
  }
  ring_wait<LOADS * (RING_ST - 2)>();
#pragma unroll
  for (int w = 0; w < 2; w++) {
    read_w(ring, w, 0u);
    take_w(w);
    unpack(0, w, 0); unpack(0, w, 1);
    d[w][0] = dn[w][0]; d[w][1] = dn[w][1];
  }
#pragma unroll
  for (int i = 0; i < 4; i++) read_x(ring, 0, 0, i >> 1, i & 1);
  uint32_t buf = 0, next = 1, into = RING_ST - 1;
  for (uint32_t s = 0; s < steps; s++) {
    const uint8_t *st = ring + buf * RING_STAGE, *sn = ring + next * RING_STAGE;
    constexpr int NT = 2 * MA;                               // tiles of a block
#pragma unroll
    for (int b = 0; b < 2; b++) {
      if (b) ring_wait<LOADS * (RING_ST - 3)>();             // the next stage is here, the one before is no longer read
#pragma unroll
      for (int x = 0; x < NT; x++) {
        const int t = x >> 1, w = x & 1;
        // four instructions of this tile (32 clocks of the matrix pipe each) and between them the scaling of the last
        // tile's result, which is there once two of them have gone out (behind the first it held up the second: 266 us
        // for 512 x 28672 x 4096), and what the next tiles, block and stages need
#pragma unroll
        for (int m = 0; m < 4; m++) {
          blk[w] = MFMA32_F16(fr[m >> 1][m & 1], wf[b][w][m & 1], m ? blk[w] : zero);
          const int pw = 1 - w, pt = w ? t : (x ? t - 1 : MA - 1);
          const float ps = w ? d[0][b] : (x ? d[1][b] : (b ? d[1][0] : dlast));
#pragma unroll
          for (int i = m ? 5 * m - 5 : 0; i < (m == 3 ? 16 : 5 * m); i++) acc[pw][pt][i] = fmaf(blk[pw][i], ps, acc[pw][pt][i]);
          if (w == 1) {                                      // its last use: the same operand of the next 32 rows
            if (t + 1 < MA) read_x(st, b, t + 1, m >> 1, m & 1);
            else if (b == 0) read_x(st, 1, 0, m >> 1, m & 1);
            else read_x(sn, 0, 0, m >> 1, m & 1);
          }
          if (b == 1 && x == 0 && m < 2) read_w(sn, m, s + 1u);
          if (S16 && b == 1 && x == 1 && m == 0) load_scales(s + RING_ST - 1u, ((p_lo + s + RING_ST - 1u) & 3u) != 0u || s + RING_ST - 1u >= steps);
          if (b == 1 && x == 1 && m >= 2) take_w(m - 2);
          if (b == 0 && m == 0) for (int u = x * 4 / NT; u < (x + 1) * 4 / NT; u++) unpack(1, u >> 1, u & 1);
          if (b == 1 && x >= 2 && m == 0) for (int u = (x - 2) * 4 / (NT - 2); u < (x - 1) * 4 / (NT - 2); u++) unpack(0, u >> 1, u & 1);
          if (b == 1) for (int u = (4 * x + m) * LOADS / (4 * NT); u < (4 * x + m + 1) * LOADS / (4 * NT); u++) load(u, s + RING_ST - 1u, into);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    dlast = d[1][1];
#pragma unroll
    for (int w = 0; w < 2; w++) { d[w][0] = dn[w][0]; d[w][1] = dn[w][1]; }
    into = buf; buf = next; next = next + 1u == RING_ST ? 0u : next + 1u;
  }
#pragma unroll
  for (int i = 0; i < 16; i++) acc[1][MA - 1][i] = fmaf(blk[1][i], dlast, acc[1][MA - 1][i]);
  ring_wait<0>();
  const uint64_t c_off = (by_val & 2u) || part || segs.count ? (uint64_t)c_val : (uint64_t)lc[0];
  const auto row = [&](int t, int i) { return m0 + t * 32u + 8u * (i >> 2) + 4u * h + (i & 3u); };
  if (!part) {
#pragma unroll
    for (int t = 0; t < MA; t++)
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const float inv = scale[2 * (uint64_t)min(row(t, i), M - 1u) + 1];
        acc[0][t][i] *= inv; acc[1][t][i] *= inv;
      }
  }
  const uint32_t n[2] = {n0 + wave * 64u + r32, n0 + wave * 64u + 32u + r32};
  store_columns<MA, 16, 2>([&](int t, int i, int w) { return acc[w][t][i]; }, row, n, M, N, kz, c_off, out, part, segs);
}

// More than 64 activation rows and few columns, or few weight rows: tiles of 32 activation rows by 128 weight rows, so that a narrow matrix
// still gives most CUs a workgroup.  A wave has 32 x 64 results of every fourth block: two waves side by side, four sharing out
// the four blocks of a step of 128 columns, whose sums meet in LDS in the order of the blocks' places.  A workgroup's step (16 KB of both planes
// of the activations, 8 of weights, 1 of scales) goes straight to LDS, a ring of three stages (four to six: 0.1 to 0.7 us slower); a wave reads the next
// step's operands, and adds up the products of the one before, under the products of this one (added up behind its own: a fifth slower over long rows).
// What bounds it: a step takes 0.44 us with a few workgroups, 0.65 with one on every CU, of which the products need 0.21; the rest is the
// vector work beside them (unpacking for 32 rows only, a multiply-add per result and block) and, with many workgroups, the activations' way out of the L2s.
// The tiled kernel, whose step of 128 columns waits for its loads (1.3 us), and so: 512 x 1536 x 1152 16.2 and 10.9 us, 189 x 1536 x 1152 15.1 and 9.8, 189 x 1152
// x 1024 13.8 and 9.4, 70 x 13824 x 1152 22.3 and 18.9.
// LDS: piece j of an activation row at j ^ (row & 15), block j of a weight row at j ^ (row / 4 & 3): no two rows that are read together meet in a bank.
#define NARROW_X 16384u
#define NARROW_W 8192u
#define NARROW_STAGE (NARROW_X + NARROW_W + 1024u)
__global__ void __launch_bounds__(512)
k_gemm_q4_narrow(const uint8_t* __restrict__ W, const __half* __restrict__ d16, const u4q_t* __restrict__ xh, const u4q_t* __restrict__ xl,
                 uint32_t K, uint32_t N, uint32_t M, uint32_t gbase, uint32_t c_val, uint32_t by_val, float* out, const uint32_t* __restrict__ lc,
                 const float* __restrict__ scale, GemmSegs segs) {
  constexpr int LOADS = 4;                                   // of a wave and stage: 2 of activations, 1 of weights, 1 of scales (which two waves ask for)
  constexpr uint32_t ST = 3;
  static_assert(ST * NARROW_STAGE >= 65536u, "the sums' way over LDS");
  __shared__ __attribute__((aligned(16))) uint8_t ring[ST * NARROW_STAGE];
  const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t r32 = lane & 31u, h = lane >> 5, side = wave & 1u, kb = wave >> 1;
  // workgroups land on the eight dies in turn: a die takes a run of tiles, those of the same activation rows next to each other
  const uint32_t tiles_n = (N + 127u) / 128u, id = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const uint32_t n0 = id % tiles_n * 128u, m0 = id / tiles_n * 32u;
  if (m0 >= M) return;
  const uint32_t nblk = K >> 5, steps = K >> 7;
  const uint32_t base = lds_byte(ring);

  // a load is a base for the wave and an offset for the lane
  uint32_t xo[2];
#pragma unroll
  for (uint32_t u = 0; u < 2; u++) {                         // 4 rows of 256 bytes an instruction; LDS: [plane][row][16 pieces]
    const uint32_t row = ((wave * 2u + u) & 7u) * 4u + (lane >> 4);
    xo[u] = (min(m0 + row, M - 1u) * (K >> 3) + ((lane & 15u) ^ (row & 15u))) << 4;
  }
  const uint32_t wr = wave * 16u + (lane >> 2), sr = (wave & 3u) * 32u + (lane >> 1);
  const uint32_t wo = (min(n0 + wr, N - 1u) * nblk + ((lane & 3u) ^ (wr >> 2 & 3u))) << 4;       // 16 rows of 64 bytes; LDS: [row][4 blocks]
  const uint32_t so = (min(n0 + sr, N - 1u) * nblk + (lane & 1u) * 2u) * 2u;                     // 32 rows of 8 bytes; LDS: [row][4]
  const u4q_t* const xp = wave >= 4u ? xl : xh;
  const auto load = [&](int i, uint32_t s, uint32_t into) {  // (steps past the end re-read the last: the count in flight stays)
    const uint64_t st = min(s, steps - 1u);
    const uint32_t at = base + into * NARROW_STAGE;
    if (i < 2) load_to_lds(xp + st * 16u, xo[i], at + (wave * 2u + i) * 1024u);
    else if (i == 2) load_to_lds(W + (((uint64_t)gbase + st * 4u) << 4), wo, at + NARROW_X + wave * 1024u);
    else load4_to_lds(d16 + gbase + st * 4u, so, at + NARROW_X + NARROW_W + (wave & 3u) * 256u);
  };

  f16q_t acc[2], blk[2][2], zero;                            // blk: a block's products, [step's parity][tile]
#pragma unroll
  for (int i = 0; i < 16; i++) { zero[i] = 0.f; acc[0][i] = 0.f; acc[1][i] = 0.f; blk[1][0][i] = 0.f; blk[1][1][i] = 0.f; }
  DEQK_INIT(dk);
  u4q_t x[2][4], raw[2][2];                                  // [step's parity][plane, half of the block], [..][tile]
  _Float16 ds[2][2];
  float d[2] = {0.f, 0.f};
  const auto add = [&](int p, int i0, int i1) {              // results i0 .. i1 of both tiles, each block's sum by its scale
#pragma unroll
    for (int i = i0; i < i1; i++) acc[i >> 4][i & 15] = fmaf(blk[p][i >> 4][i & 15], d[i >> 4], acc[i >> 4][i & 15]);
  };
  const auto read = [&](int i, int p, uint32_t buf) {
    const uint8_t* const st = ring + buf * NARROW_STAGE;
    if (i < 4) x[p][i] = *(const u4q_t*)(st + (i >> 1) * 8192u + r32 * 256u + (((4u * kb + 2u * (i & 1) + h) ^ (r32 & 15u)) << 4));
    else {
      const uint32_t row = side * 64u + (i - 4) * 32u + r32;
      raw[p][i - 4] = *(const u4q_t*)(st + NARROW_X + row * 64u + ((kb ^ (row >> 2 & 3u)) << 4));
      ds[p][i - 4] = *(const _Float16*)(st + NARROW_X + NARROW_W + row * 8u + kb * 2u);
    }
  };
#pragma unroll
  for (uint32_t s = 0; s < ST; s++)
#pragma unroll
    for (int i = 0; i < LOADS; i++) load(i, s, s);
  ring_wait<LOADS * (ST - 1)>();
#pragma unroll
  for (int i = 0; i < 6; i++) read(i, 0, 0);
  uint32_t buf = 0;
  const auto step = [&](int p, uint32_t s) {
    const uint32_t next = buf + 1u == ST ? 0u : buf + 1u;
    ring_wait<LOADS * (ST - 2)>();                           // the next step is here, this one's operands are in registers
    u4q_t wf[2][2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      wf[t][0] = deq_word(h ? raw[p][t].y : raw[p][t].x, dk);
      wf[t][1] = deq_word(h ? raw[p][t].w : raw[p][t].z, dk);
    }
#pragma unroll
    for (int m = 0; m < 4; m++) {
#pragma unroll
      for (int t = 0; t < 2; t++) blk[p][t] = MFMA32_F16(x[p][m], wf[t][m & 1], m ? blk[p][t] : zero);
      add(1 - p, 8 * m, 8 * m + 8);                          // (of the step before: its products are there)
      if (m < 3) { read(2 * m, 1 - p, next); read(2 * m + 1, 1 - p, next); }
      load(m, s + ST, buf);
      __builtin_amdgcn_sched_barrier(0);
    }
    d[0] = (float)ds[p][0]; d[1] = (float)ds[p][1];
    buf = next;
  };
  for (uint32_t s = 0; s < steps; s += 2u) {
    step(0, s);
    if (s + 1u < steps) step(1, s + 1u);
  }
  if (steps & 1u) add(0, 0, 32); else add(1, 0, 32);
  ring_wait<0>();
  // the waves' sums: eight results of each lane a wave, quads of them beside each other
  f4q_t* const sums = (f4q_t*)ring;
#pragma unroll
  for (int q = 0; q < 8; q++)
    sums[(wave * 8u + q) * 64u + lane] = (f4q_t){acc[q >> 2][4 * (q & 3)], acc[q >> 2][4 * (q & 3) + 1], acc[q >> 2][4 * (q & 3) + 2], acc[q >> 2][4 * (q & 3) + 3]};
  __syncthreads();
  f4q_t y[2];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    f4q_t v[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; k++) v[k] = sums[((k * 2u + side) * 8u + kb * 2u + q) * 64u + lane];
    y[q] = ((v[0] + v[1]) + v[2]) + v[3];
  }
  const auto row = [&](int, int i) { return m0 + 16u * (kb & 1u) + 8u * (i >> 2) + 4u * h + (i & 3u); };
#pragma unroll
  for (int i = 0; i < 8; i++) y[i >> 2][i & 3] *= scale[2 * (uint64_t)min(row(0, i), M - 1u) + 1];
  const uint64_t c_off = (by_val & 2u) || segs.count ? (uint64_t)c_val : (uint64_t)lc[0];
  const uint32_t n[1] = {n0 + side * 64u + (kb >> 1) * 32u + r32};
  store_columns<1, 8, 1>([&](int, int i, int) { return y[i >> 2][i & 3]; }, row, n, M, N, 0u, c_off, out, nullptr, segs);
}

// 2 .. 64 activation rows: the weights are read once, so what counts is how fast they stream, and what stands in its way is
// the activations, of which a 16-row operand of 32 columns is 1 KB beside 288 bytes of weights.  So
//   * the rows' two planes are stacked: 2 M operand rows (xh of every row, then xl), NT tiles of 16, one instruction per tile and
//     block -- 8 rows fill one tile, 24 rows three; the planes' sums are added at the end.  9 .. 16 rows (PAIR): a tile a plane, and
//     both instructions of a block go to one sum;
//   * one tile has 4, 8 or 16 rows in memory, two as many as there are in fours: every CU reads them all, and over long K that is what
//     counts (9 rows, 4096 x 14336: 19.7 us with both planes in stacked tiles of 16, 16.1 so; 2 rows 14.2 and 10.4);
//   * operands go from memory to registers in the instruction's layout, without LDS: a wave reads 16 rows x 64 bytes at a time;
//   * the NWV waves of a workgroup share R tiles of 16 weight rows and take every NWV-th step of K (128 columns) each, so a
//     workgroup reads its activations once, and as many weight rows as a CU has share them.
// Weights are asked for D steps ahead, activations DA.  The waves' tiles are summed through LDS in wave order.
// The weights come by ordinary loads: a step takes half a line of a row and another wave's step the other half, which it finds in
// the L1.  Marked as read once, every line was asked of the L2 twice (8 rows, 4096 x 4096: 68,000 of 422,000 requests; the same
// bytes from memory), and 8 rows took 6.0 us for 4096 x 4096 (5.0 so), 8.2 for 6144 x 4096 (7.2), 16.6 for 4096 x 14336 (14.2), 8.3
// for 1152 x 6912 (6.15); 24 rows 8.6 (7.7), 11.7 (10.3), 26 (24), 13.0 (10.2).
// What bounds it is the way from the L2 for one tile of weights (of a 128-column step 4 KB are activations, 1.2 KB weights) and the
// vector work for four (75 instructions a step and tile, 36 of them unpacking).
// us, rows ready, the K-split kernel before (a tile of activations staged by every wave, both planes apart) and this one: 8 rows
// 4096 x 4096 6.5 and 5.0, 6144 x 4096 9.6 and 7.2, 4096 x 14336 16.3 and 14.2, 13824 x 1152 8.7 and 6.4; 24 rows 13.3 and 7.7, 18.5 and 10.3,
// 39 and 24, 15.0 and 8.7, 28672 x 4096 48 and 32; 32 rows 13.2 and 8.8, 19.2 and 12.1, 39.6 and 28.9, 14.9 and 9.9, 50 and 37; 9 rows 6.6
// and 5.25, 9.5 and 7.2, 16.2 and 16.1, 8.7 and 6.8, 1152 x 6912 8.1 and 6.7; 16 rows 7.2 and 6.0, 10.8 and 7.6, 20.2 and 19.2, 9.1 and 6.9,
// 8.3 and 7.3 (eight waves a step ahead; 16 waves two steps ahead 4096 x 14336 20.1).
// (segs.glu: tiles of a wave are gate, up, gate, up ...: the gated activation is stored from here.)
template <int NT, int R, int NWV, int D, int DA, bool PAIR>
__global__ void __launch_bounds__(64 * NWV)
k_gemm_q4_rows(const uint8_t* __restrict__ W, const __half* __restrict__ d16, const u4q_t* __restrict__ x, uint32_t tiles_r, uint32_t K, uint32_t N, uint32_t M, uint32_t b_val, uint32_t c_val, uint32_t by_val, float* out,
               const uint32_t* __restrict__ lb, const uint32_t* __restrict__ lc, const float* __restrict__ scale, GemmSegs segs) {
  // (the first 14 dwords of the arguments are in registers when a wave starts; by_val bit 0 / 1: the weights' / the
  // result's element offset of op 0 is b_val / c_val -- known on the host -- instead of a load from lb / lc, which
  // the first weight loads would have to wait for)
  constexpr int RC = R >= 2 ? 2 : 1;
  static_assert(DA == 1 || DA == D, "activations one step ahead, or as many as the weights");
  constexpr int NA = PAIR ? NT / 2 : NT;                     // sums of a tile of weights
  __shared__ float part[NWV * RC * NA * 256];                // [wave][tile of a pair][sums][i][lane]
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t r16 = lane & 15u, g = lane >> 4, op = blockIdx.z;
  const bool glum = R >= 2 && segs.glu != 0u;
  const uint64_t c_off = (by_val & 2u) ? (uint64_t)c_val : lc ? (uint64_t)lc[op] : 0ull, gbase = ((by_val & 1u) ? (uint64_t)b_val : (uint64_t)lb[op]) >> 5;
  const uint32_t nblk = K >> 5, kw = K >> 3, steps = nblk >> 2;
  const uint8_t* const Wb = W + (gbase << 4);
  const uint16_t* const Db = (const uint16_t*)d16 + gbase;
  // Weight loads: lane -> (row lane / 4, block lane % 4 of the step): the four lanes of a quad read 64 contiguous bytes of one
  // row, one request to the L1 instead of four; a permute brings each block to the lane that consumes it
  const int perm_addr = (int)((4u * r16 + g) << 2);
  const auto first_row = [&](int r) {
    return glum ? (blockIdx.x * (uint32_t)(R / 2) + (uint32_t)(r >> 1)) * 16u + (r & 1 ? N >> 1 : 0u) : (blockIdx.x * (uint32_t)R + (uint32_t)r) * 16u;
  };
  uint32_t wo[R];                                            // block index from Wb on (a Q4 map here has fewer than 2^32 elements)
#pragma unroll
  for (int r = 0; r < R; r++) wo[r] = min(first_row(r) + (lane >> 2), N - 1u) * nblk + (lane & 3u);
  const uint32_t tiles = tiles_r & 255u, rt = tiles_r >> 8;  // operand tiles and their rows (lanes past them: the last one's again)
  const u4q_t* const xb = x + (uint64_t)op * tiles * kw * rt;
  const uint32_t xlane = (g * rt + min(r16, rt - 1u)) * 16u;
  f4q_t acc[R][NA];
#pragma unroll
  for (int r = 0; r < R; r++)
#pragma unroll
    for (int t = 0; t < NA; t++) acc[r][t] = (f4q_t){0.f, 0.f, 0.f, 0.f};
  DEQK_INIT(dk);

  u4q_t qn[D][R], xn[DA][2][NT][2];                          // [steps ahead]; activations by pairs of blocks
  uint16_t dn[D][R];
  const auto fetch_w = [&](int slot, uint32_t s) {
    uint64_t at = min(s, steps - 1u) * 4u;
    asm volatile("" : "+s"(at));                             // (a wave's base and a lane's offset: no address arithmetic)
    const uint8_t *wp = Wb + at * 16u, *dp = (const uint8_t*)(Db + at);
#pragma unroll
    for (int r = 0; r < R; r++) {
      qn[slot][r] = *(const u4q_t*)(wp + (wo[r] << 4));
      dn[slot][r] = *(const uint16_t*)(dp + (wo[r] << 1));
    }
  };
  const auto fetch_x = [&](int slot, int u, uint32_t s) {
    const uint64_t at = (uint64_t)(min(s, steps - 1u) * 16u + u * 8u) * rt;
#pragma unroll
    for (int t = 0; t < NT; t++) {                           // (a tile past the last: its sums are not used)
      uint64_t from = (uint64_t)min((uint32_t)t, tiles - 1u) * kw * rt + at;
      asm volatile("" : "+s"(from));
      const uint8_t* p = (const uint8_t*)(xb + from);
      xn[slot][u][t][0] = *(const u4q_t*)(p + xlane); xn[slot][u][t][1] = *(const u4q_t*)(p + rt * 64u + xlane);
    }
    asm volatile("" ::: "memory");                           // the loads stay here
  };
  // one step from slot `ws` / `xs`; more: the loads of the steps that take its place
  const auto step = [&](int ws, int xs, bool more, uint32_t s) {
    u4q_t q[R];
    h4q_t ds[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
      const u4q_t v = qn[ws][r];
      q[r] = transpose_blocks((u4q_t){(uint32_t)__builtin_amdgcn_ds_bpermute(perm_addr, (int)v.x), (uint32_t)__builtin_amdgcn_ds_bpermute(perm_addr, (int)v.y),
                                      (uint32_t)__builtin_amdgcn_ds_bpermute(perm_addr, (int)v.z), (uint32_t)__builtin_amdgcn_ds_bpermute(perm_addr, (int)v.w)});
      ds[r] = gather_scales16((uint32_t)__builtin_amdgcn_ds_bpermute(perm_addr, (int)dn[ws][r]));
    }
    if (more) fetch_w(ws, s + (uint32_t)D * NWV);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 2; u++) {
#pragma unroll
      for (int e = 0; e < 2; e++) {
        const int b = 2 * u + e;
        u4q_t wq[R];
#pragma unroll
        for (int r = 0; r < R; r++) wq[r] = deq_word(b == 0 ? q[r].x : b == 1 ? q[r].y : b == 2 ? q[r].z : q[r].w, dk);
#pragma unroll
        for (int t = 0; t < NA; t++) {
          f4q_t blk[R];
#pragma unroll
          for (int r = 0; r < R; r++) blk[r] = MFMA_F16(xn[xs][u][t][e], wq[r], ((f4q_t){0.f, 0.f, 0.f, 0.f}));
          if (PAIR)
#pragma unroll
            for (int r = 0; r < R; r++) blk[r] = MFMA_F16(xn[xs][u][NT - NA + t][e], wq[r], blk[r]);
#pragma unroll
          for (int r = 0; r < R; r++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[r][t][i] = fmaf(blk[r][i], (float)ds[r][b], acc[r][t][i]);
        }
        __builtin_amdgcn_sched_barrier(0);                   // (blocks overlapped any further cost registers)
      }
      if (more || DA < D) fetch_x(xs, u, s + (uint32_t)DA * NWV);
    }
  };
  const uint32_t cnt = wave < steps ? (steps - wave + NWV - 1u) / NWV : 0u;
  uint32_t i = 0, s = wave;
#pragma unroll
  for (int d = 0; d < D; d++) {
    fetch_w(d, s + (uint32_t)d * NWV);
    if (d < DA) { fetch_x(d, 0, s + (uint32_t)d * NWV); fetch_x(d, 1, s + (uint32_t)d * NWV); }
  }
  for (; i + (uint32_t)D < cnt; i += (uint32_t)D)            // (steps past the end ask for the last one again)
#pragma unroll
    for (int d = 0; d < D; d++, s += NWV) step(d, DA == 1 ? 0 : d, true, s);
#pragma unroll
  for (int d = 0; d < D; d++, s += NWV)
    if (i + (uint32_t)d < cnt) step(d, DA == 1 ? 0 : d, false, s);

#pragma unroll
  for (int r0 = 0; r0 < R; r0 += RC) {
    if (r0) __syncthreads();
#pragma unroll
    for (int r = 0; r < RC; r++)
#pragma unroll
      for (int t = 0; t < NA; t++)
#pragma unroll
        for (int k = 0; k < 4; k++) part[((wave * RC + r) * NA + t) * 256u + k * 64u + lane] = acc[r0 + r][t][k];
    __syncthreads();
    // how: 0 one matrix, 1 and the add behind it, 2 stacked matrices (one by the stacked ones' places: 40 x 28672 x 1152 25.0 us, 23.2 so)
    const auto rows = [&](auto how) {
      for (uint32_t idx = tid; idx < M * 16u; idx += 64u * NWV) {
        // activation row `row` of tile column c: operand rows `row` and M + row of every wave (PAIR: row `row` of the one sum)
        const uint32_t row = idx >> 4, c = idx & 15u, lo = M + row;
        const auto place = [&](uint32_t v) { return (v >> 4) * 256u + (v & 3u) * 64u + ((v >> 2) & 3u) * 16u + c; };
        const float inv = scale[2 * ((uint64_t)op * M + row) + 1];
        float y[RC], old[RC];
        ColumnPlace to[RC];
#pragma unroll
        for (int r = 0; r < RC; r++) {
          const uint32_t n = min(first_row(r0 + r) + c, N - 1u);
          if (how == 2) to[r] = column_place(n, N, c_off, out, segs);
          if (how == 1) old[r] = out[segs.res + (uint64_t)row * N + n];
        }
#pragma unroll
        for (int r = 0; r < RC; r++) {
          float a = 0.f, b = 0.f;
#pragma unroll
          for (uint32_t w = 0; w < NWV; w++) {
            const float* p = part + (w * RC + r) * NA * 256u;
            a += p[place(row)];
            if (!PAIR) b += p[place(lo)];
          }
          y[r] = (a + b) * inv;
        }
#pragma unroll
        for (int r = 0; r < RC; r++) {
          const uint32_t n = first_row(r0 + r) + c;
          if (n >= (glum && !(r & 1) ? N >> 1 : N)) continue;
          if (how == 2) to[r].col[(uint64_t)row * to[r].step] = y[r];
          else out[c_off + (uint64_t)row * N + n] = y[r];
          if (how == 1) out[segs.dst + (uint64_t)row * N + n] = old[r] + y[r];
        }
        if (how == 2 && glum && first_row(r0) + c < (N >> 1))   // act(gate) * up, as the element-wise op computes it
          out[segs.dst + (uint64_t)row * (N >> 1) + first_row(r0) + c] = (segs.glu == 34u ? gelu_tanh(y[0]) : y[0] / (1.0f + expf(-y[0]))) * y[RC - 1];
      }
    };
    if (segs.count) rows(std::integral_constant<int, 2>{});
    else if (segs.add) rows(std::integral_constant<int, 1>{});
    else rows(std::integral_constant<int, 0>{});
  }
}

// Q8_0 weights (the LM head of a lockstep batch) under at most 32 activation rows: the weights are read once and nothing is
// reused, so the work is bound by how fast they stream.  The four waves of a workgroup share R tiles of 16 weight rows and
// take every fourth step of K each; the partial tiles are summed in wave order at the end.
// Lane group g wants block g of the step whole, piece j of it for instruction j: of the operand tiles those are 256 bytes in one
// piece, so the first plane's go straight to registers, refilled behind the instructions that used them; a lane past the last row
// reads that row again.  us, rows ready: staged through LDS a step ahead, whole tiles of both planes, 128256 x 4096 8 rows 128, 32 rows
// 165, 16000 x 8192 40.8 and 57.5, 4096 x 4096 32 rows 14.1; so 114, 157, 32, 52, 10.3 (from rows of the first plane, staged: 114, 158,
// 33.3, 51.8, 10.4).
// The weights are blocks of 32 code bytes, w = d (code - 128): two 16-byte loads per block, bytes widened with a byte permute
// into the fp16 pairs (1024 + code), then -1152 and d.  `lc` null: the result rows go to out[row * N + n] (a scratch buffer of
// the caller).
template <int MT, int R>
__global__ void __launch_bounds__(256)
k_gemm_q8_f16_ksplit(const uint8_t* __restrict__ W, const __half* __restrict__ d16, const u4q_t* __restrict__ x, uint32_t tiles_r,
                     uint32_t K, uint32_t N, uint32_t M, uint32_t b_val, uint32_t c_val, uint32_t by_val, float* out,
                     const uint32_t* __restrict__ lb, const uint32_t* __restrict__ lc, const float* __restrict__ scale,
                     GemmSegs segs) {
  // (by_val bit 0 / 1: the weights' / the result's element offset of op 0 is b_val / c_val -- known on the host -- instead of
  // a load from lb / lc, which the first weight loads would have to wait for)
  constexpr uint32_t NWV = 4u;
  __shared__ float part[(NWV - 1u) * R * MT * 4u * 64u];
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t r16 = lane & 15u, g = lane >> 4;
  const uint32_t op = blockIdx.z;
  const uint64_t c_off = (by_val & 2u) ? (uint64_t)c_val : lc ? (uint64_t)lc[op] : 0ull;
  const uint64_t gbase = ((by_val & 1u) ? (uint64_t)b_val : (uint64_t)lb[op]) >> 5;
  const uint32_t nblk = K >> 5, kw = K >> 3;
  // Weight loads: lane -> (row lane / 4, block lane % 4 of the step): the lanes of a quad read neighbouring blocks of one row.
  // A cross-lane permute brings each 16-byte piece (and its scale) to the lane that consumes it.
  const uint32_t lrow = lane >> 2, lblk = lane & 3u;
  const int perm_addr = (int)((4u * r16 + g) << 2);
  // segs.glu (R = 2, the matrix is [gate rows; up rows], N / 2 a multiple of 16): the workgroup's first tile is 16
  // gate rows and its second the 16 up rows that belong to them, so the gated activation can be stored from here
  const bool glum = R == 2 && segs.glu != 0u;
  uint32_t trow0[R], nrow[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    trow0[r] = glum ? (uint32_t)r * (N >> 1) + blockIdx.x * 16u : blockIdx.x * (16u * R) + r * 16u;
    nrow[r] = min(trow0[r] + lrow, N - 1u);
  }

  f4q_t acc[R][MT];
#pragma unroll
  for (int r = 0; r < R; r++)
#pragma unroll
    for (int t = 0; t < MT; t++) acc[r][t] = (f4q_t){0.f, 0.f, 0.f, 0.f};
  DEQK_INIT(dk);
  const h2q_t off_q8 = {(_Float16)-1152.f, (_Float16)-1152.f};

  // (rows 16 t .. of the first plane; there is a tile of them for every t)
  const uint32_t tiles = tiles_r & 255u, rt = tiles_r >> 8;  // operand tiles and their rows
  const u4q_t* xp[MT];
#pragma unroll
  for (uint32_t t = 0; t < MT; t++) xp[t] = x + (((uint64_t)op * tiles + t) * kw + g * 4u) * rt + min(r16, M - 1u - t * 16u);
  u4q_t xn[MT][4], qn[R], qn2[R];
  _Float16 dn[R];
  const auto fetch_w = [&](uint32_t kb) {
    kb = min(kb, nblk - 4u);
#pragma unroll
    for (int r = 0; r < R; r++) {
      const uint64_t gi = gbase + (uint64_t)nrow[r] * nblk + kb + lblk;
      qn[r] = *(const u4q_t*)(W + (gi << 5));
      qn2[r] = *(const u4q_t*)(W + (gi << 5) + 16);
      dn[r] = __builtin_bit_cast(_Float16, d16[gi]);
    }
  };
  const auto fetch_x = [&](uint32_t kb, int j) {
    kb = min(kb, nblk - 4u);
#pragma unroll
    for (int t = 0; t < MT; t++) xn[t][j] = xp[t][(uint64_t)kb * (4u * rt) + (uint32_t)j * rt];
  };
  fetch_w(wave * 4u);
#pragma unroll
  for (int j = 0; j < 4; j++) fetch_x(wave * 4u, j);

  for (uint32_t kb0 = wave * 4u; kb0 < nblk; kb0 += 4u * NWV) {
    // the step's blocks and scales, moved to the lanes that consume them
    u4q_t q[R], q2[R];
    h2q_t d2[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
#define PERM_U4(v) (u4q_t){(uint32_t)__builtin_amdgcn_ds_bpermute(perm_addr, (int)(v).x), (uint32_t)__builtin_amdgcn_ds_bpermute(perm_addr, (int)(v).y), \
                           (uint32_t)__builtin_amdgcn_ds_bpermute(perm_addr, (int)(v).z), (uint32_t)__builtin_amdgcn_ds_bpermute(perm_addr, (int)(v).w)}
      q[r] = PERM_U4(qn[r]);
      q2[r] = PERM_U4(qn2[r]);
#undef PERM_U4
      const uint32_t dbits = (uint32_t)__builtin_amdgcn_ds_bpermute(perm_addr, (int)__builtin_bit_cast(uint16_t, dn[r]));
      const _Float16 dl = __builtin_bit_cast(_Float16, (uint16_t)dbits);
      d2[r] = (h2q_t){dl, dl};
    }
    fetch_w(kb0 + 4u * NWV);
    asm volatile("" ::: "memory");                           // the loads stay here
    __builtin_amdgcn_sched_barrier(0);
    // lane group g holds block g whole; instruction j takes code bytes 8j .. 8j+7 of each of the four blocks, scaled before
    // the product
#pragma unroll
    for (int j = 0; j < 4; j++) {
      u4q_t wq[R];
#pragma unroll
      for (int r = 0; r < R; r++) {
        // piece j = code bytes 8j .. 8j+7 in two words; pair p = (byte p of the first, byte p of the second)
        const uint32_t w0 = j == 0 ? q[r].x : j == 1 ? q[r].z : j == 2 ? q2[r].x : q2[r].z;
        const uint32_t w1 = j == 0 ? q[r].y : j == 1 ? q[r].w : j == 2 ? q2[r].y : q2[r].w;
        uint32_t o[4];
#pragma unroll
        for (uint32_t p = 0; p < 4; p++) {
          const uint32_t t = __builtin_amdgcn_perm(w1, w0, 0x0C000C00u | ((4u + p) << 16) | p) | dk.magic_lo;
          o[p] = __builtin_bit_cast(uint32_t, (h2q_t)((__builtin_bit_cast(h2q_t, t) + off_q8) * d2[r]));
        }
        wq[r] = (u4q_t){o[0], o[1], o[2], o[3]};
      }
#pragma unroll
      for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < R; r++) acc[r][t] = MFMA_F16(xn[t][j], wq[r], acc[r][t]);
      fetch_x(kb0 + 4u * NWV, j);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // sum the waves' tiles in wave order; wave 0 stores
  if (wave > 0) {
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
      for (int t = 0; t < MT; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) part[((((wave - 1u) * R + r) * MT + t) * 4u + i) * 64u + lane] = acc[r][t][i];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (uint32_t w = 0; w < NWV - 1u; w++)
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
      for (int t = 0; t < MT; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) acc[r][t][i] += part[(((w * R + r) * MT + t) * 4u + i) * 64u + lane];
  // lane (r16, g) holds D[4g + i][r16]: activation rows 16 t + 4g + i, weight row r16 of tile r
  const auto row_of = [&](int t, int i) { return t * 16u + 4u * g + i; };
#pragma unroll
  for (int t = 0; t < MT; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float inv = scale[2 * ((uint64_t)op * M + min(row_of(t, i), M - 1u)) + 1];
#pragma unroll
      for (int r = 0; r < R; r++) acc[r][t][i] *= inv;
    }
  uint32_t nn[R];
#pragma unroll
  for (int r = 0; r < R; r++) nn[r] = trow0[r] + r16;
  store_columns<MT, 4, R>([&](int t, int i, int r) { return acc[r][t][i]; }, row_of, nn, M, N, 0u, c_off, out, nullptr, segs);
  if (glum && trow0[0] + r16 < (N >> 1))         // act(gate) * up, as the element-wise op computes it
#pragma unroll
  for (int t = 0; t < MT; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t row = row_of(t, i);
      if (row < M) {
        const float a = acc[0][t][i], b = acc[R - 1][t][i];
        out[segs.dst + (uint64_t)row * (N >> 1) + trow0[0] + r16] =
            segs.glu == 34u ? gelu_tanh(a) * b : (a / (1.0f + expf(-a))) * b;
      }
    }
}

// 9 .. 16 rows and many weight rows: the waves of a workgroup take 16 weight rows each and share ONE activation tile per
// step of K, staged through LDS once for all of them (the tile, both planes of all 16 rows, is 7x the bytes of a wave's
// weights: fetched by every wave, those requests to the L1, not HBM, would set the pace).
// A macro step is two steps of K (256 weights).  Registers hold rings of what is on its way: the workgroup's next
// four activation macro tiles (a thread's share: one or two pieces per plane each) and each wave's weights of the next
// four macro steps, so a CU keeps ~10 KB per wave in flight; LDS holds two macro tiles, one being read by the matrix
// instructions while the next is written, with one barrier per macro step.  Every load is issued on every path
// (clamped to the last step of K): the waits stay counted.
// segs.count: stacked matrices, as above.  segs.glu: [gate rows; up rows]: the first half of the waves takes gate
// tiles, the second half the up tiles that belong to them; the up waves hand their results over in LDS and the
// gate waves also store act(gate) * up at segs.dst.
#define R16_MS 2u
template <int NW>
__global__ void __launch_bounds__(64 * NW)
k_gemm_q4_f16_rows16(const uint8_t* __restrict__ W, const __half* __restrict__ d16, const u4q_t* __restrict__ x, uint32_t tiles_r,
                     uint32_t K, uint32_t N, uint32_t M, uint32_t b_val, uint32_t c_val, uint32_t by_val, float* out,
                     const uint32_t* __restrict__ lb, const uint32_t* __restrict__ lc, const float* __restrict__ scale,
                     GemmSegs segs) {
  // (the first 14 dwords of the arguments are in registers when a wave starts; by_val bit 0 / 1: the weights' / the
  // result's element offset of op 0 is b_val / c_val -- known on the host -- instead of a load from lb / lc, which
  // the first weight loads would have to wait for)
  constexpr uint32_t ROWB = 272u, TILE = 16u * ROWB, NT = 64u * NW;
  constexpr uint32_t PIECES = R16_MS * 256u;                 // 16-byte pieces per plane and macro step
  constexpr uint32_t NP = (PIECES + NT - 1u) / NT;           // per thread
  __shared__ __attribute__((aligned(16))) uint8_t xs_all[2u * 2u * R16_MS * TILE];   // [buffer][plane][step of the macro step]
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t r16 = lane & 15u, g = lane >> 4, op = blockIdx.z;
  const bool glum = segs.glu != 0u;
  // first weight row of the wave's tile (glu: tb = the tile's first row within its half of the matrix)
  const uint32_t tb = glum ? blockIdx.x * (8u * NW) + (wave % (NW / 2u)) * 16u : blockIdx.x * (16u * NW) + wave * 16u;
  const uint32_t n0 = glum && wave >= NW / 2u ? (N >> 1) + tb : tb;
  const uint64_t c_off = (by_val & 2u) ? (uint64_t)c_val : lc ? (uint64_t)lc[op] : 0ull;
  const uint64_t gbase = ((by_val & 1u) ? (uint64_t)b_val : (uint64_t)lb[op]) >> 5;
  const uint32_t nblk = K >> 5, kw = K >> 3, steps = nblk >> 2, macros = (steps + R16_MS - 1u) / R16_MS;
  const uint32_t lrow = lane >> 2, lblk = lane & 3u;
  const int perm_addr = (int)((4u * r16 + g) << 2);
  const uint64_t wrow = gbase + (uint64_t)min(n0 + lrow, N - 1u) * nblk + lblk;
  DEQK_INIT(dk);
  f4q_t acc = {0.f, 0.f, 0.f, 0.f};

  // a thread's pieces of a macro tile: piece w -> (step w / 256, block (w / 64) % 4 of the step, piece (w / 16) % 4 of the block,
  // row w % 16).  Second plane: the second tile
  const uint32_t rt = tiles_r >> 8;                          // rows of a tile
  uint64_t xoff[NP], xloff[NP];
  uint32_t xlds[NP], xst[NP];
#pragma unroll
  for (uint32_t u = 0; u < NP; u++) {
    const uint32_t w = min(tid + u * NT, PIECES - 1u), row = w & 15u, pc = (w >> 4) & 15u;
    xst[u] = w >> 8;
    xoff[u] = ((uint64_t)op * 2u * kw + pc) * rt + min(row, M - 1u);   // + 16 rt pieces per step of K
    xloff[u] = xoff[u] + (uint64_t)kw * rt;
    xlds[u] = xst[u] * TILE + row * ROWB + pc * 16u;
  }
  struct ActR { u4q_t h[NP], l[NP]; };
  struct WtR { u4q_t q[R16_MS]; uint32_t d[R16_MS]; };
  ActR a0, a1, a2, a3;
  WtR w0, w1, w2, w3;
  // (steps past the end of K ask for the last step again: not used)
  auto fetch_a = [&](ActR& a, uint32_t m) {
#pragma unroll
    for (uint32_t u = 0; u < NP; u++) {
      const uint64_t at = (uint64_t)min(m * R16_MS + xst[u], steps - 1u) * (16u * rt);
      a.h[u] = x[xoff[u] + at]; a.l[u] = x[xloff[u] + at];
    }
  };
  auto fetch_w = [&](WtR& w, uint32_t m) {
#pragma unroll
    for (uint32_t s = 0; s < R16_MS; s++) {
      const uint64_t gi = wrow + min(m * R16_MS + s, steps - 1u) * 4u;
      w.q[s] = *(const u4q_t*)(W + (gi << 4));
      w.d[s] = (uint32_t)((const uint16_t*)d16)[gi];
    }
  };
  auto put_a = [&](const ActR& a, uint32_t buf) {
    uint8_t* b = xs_all + buf * (2u * R16_MS * TILE);
#pragma unroll
    for (uint32_t u = 0; u < NP; u++)
      if (NT * NP == PIECES || tid + u * NT < PIECES) {
        *(u4q_t*)(b + xlds[u]) = a.h[u];
        *(u4q_t*)(b + R16_MS * TILE + xlds[u]) = a.l[u];
      }
  };
  auto compute = [&](const WtR& w, uint32_t m, uint32_t buf) {
    const uint8_t* b0 = xs_all + buf * (2u * R16_MS * TILE);
#pragma unroll
    for (uint32_t s = 0; s < R16_MS; s++) {
      u4q_t q = {(uint32_t)__builtin_amdgcn_ds_bpermute(perm_addr, (int)w.q[s].x), (uint32_t)__builtin_amdgcn_ds_bpermute(perm_addr, (int)w.q[s].y),
                 (uint32_t)__builtin_amdgcn_ds_bpermute(perm_addr, (int)w.q[s].z), (uint32_t)__builtin_amdgcn_ds_bpermute(perm_addr, (int)w.q[s].w)};
      const uint32_t dbits = (uint32_t)__builtin_amdgcn_ds_bpermute(perm_addr, (int)w.d[s]);
      q = transpose_blocks(q);
      const f4q_t ds = gather_scales(__builtin_bit_cast(_Float16, (uint16_t)dbits));
      if (m * R16_MS + s < steps) {     // (uniform; the last macro step of an odd number of steps is half empty)
        const uint8_t* xs = b0 + s * TILE;
        const uint8_t* xs2 = xs + R16_MS * TILE;
#pragma unroll
        for (int b = 0; b < 4; b++) {
          const u4q_t wq = deq_word(b == 0 ? q.x : b == 1 ? q.y : b == 2 ? q.z : q.w, dk);
          const uint32_t xo = r16 * ROWB + b * 64u + g * 16u;
          const u4q_t ah = *(const u4q_t*)(xs + xo), al = *(const u4q_t*)(xs2 + xo);
          f4q_t blk = MFMA_F16(ah, wq, ((f4q_t){0.f, 0.f, 0.f, 0.f}));
          blk = MFMA_F16(al, wq, blk);
          const float d = ds[b];
#pragma unroll
          for (int i = 0; i < 4; i++) acc[i] = fmaf(blk[i], d, acc[i]);
        }
      }
    }
  };
  // prologue: activation tiles 0 .. 4 and weights 0 .. 3, in the order the loop issues them (a tile, then the weights
  // that go with it: loads return in order, and the tile is waited for first), so that the loop's first wait finds
  // the same loads behind its tile whether it is entered from here or from its own end
  fetch_a(a0, 0u);
  fetch_a(a1, 1u); fetch_w(w0, 0u); fetch_a(a2, 2u); fetch_w(w1, 1u); fetch_a(a3, 3u); fetch_w(w2, 2u);
  asm volatile("" ::: "memory");   // the loads stay here: none of them is moved below the first tile's wait
  __builtin_amdgcn_sched_barrier(0);
  put_a(a0, 0u);
  __builtin_amdgcn_sched_barrier(0);
  fetch_a(a0, 4u); fetch_w(w3, 3u);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();
  // macro step m: tile m + 1 goes to LDS, tile m + 5 and the weights of m + 4 are asked for, m is computed
#define R16_STEP(AR, WR, mm)                                       \
  {                                                                \
    put_a(AR, ((mm) + 1u) & 1u);                                   \
    __builtin_amdgcn_sched_barrier(0);                             \
    fetch_a(AR, (mm) + 5u);                                        \
    __builtin_amdgcn_sched_barrier(0);                             \
    compute(WR, (mm), (mm) & 1u);                                  \
    __builtin_amdgcn_sched_barrier(0);                             \
    fetch_w(WR, (mm) + 4u);                                        \
    __builtin_amdgcn_sched_barrier(0);                             \
    __syncthreads();                                               \
  }
  // (four macro steps per round and one way out: steps past the end of K compute nothing)
  for (uint32_t m = 0; m < macros; m += 4u) {
    R16_STEP(a1, w0, m);
    R16_STEP(a2, w1, m + 1u);
    R16_STEP(a3, w2, m + 2u);
    R16_STEP(a0, w3, m + 3u);
  }
#undef R16_STEP
  // lane (r16, g) holds D[4g + i][r16]: activation row 4g + i, weight row n0 + r16
  const uint32_t n = n0 + r16;
  float y[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t row = min(4u * g + i, M - 1u);
    y[i] = acc[i] * scale[2 * ((uint64_t)op * M + row) + 1];
  }
  float* ybuf = (float*)xs_all;            // the up waves' tiles, [wave - NW / 2][i][lane]
  if (glum && wave >= NW / 2u) {
#pragma unroll
    for (int i = 0; i < 4; i++) ybuf[((wave - NW / 2u) * 4u + i) * 64u + lane] = y[i];
  }
  if (glum) __syncthreads();
  const bool n_ok = glum ? tb + r16 < (N >> 1) : n < N;
  if (!segs.count) {
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (4u * g + i < M && n_ok) out[c_off + (uint64_t)(4u * g + i) * N + n] = y[i];
    return;
  }
  const ColumnPlace to = column_place(n, N, c_off, out, segs);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t row = 4u * g + i;
    if (row >= M || !n_ok) continue;
    to.col[(uint64_t)row * to.step] = y[i];
    if (glum && wave < NW / 2u) {
      const float a = y[i], b = ybuf[(wave * 4u + i) * 64u + lane];
      out[segs.dst + (uint64_t)row * (N >> 1) + n] = segs.glu == 34u ? gelu_tanh(a) * b : (a / (1.0f + expf(-a))) * b;
    }
  }
}

// The same conversion with the row held in registers: 1024 threads, thread t owns the 8-element words
// t, t + 1024, ... (NW of them; K <= 8192 NW), so the row makes one trip from memory instead of two
// dependent passes -- the rows of a decode batch are few and each workgroup's latency is the launch's.
// GLU: the rows are first produced here, as the gated activation of two inputs (element offsets glu.a, glu.b; the
// float32 result goes to glu.d, as the element-wise op stores it: op2 34 = GELU(a) b, 35 = SiLU(a) b), so the op and
// the conversion of its result are one launch and one trip.
struct GluSrc { uint32_t op, a, b, d; };
template <int NW, bool GLU>
__global__ void __launch_bounds__(1024)
k_act_f16_regs(const float* act, uint32_t K, uint32_t M, uint32_t a_val, uint32_t by_parts, uint4* xf, float* scale,
               float* act_out, const uint32_t* __restrict__ la, GluSrc glu, ActForm form) {
  // (by_parts: act_parts, and below it one bit: the rows start at element a_val -- known on the host -- instead of la[op], a load
  // the rows' loads would wait for; with GLU a_val is glu.a.  Both are in registers when a wave starts)
  __shared__ float red[16];
  const uint32_t op = blockIdx.y, tid = threadIdx.x, kw = K >> 3;
  const uint32_t parts = by_parts >> 1;
  uint32_t row = blockIdx.x, w0 = 0, w1 = kw;                // the words this workgroup stores
  if (parts) {
    const uint32_t unit = (blockIdx.x >> 6) * 8u + (blockIdx.x & 7u), share = (kw / parts + 8u) & ~7u;
    row = unit / parts * 8u + ((blockIdx.x >> 3) & 7u);
    w0 = unit % parts * share; w1 = min(kw, w0 + share);
    if (row >= M || w0 >= kw) return;
  }
  const float* x = act + (by_parts & 1u ? (uint64_t)a_val : (uint64_t)la[op]) + (uint64_t)row * K;
  f4qu_t v0[NW], v1[NW];
  float m = 0.f;
#pragma unroll
  for (int u = 0; u < NW; u++) {
    const uint32_t w = tid + 1024u * u;
    if (w < kw) {
      v0[u] = *(const f4qu_t*)(x + w * 8u);
      v1[u] = *(const f4qu_t*)(x + w * 8u + 4u);
      if (GLU) {
        const float* y = act + (uint64_t)glu.b + (uint64_t)row * K + w * 8u;
        const f4qu_t y0 = *(const f4qu_t*)y, y1 = *(const f4qu_t*)(y + 4);
        auto f = [&](float a, float b) { return glu.op == 34u ? gelu_tanh(a) * b : (a / (1.0f + expf(-a))) * b; };
        v0[u] = (f4qu_t){f(v0[u].x, y0.x), f(v0[u].y, y0.y), f(v0[u].z, y0.z), f(v0[u].w, y0.w)};
        v1[u] = (f4qu_t){f(v1[u].x, y1.x), f(v1[u].y, y1.y), f(v1[u].z, y1.z), f(v1[u].w, y1.w)};
        float* d = act_out + (uint64_t)glu.d + (uint64_t)row * K + w * 8u;
        if (w >= w0 && w < w1) { *(f4qu_t*)d = v0[u]; *(f4qu_t*)(d + 4) = v1[u]; }
      }
      m = fmaxf(m, fmaxf(fmaxf(fmaxf(fabsf(v0[u].x), fabsf(v0[u].y)), fmaxf(fabsf(v0[u].z), fabsf(v0[u].w))),
                         fmaxf(fmaxf(fabsf(v1[u].x), fabsf(v1[u].y)), fmaxf(fabsf(v1[u].z), fabsf(v1[u].w)))));
    }
  }
  m = wave_max(m);
  if ((tid & 63u) == 0) red[tid >> 6] = m;
  __syncthreads();
  m = red[0];
#pragma unroll
  for (int i = 1; i < 16; i++) m = fmaxf(m, red[i]);
  const uint32_t e = (__float_as_uint(m) >> 23) & 0xFFu;
  float s = 1.f, inv = 1.f;
  if (e >= 14u && e <= 254u) { s = __uint_as_float((267u - e) << 23); inv = __uint_as_float((e - 13u) << 23); }
  if (tid == 0 && w0 == 0) {
    scale[2 * ((uint64_t)op * M + row)] = s;
    scale[2 * ((uint64_t)op * M + row) + 1] = inv;
  }
#pragma unroll
  for (int u = 0; u < NW; u++) {
    const uint32_t w = tid + 1024u * u;
    if (w < w0 || w >= w1) continue;
    const float v[8] = {v0[u].x * s, v0[u].y * s, v0[u].z * s, v0[u].w * s, v1[u].x * s, v1[u].y * s, v1[u].z * s, v1[u].w * s};
    uint4 hi, lo;
    split_word(v, &hi, &lo);
    xf[act_piece(form, op, row, w, 0u)] = hi;
    xf[act_piece(form, op, row, w, 1u)] = lo;
  }
}

static float* g_scale_buf = nullptr;
static uint4* g_xh_buf = nullptr;     // fp16 activations, both planes, as their ActForm places them
static size_t g_xh_cap = 0;           // in bytes
static size_t g_scale_cap = 0;
// The rows last converted into g_xh_buf / g_scale_buf, and the launch and upload counts right after the
// matmul that used them: while both counts stand still nothing has written device memory since, so a
// matmul over the same rows (K and V after Q, up after gate) skips the conversion launch.  (The form
// follows from M and K; plane = bytes of one plane.)
static struct { const void* buf; uint64_t a; uint32_t M, K; uint64_t dispatch, mem_gen; size_t plane; bool valid; } g_xh_key = {};

static float* g_part_buf = nullptr;   // raw sums of the shares of a K-split launch
static size_t g_part_cap = 0;
static bool ensure_part_buf(size_t floats) {
  if (floats <= g_part_cap) return true;
  layout_changed();
  if (g_part_buf) { hipStreamSynchronize(g.stream); hipFree(g_part_buf); }
  g_part_cap = floats;
  if (hipMalloc((void**)&g_part_buf, g_part_cap * sizeof(float)) != hipSuccess) { (void)hipGetLastError(); g_part_buf = nullptr; g_part_cap = 0; return false; }
  return true;
}

static bool ensure_act_bufs(size_t scale_floats, size_t xh_bytes) {
  if (scale_floats > g_scale_cap) {
    layout_changed();
    if (g_scale_buf) { hipStreamSynchronize(g.stream); hipFree(g_scale_buf); }
    g_xh_key.valid = false;
    g_scale_cap = std::max<size_t>(scale_floats, 8192);
    if (hipMalloc((void**)&g_scale_buf, g_scale_cap * sizeof(float)) != hipSuccess) { g_scale_buf = nullptr; g_scale_cap = 0; return false; }
  }
  if (xh_bytes > g_xh_cap) {
    layout_changed();
    if (g_xh_buf) { hipStreamSynchronize(g.stream); hipFree(g_xh_buf); }
    g_xh_key.valid = false;
    g_xh_cap = xh_bytes;
    if (hipMalloc((void**)&g_xh_buf, g_xh_cap) != hipSuccess) { g_xh_buf = nullptr; g_xh_cap = 0; return false; }
  }
  return true;
}

// The form in which a matmul of M rows reads its activations, and the bytes of n_ops of them
static ActForm act_form(uint32_t M, uint32_t K, uint32_t n_ops, size_t* bytes) {
  const uint32_t kw = K >> 3, tiles = M <= 64 && (K & 127u) == 0 ? cdiv(2 * M, 16) : 0u, second = tiles == 2 ? 16u : M;
  const uint32_t rows = tiles == 2 ? cdiv(M, 4) * 4 : M <= 2 ? 4u : M <= 4 ? 8u : 16u;
  *bytes = tiles ? (size_t)n_ops * tiles * rows * 2 * K : (size_t)n_ops * M * K * 4;
  return {M, kw, tiles, second, rows, (uint64_t)n_ops * M * kw};
}

// Workgroups a row of k_act_f16_regs, 0: one, in the grid's order.  In operand tiles a row's pieces lie apart, a store of 64 of them 64
// requests where a row in one piece takes 16, and eight rows share a line: so several workgroups read a row and store a share of it
// each, and those of eight rows and a share follow each other on one die (workgroups land on the eight in turn), whose L2 then has
// the line whole.  us, conversion and matmul, one workgroup a row anywhere and so: 8 rows 4096 x 14336 20.4 and 18.8, 4096 x 4096 8.6
// and 8.1; 16 rows 24.6 and 22.9, 9.5 and 9.1, 1152 x 6912 12.3 and 11.4; 32 rows 35.2 and 32.3, 13.6 and 12.5, 18.0 and 17.0; 64 rows 43.2
// and 41.0, 21.8 and 20.1, 29.2 and 27.9.
static uint32_t act_parts(const ActForm& f) { return !f.tiles ? 0u : f.M <= 8 ? 8u : 4u; }
static uint32_t act_grid(const ActForm& f) { return f.tiles ? cdiv(cdiv(f.M, 8) * act_parts(f), 8) * 64u : f.M; }

bool gemm_act_slots(uint32_t M, uint32_t K, float** scale, uint4** x, ActForm* form) {
  if (tuning("ADAMAH_GEMM_REUSE", 1) == 0) return false;
  size_t bytes;
  *form = act_form(M, K, 1, &bytes);
  if (!ensure_act_bufs((size_t)2 * M, bytes)) return false;
  g_xh_key.valid = false;   // the buffers are about to be rewritten
  *scale = g_scale_buf;
  *x = g_xh_buf;
  return true;
}

void gemm_act_mark(const void* buf, uint64_t a, uint32_t M, uint32_t K) {
  g_xh_key = {buf, a, M, K, g.stats.dispatch, g.mem_gen, (size_t)M * K * 2, true};
}

// Gated activation (op2 34 / 35) of the [M, K] rows at a and b into the rows at d, together with the fp16 form of
// the result that a batched matmul over those rows reads: one launch, and the matmul that follows skips its
// conversion.  false: not taken (nothing launched).
bool launch_glu_act_f16(const Map* ma, uint32_t op, uint32_t a, uint32_t b, uint32_t d, uint32_t M, uint32_t K) {
  if (K > 16384u || (K & 7u) || M == 0 || knob("ADAMAH_ACT_REGS", 1) == 0) return false;
  float* scale; uint4* xf; ActForm form;
  if (!gemm_act_slots(M, K, &scale, &xf, &form)) return false;
  float* act = (float*)ma->buf;
  const GluSrc glu = {op, a, b, d};
  // (the caller has seen to it that d touches neither a nor b: several workgroups may read a row)
  if (K <= 8192) k_act_f16_regs<1, true><<<dim3(act_grid(form), 1), 1024, 0, g.stream>>>(act, K, M, a, 1u | act_parts(form) << 1, xf, scale, act, nullptr, glu, form);
  else k_act_f16_regs<2, true><<<dim3(act_grid(form), 1), 1024, 0, g.stream>>>(act, K, M, a, 1u | act_parts(form) << 1, xf, scale, act, nullptr, glu, form);
  count_launch();
  gemm_act_mark(ma->buf, d, M, K);
  return true;
}

// Merge of the attention slices of a lockstep step, one workgroup per sequence: the outputs of all the sequence's
// heads (partial[(row * heads + head) * splits + s] = {max, sum, values[D]}, at most 8 slices) are merged with the
// operations of the stand-alone merge kernel in their order, stored as the float32 row out[o0 + row * K ...]
// (K = heads * D), and converted to the fp16 form the O-projection's matmul reads -- the row is in registers, so its
// maximum costs one workgroup-wide reduction instead of a launch.
template <int NW>
__global__ void __launch_bounds__(1024)
k_attn_merge_rows_f16(float* out, const float* __restrict__ partial, uint32_t o0, uint32_t M, uint32_t K, uint32_t D,
                      uint32_t splits, float* scale, uint4* xf, ActForm form) {
  __shared__ float red[16];
  const uint32_t row = blockIdx.x, tid = threadIdx.x, kw = K >> 3, heads = K / D, stride = D + 2u, last = splits - 1u;
  float v[NW][8];
  float m = 0.f;
#pragma unroll
  for (int u = 0; u < NW; u++) {
    const uint32_t w = min(tid + 1024u * u, kw - 1u), head = (w * 8u) / D, j0 = (w * 8u) % D;
    const float* pp = partial + (uint64_t)(row * heads + head) * splits * stride;
    float ms[8], ls[8];
#pragma unroll
    for (uint32_t sp = 0; sp < 8u; sp++) { const float* ps = pp + (uint64_t)min(sp, last) * stride; ms[sp] = ps[0]; ls[sp] = ps[1]; }
    float Mx = -9.99999968e+37f;
#pragma unroll
    for (uint32_t sp = 0; sp < 8u; sp++) Mx = sp < splits ? fmaxf(Mx, ms[sp]) : Mx;
    float e[8], t[8];
#pragma unroll
    for (uint32_t sp = 0; sp < 8u; sp++) {
      e[sp] = sp < splits ? expf(ms[sp] - Mx) : 0.f;
      t[sp] = sp < splits ? fmaf(ls[sp], e[sp], 0.f) : 0.f;
    }
    // the sum of a 64-lane butterfly over lanes 0 .. 7, as the merge kernel takes it
    const float invL = 1.0f / (((t[0] + t[4]) + (t[2] + t[6])) + ((t[1] + t[5]) + (t[3] + t[7])));
    float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (uint32_t half = 0; half < 2u; half++) {
      if (half == 1u && splits <= 4u) break;
      f4qu_t a[4], b[4];
#pragma unroll
      for (uint32_t q = 0; q < 4u; q++) {
        const float* ps = pp + (uint64_t)min(half * 4u + q, last) * stride + 2 + j0;
        a[q] = *(const f4qu_t*)ps; b[q] = *(const f4qu_t*)(ps + 4);
      }
#pragma unroll
      for (uint32_t q = 0; q < 4u; q++) {
        const uint32_t sp = half * 4u + q;
        const float wg = e[sp];
        if (sp < splits) {
          o[0] += fmaf(a[q].x, wg, 0.f); o[1] += fmaf(a[q].y, wg, 0.f); o[2] += fmaf(a[q].z, wg, 0.f); o[3] += fmaf(a[q].w, wg, 0.f);
          o[4] += fmaf(b[q].x, wg, 0.f); o[5] += fmaf(b[q].y, wg, 0.f); o[6] += fmaf(b[q].z, wg, 0.f); o[7] += fmaf(b[q].w, wg, 0.f);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < 8; k++) v[u][k] = o[k] * invL;
    if (tid + 1024u * u < kw) {
      float* d = out + (uint64_t)o0 + (uint64_t)row * K + w * 8u;
      *(f4qu_t*)d = (f4qu_t){v[u][0], v[u][1], v[u][2], v[u][3]};
      *(f4qu_t*)(d + 4) = (f4qu_t){v[u][4], v[u][5], v[u][6], v[u][7]};
#pragma unroll
      for (int k = 0; k < 8; k++) m = fmaxf(m, fabsf(v[u][k]));
    }
  }
  m = wave_max(m);
  if ((tid & 63u) == 0) red[tid >> 6] = m;
  __syncthreads();
  m = red[0];
#pragma unroll
  for (int i = 1; i < 16; i++) m = fmaxf(m, red[i]);
  const uint32_t ex = (__float_as_uint(m) >> 23) & 0xFFu;
  float s = 1.f, inv = 1.f;
  if (ex >= 14u && ex <= 254u) { s = __uint_as_float((267u - ex) << 23); inv = __uint_as_float((ex - 13u) << 23); }
  if (tid == 0) { scale[2 * (uint64_t)row] = s; scale[2 * (uint64_t)row + 1] = inv; }
#pragma unroll
  for (int u = 0; u < NW; u++) {
    const uint32_t w = tid + 1024u * u;
    if (w >= kw) continue;
    const float x[8] = {v[u][0] * s, v[u][1] * s, v[u][2] * s, v[u][3] * s, v[u][4] * s, v[u][5] * s, v[u][6] * s, v[u][7] * s};
    uint4 hi, lo;
    split_word(x, &hi, &lo);
    xf[act_piece(form, 0u, row, w, 0u)] = hi;
    xf[act_piece(form, 0u, row, w, 1u)] = lo;
  }
}

// The launch of the kernel above: M sequences' merged heads as rows [M, K] at element o0 of the map, plus their fp16
// form for the matmul that follows.  false: not taken (nothing launched).
bool launch_attn_merge_rows_f16(const Map* ma, const float* partial, uint32_t o0, uint32_t M, uint32_t K, uint32_t D,
                                uint32_t splits) {
  if (K > 8192u || (K & 7u) || (D & 7u) || K % D || splits < 2 || splits > 8 || M == 0 || knob("ADAMAH_ACT_REGS", 1) == 0) return false;
  float* scale; uint4* xf; ActForm form;
  if (!gemm_act_slots(M, K, &scale, &xf, &form)) return false;
  k_attn_merge_rows_f16<1><<<M, 1024, 0, g.stream>>>((float*)ma->buf, partial, o0, M, K, D, splits, scale, xf, form);
  count_launch();
  gemm_act_mark(ma->buf, o0, M, K);
  return true;
}

// Forget converted rows (after a stream capture: the launch count is rewound there, and the note must not
// survive into a later state with the same count).
void gemm_act_forget() { g_xh_key.valid = false; }

// How a one-op Q4 matmul of more than 32 rows over a matrix [N, K] from element b on (b < 0: not known here) runs: ma > 1
// k_gemm_q4_ring<ma>, 1 k_gemm_q4_narrow, 0 the tiled kernel, over how many shares of K; -1 k_gemm_q4_rows.
// (All us with the conversion of the rows.)  33 .. 64 rows: k_gemm_q4_rows where a CU has few tiles of 16 weight rows and K is not long, by its time for a round of
// tiles and a 128-column step (48 rows: 4096 x 4096 16.0, tiled 21.5, 6144 x 4096 17.4 and 23.7; 4096 x 14336 38.1 and 32.7; 64 rows:
// 28672 x 4096 66.5 and 57.6).  Otherwise tiled; its 64 x 256 tile over shares takes 3 us a 128-column step and 11 for the two launches while no CU has
// a second one, 4.7 and 17.8 beyond, and a pass over the sums each (48 x 4096 x 14336: 142 in one, 33 over 16 shares; 64 x 28672 x 2048
// 36.7 in one, 38.5 in four, 64 x 28672 x 4096 63.5 and 57.6).
// More: the least of these estimates.  Over 850 products of 65 .. 2100 rows by 64 .. 33000 x 128 .. 14336 the plan it picks takes, against the best of tiled, narrow
// and the ring's own plan, 2.8 % longer in the mean under 2048 columns (40 % at most, 551 rows of 6096 x 1792: 57 tiled, 41 over two shares of the ring,
// whose estimates lie above what it takes), 11 % from there on (91 %, 65 rows of 4096 x 2048: 22.5 tiled, 11.7 narrow, which has no part there).  Tiled, by the
// tile it would take
// (below): 128-column steps of 1.27 us while no CU has a second 64 x 64 tile and 0.72 more for each further one, 4.0 and 2.7
// more for every two rounds of 64 x 128, 4.6 a round of 256 x 128.  Ring: 64-column steps of 1.7 (ma = 2), 2.35 (3) or 3.0 us (4), up to a
// quarter more as the CUs fill; shares cost their second launch and a pass over the sums each, where N is no multiple of four two and a
// half (a result at a time, one share behind the other: 88 rows of 9007 x 5760 50 over 7 shares of 64 rows a workgroup, 57 over
// 13 of 96, of 9008 x 5760 45 and 41; 730 of 559 x 11904 65 over 10, 74 over 16 of 96, of 560 56 and 55).  (Without and with 96 rows a
// workgroup: 28672 x 4096 under 150 rows 106 and 98, 192 103 and 99, 288 174 and 139, 384 177 and 165;
// 4096 x 14336 288 89 and 83, 384 104 and 101; 6144 x 4096 480 68 and 63.)
// The ring reads the scales of two blocks as one word and keeps a lane's place in the rows in 32 bits (in the matrix too: a Q4
// map here has fewer than 2^32 elements): matrices that begin at an odd block stay on the tiled kernel, a narrow one from 128
// rows on over 2 .. 4 shares (256 x 128 tile; 512 x 4096 x 14336 from an odd block: 234 us in one, 160 in four).
// Rows of fewer than 2048 columns: also k_gemm_q4_narrow, in steps of 128 columns of 0.42 us with few workgroups, 0.67 with one on every CU, and 3
// a round of workgroups beside them (512 x 1536 x 1152 estimated 11.5, measured 12.5, tiled 19.3; 189 x 13824 x 1152 30.1, 28.4, tiled 29.8;
// 512 x 13824 x 1152 66, 62, ring 44), where that is a tenth less than the ring's estimate, which is above what the ring takes by that and more (512 x 6912 x 1920
// estimated 55 and 56, measured 54.5 and 47), else, where it is less than tiled, the ring (320 x 6912 x 1536 without the conversion 30.0, tiled 32.9, ring 28.7).  Longer rows go to the ring over shares of K, which is the better one where there are many of them and
// where the matrix is narrow: 512 x 4096 x 4096 51 and here 56, 70 x 1152 x 6912 26 and 36 (between them not everywhere: 189 x 4096 x 4096 32 and 28).
struct GemmPlan { int ma; uint32_t shares; };
static GemmPlan gemm_plan(uint64_t M, uint64_t K, uint64_t N, int64_t b) {
  const auto up = [](uint64_t x, uint64_t y) { return (x + y - 1) / y; };
  const auto wgs = [&](uint64_t n, uint64_t m) { return up(N, n) * up(M, m); };
  const uint64_t cu = (uint64_t)g.n_cu, steps = up(K, 128), pairs = K / 64, most = tuning("ADAMAH_GEMM_SPLITK", 1) ? 16 : 1;
  const int ring = tuning("ADAMAH_GEMM_RING", 1);
  const double pass = (double)M * (double)N * 4.0 / 4.5e6;                // one pass over a result
  double best = 0.55 + 0.72 * (double)up(wgs(64, 64), cu);                // (per step)
  if (M > 64 && wgs(256, 128) * 4 >= 3 * cu) best = 4.6 * (double)up(wgs(256, 128), cu);
  else if (M > 64 && wgs(64, 128) >= 2 * cu) best = 1.3 + 2.7 * (double)up(wgs(64, 128), 2 * cu);
  best = 4.5 + best * (double)steps;
  if (M <= 64) {
    uint64_t sp = std::min<uint64_t>(most, std::max<uint64_t>(1, 2 * cu / up(N, 256)));
    while (sp > 1 && K / sp < 512u) sp--;
    const bool alone = up(N, 256) * sp <= cu;
    const double us = (alone ? 3.0 : 4.7) * (double)up(steps, sp) + (alone ? 11.0 : 17.8) + (double)(sp + 1) * pass;
    const uint64_t two = up(N, 16) > cu ? 2 : 1, rounds = up(up(N, 16 * two), cu);
    const double step = M <= 48 ? (two > 1 ? 0.43 : 0.31) : two > 1 ? 0.53 : 0.40;
    if (4.0 + (double)(rounds * steps) * step < std::min(best, sp > 1 ? us : best)) return {-1, 1};
    return {0, sp > 1 && us < best ? (uint32_t)sp : 1u};
  }
  if (ring == 0 || b < 0 || ((b >> 5) & 1) || M * K * 2 >= (1ull << 32)) {
    const uint64_t w = wgs(256, 128);
    if (M < 128 || w * 4 >= 3 * cu) return {0, 1};
    uint64_t sp = std::min<uint64_t>(std::min<uint64_t>(4, most), cu / std::max<uint64_t>(1, w));
    while (sp > 1 && K / sp < 1024u) sp--;
    return {0, sp > 1 && w * sp * 4 >= 3 * cu ? (uint32_t)sp : 1u};
  }
  if (ring == 3) return {1, 1};
  if (ring == 2) best = 1e30;
  GemmPlan p = {0, 1};
  const double tiled = best;
  double rings = 1e30;
  GemmPlan of_rings = p;
  for (int ma = 2; ma <= 4; ma++) {
    const uint64_t tiles = wgs(512, 32 * (uint64_t)ma);
    for (uint64_t sp = 1; sp <= most && (sp == 1 || (sp * 4 <= pairs && tiles * sp <= cu)); sp++) {
      const double full = std::min(1.0, (double)(tiles * sp) / (double)cu), step = ma == 2 ? 1.7 + 0.35 * full : ma == 3 ? 2.35 + 0.6 * full : 3.0 + 0.8 * full;
      const double sums = sp == 1 ? 0.0 : N % 4 == 0 ? 9.0 + (double)(sp + 1) * pass : 7.0 + (2.5 * (double)sp - 3.0) * pass;
      const double us = (double)up(tiles * sp, cu) * ((double)up(pairs, sp) * step + 7.0) + sums;
      if (us < rings) { rings = us; of_rings = {ma, (uint32_t)sp}; }
      if (us < best) { best = us; p = of_rings; }
    }
  }
  if (ring == 1 && K < 2048) {
    const uint64_t tiles = wgs(128, 32);
    const double full = std::min(1.0, (double)tiles / (double)cu), us = 3.0 + (double)up(tiles, cu) * ((0.42 + 0.25 * full) * (double)steps + 3.0);
    if (us < tiled) p = us < 0.9 * rings ? GemmPlan{1, 1} : of_rings;
  }
  return p;
}
// Whether the matmul's launches also store an add that consumes its result (more than 32 rows, one op)
bool gemm_q4_adds(uint32_t M, uint32_t K, uint32_t N, int64_t b) {
  const GemmPlan p = gemm_plan(M, K, N, b);
  return p.ma != 0 || p.shares > 1;
}

// Preconditions (checked by the caller against the host copies of the handles): Q4 map whose blocks
// in range are in the block16 layout, K a multiple of 128, weight bases block aligned, all operands
// in range.
int launch_gemm_q4_mfma(const Map* ma, const Map* mw, const uint32_t* la, const uint32_t* lb, const uint32_t* lc,
                        uint32_t M, uint32_t K, uint32_t N, uint32_t n_ops, bool q8, float* out, int64_t a_host,
                        int64_t c_host, const GemmSegs* segs, int64_t b_host) {
  // offsets of op 0 the host knows go to the kernels by value
  const uint32_t b_val = b_host >= 0 ? (uint32_t)b_host : 0u, c_val = c_host >= 0 ? (uint32_t)c_host : 0u;
  const uint32_t by_val = n_ops == 1 ? ((b_host >= 0 ? 1u : 0u) | (c_host >= 0 ? 2u : 0u)) : 0u;
  if (((q8 || out) && M > 32) || ((out || segs) && n_ops != 1) || (out && segs) || (segs && segs->glu && M > 32) ||
      (segs && segs->add && M > 32 && (n_ops != 1 || q8 || !gemm_q4_adds(M, K, N, b_host))))
    return ADAMAH_ERR_INVALID;
  GemmSegs sg = {};
  if (segs) sg = *segs;
  const size_t need = (size_t)2 * M * n_ops;
  const size_t plane = (size_t)n_ops * M * K * 2;
  size_t act_bytes;
  const ActForm form = act_form(M, K, n_ops, &act_bytes);
  const bool reuse = g_xh_key.valid && n_ops == 1 && a_host >= 0 && g_xh_key.buf == ma->buf && g_xh_key.a == (uint64_t)a_host &&
                     g_xh_key.M == M && g_xh_key.K == K && g_xh_key.dispatch == g.stats.dispatch &&
                     g_xh_key.mem_gen == g.mem_gen && g_xh_key.plane == plane && tuning("ADAMAH_GEMM_REUSE", 1) != 0;
  g_xh_key.valid = false;
  // after the matmul: the converted rows stay usable if the result did not land on them
  auto keep = [&]() {
    if (n_ops != 1 || a_host < 0 || (c_host < 0 && !out)) return;
    const uint64_t a0 = (uint64_t)a_host, a1 = a0 + (uint64_t)M * K, c0 = (uint64_t)c_host, c1 = c0 + (uint64_t)M * N;
    if (!out && c0 < a1 && a0 < c1) return;
    g_xh_key = {ma->buf, a0, M, K, g.stats.dispatch, g.mem_gen, plane, true};
  };
  if (!reuse && !ensure_act_bufs(need, act_bytes)) return ADAMAH_ERR_MEMORY;
  float* act = (float*)ma->buf;
  uint32_t mt = M <= 16 ? 1 : M <= 32 ? 2 : M <= 64 ? 4 : 8;
  uint4* const xh = g_xh_buf;
  uint4* const xl = (uint4*)((uint8_t*)g_xh_buf + plane);
  if (!reuse) {
    if (K <= 16384 && knob("ADAMAH_ACT_REGS", 1) != 0) {
      if (K <= 8192) k_act_f16_regs<1, false><<<dim3(act_grid(form), n_ops), 1024, 0, g.stream>>>(act, K, M, a_host >= 0 ? (uint32_t)a_host : 0u, ((a_host >= 0 && n_ops == 1) ? 1u : 0u) | act_parts(form) << 1, xh, g_scale_buf, act, la, GluSrc{}, form);
      else k_act_f16_regs<2, false><<<dim3(act_grid(form), n_ops), 1024, 0, g.stream>>>(act, K, M, a_host >= 0 ? (uint32_t)a_host : 0u, ((a_host >= 0 && n_ops == 1) ? 1u : 0u) | act_parts(form) << 1, xh, g_scale_buf, act, la, GluSrc{}, form);
    } else
      k_act_f16<<<dim3(M, n_ops), 256, 0, g.stream>>>(act, la, M, K, g_scale_buf, xh, form);
    count_launch();
  }
  if (sg.glu && (sg.count != 2 || sg.n[0] != sg.n[1] || (sg.n[0] & 15u))) return ADAMAH_ERR_INVALID;
  float* const dst = out ? out : act;
  const uint32_t* const lcd = out ? nullptr : lc;
  const uint32_t by_dst = out ? (by_val & 1u) : by_val, tiles16 = cdiv(N, 16), cu = (uint32_t)g.n_cu;
  GemmPlan plan = n_ops == 1 && !q8 && !out && M > 32 ? gemm_plan(M, K, N, b_host) : GemmPlan{0, 1};
  if (q8) {
    const uint32_t R = sg.glu || (uint64_t)cdiv(N, 32) * cdiv(M, 16 * mt) * n_ops >= 2ull * cu ? 2 : 1;
    const dim3 grid(cdiv(N, 16 * R), 1, n_ops);
    // Two tiles of weights over long rows: LDS that nothing uses, so that a CU takes four workgroups and not five (128256 x 4096, 2, 8,
    // 9 and 16 rows: 111, 116, 130 and 135 us with five, 106, 113, 123 and 131 with four; 262144 x 1152: 60, 69, 75, 79 and 67, 77, 81, 84)
    const size_t spare = mt == 1 && R == 2 && K >= 2048 ? 28000 : 0;
#define GK(T, RR) k_gemm_q8_f16_ksplit<T, RR><<<grid, 256, spare, g.stream>>>(mw->buf, mw->d16, (const u4q_t*)xh, form.tiles | form.rows << 8, K, N, M, b_val, c_val, by_dst, dst, lb, lcd, g_scale_buf, sg)
    if (mt == 1) { if (R == 2) GK(1, 2); else GK(1, 1); }
    else { if (R == 2) GK(2, 2); else GK(2, 1); }
#undef GK
    count_launch();
    keep();
    return check_launch();
  }
  // 9 .. 16 activation rows and workgroups of 128 weight rows for three quarters of the CUs: the form whose eight waves share an
  // activation tile in LDS (us, this and k_gemm_q4_rows with four tiles: 16 rows 28672 x 4096 23.8 and 24.1, 65536 x 2048 25.3 and 30.1; 9 rows 24.8 and
  // 24.1, 24.9 and 29.5; 8 rows 24.9 and 19.9, 25.1 and 21.3.  With two tiles a workgroup k_gemm_q4_rows takes 22.7, 24.0, 22.0 and 22.5
  // for the four of 16 and 9 rows: the line is older than that)
  const uint32_t wgs16 = cdiv(sg.glu ? N / 2 : N, sg.glu ? 64u : 128u);
  if (form.tiles == 2 && !sg.add && (uint64_t)wgs16 * 4 >= 3ull * cu && tuning("ADAMAH_GEMM_ROWS16", 1) != 0) {
    k_gemm_q4_f16_rows16<8><<<dim3(wgs16, 1, n_ops), 512, 0, g.stream>>>(mw->buf, mw->d16, (const u4q_t*)xh, form.tiles | form.rows << 8, K, N, M, b_val, c_val, by_dst,
                                                                        dst, lb, lcd, g_scale_buf, sg);
    count_launch();
    keep();
    return check_launch();
  }
  if (M <= 32 || plan.ma < 0) {
    // As many tiles of 16 weight rows to a workgroup as a CU has: one workgroup per CU reads its activations once (8 rows: 4096 x
    // 4096 one tile 4.9 us, two 6.8; 6144 x 4096 two 6.7, four 10.0; 13824 x 1152 four 6.4, one 9.2).  One and two tiles
    // of weights take the same number of waves, so that a stacked matrix has the same sums as its parts; eight where 16 waves
    // are slower (9 .. 16 rows) or would not have the registers (more operand tiles, four tiles of weights)
    const uint32_t R = tiles16 <= cu && !sg.glu ? 1 : tiles16 <= 2 * cu || form.tiles > 4 ? 2 : 4;
    const dim3 grid(sg.glu ? cdiv(N / 2, 8 * R) : cdiv(N, 16 * R), 1, n_ops);
#define GW(T, RR, W, D, DA) k_gemm_q4_rows<T, RR, W, D, DA, T == 2><<<grid, 64 * W, 0, g.stream>>>(mw->buf, mw->d16, (const u4q_t*)xh, form.tiles | form.rows << 8, K, N, M, b_val, c_val, by_dst, dst, lb, lcd, g_scale_buf, sg)
#define GWT(T) do { if (R == 1) GW(T, 1, 8, 2, 1); else if (R == 2) GW(T, 2, 8, 2, 1); else GW(T, 4, 8, 1, 1); } while (0)
    if (form.tiles == 1) { if (R == 1) GW(1, 1, 16, 2, 2); else if (R == 2) GW(1, 2, 16, 2, 2); else GW(1, 4, 8, 1, 1); }
    else if (form.tiles == 2) { if (R == 1) GW(2, 1, 8, 1, 1); else if (R == 2) GW(2, 2, 8, 1, 1); else GW(2, 4, 8, 1, 1); }
    else if (form.tiles == 3) GWT(3);
    else if (form.tiles == 4) GWT(4);
    else if (form.tiles <= 6) { if (R == 1) GW(6, 1, 8, 2, 1); else GW(6, 2, 8, 1, 1); }
    else { if (R == 1) GW(8, 1, 8, 2, 1); else GW(8, 2, 8, 1, 1); }
#undef GWT
#undef GW
    count_launch();
    keep();
    return check_launch();
  }
  const auto wgs = [&](uint32_t rows_per_wg, uint32_t t) { return (uint64_t)cdiv(N, rows_per_wg) * cdiv(M, 16 * t) * n_ops; };
  const uint64_t want = 2ull * (uint64_t)g.n_cu;
  const auto add_up = [&](uint32_t shares) {
    const uint64_t quads = ((uint64_t)M * N + 3) / 4;
    const auto go = [&](auto* kernel) { kernel<<<cdiv(quads, 256), 256, 0, g.stream>>>(g_part_buf, shares, M, N, act, c_val, by_val, lc, g_scale_buf, sg); };
    switch (shares) {
      case 2: go(k_gemm_splitk_sum<2>); break;
      case 3: go(k_gemm_splitk_sum<3>); break;
      case 4: go(k_gemm_splitk_sum<4>); break;
      case 5: go(k_gemm_splitk_sum<5>); break;
      case 6: go(k_gemm_splitk_sum<6>); break;
      case 7: go(k_gemm_splitk_sum<7>); break;
      case 8: go(k_gemm_splitk_sum<8>); break;
      default: go(k_gemm_splitk_sum<0>); break;
    }
    count_launch();
  };
  if (plan.shares > 1 && !ensure_part_buf((size_t)plan.shares * M * N)) {
    if (sg.add && !plan.ma) return ADAMAH_ERR_MEMORY;        // (the tiled kernel in one launch stores no add; narrow tiles do, of what the ring takes)
    plan = {sg.add ? 1 : 0, 1};
  }
  if (plan.ma == 1) {
    const uint32_t run = cdiv(cdiv(N, 128) * cdiv(M, 32), 8);
    k_gemm_q4_narrow<<<run * 8, 512, 0, g.stream>>>(mw->buf, mw->d16, (const u4q_t*)xh, (const u4q_t*)xl, K, N, M, (uint32_t)(b_host >> 5), c_val, by_val, act, lc, g_scale_buf, sg);
    count_launch();
    keep();
    return check_launch();
  }
  if (plan.ma) {
    const uint32_t pairs = K >> 6, per = cdiv(pairs, plan.shares), shares = cdiv(pairs, per);
    // Tiles in runs per die where the dies would not each have whole runs of weight rows anyway, few shares leave the weights
    // the larger part, and it loads the dies as evenly (400 x 6144 x 4096 over three shares, 33 workgroups on a die: 99 us, 70)
    const uint32_t tn = cdiv(N, 512), tm = cdiv(M, 32 * plan.ma), tiles = tn * tm, run = cdiv(tiles, 8);
    const bool runs = tn % 8 != 0 && tm > 1 && shares <= 2 && run * 64 <= tiles * 9 && cdiv(run * shares * 8, g.n_cu) <= cdiv(tiles * shares, g.n_cu);
    const dim3 grid(runs ? run * 8 : tn, runs ? 1 : tm, shares);
#define GRS(T, S) k_gemm_q4_ring<T, S><<<grid, 512, 0, g.stream>>>(mw->buf, mw->d16, (const u4q_t*)xh, (const u4q_t*)xl, K, N, M, (uint32_t)(b_host >> 5), c_val, by_val | (runs ? 4u : 0u), per, act, shares > 1 ? g_part_buf : nullptr, lc, g_scale_buf, sg)
#define GR(T) do { if (s16) GRS(T, true); else GRS(T, false); } while (0)
    const bool s16 = K % 256u == 0u && ((b_host >> 5) & 7) == 0;
    if (plan.ma == 2) GR(2); else if (plan.ma == 3) GR(3); else GR(4);
#undef GR
#undef GRS
    count_launch();
    if (shares > 1) add_up(shares);
    keep();
    return check_launch();
  }
  if (plan.shares > 1) {                         // 256 weight rows a workgroup over shares of K
    const uint32_t kper = cdiv(cdiv(K >> 5, plan.shares), 4u) * 4u, shares = cdiv(K >> 5, kper);
#define GS(T, F) k_gemm_q4_f16_tiled<T, 2, 8, F><<<dim3(cdiv(N, 256), cdiv(M, 16 * T), shares), 512, 0, g.stream>>>(mw->buf, mw->d16, (const u4q_t*)xh, form, K, N, M, b_val, c_val, by_val, act, lb, lc, g_scale_buf, sg, shares, kper, g_part_buf)
    if (mt == 4) GS(4, true); else GS(8, false);      // (four tiles of rows: at most 64 of them)
#undef GS
    count_launch();
    add_up(shares);
    keep();
    return check_launch();
  }
  // Tile per workgroup: 16 NW R weight rows x 16 MT activation rows (NW waves with R tiles of 16 weight rows each).
  // Every workgroup stages its activation tile (two fp16 planes: 64 KB per step of 128 weights at MT = 8) from L2,
  // while its weights are 4.5 bits each, so the bytes a workgroup moves per flop fall with the number of weight
  // rows it covers: 512 (eight waves, R = 4) where the matrix still gives most CUs a workgroup, else 128 / 64.
  uint32_t R = 1, NW = 4;
  if (mt == 8) {
    if (wgs(256, 8) * 4 >= 3ull * (uint64_t)g.n_cu) { R = 2; NW = 8; }
    else if (wgs(128, 8) >= want) R = 2;
    else if (wgs(64, 8) >= want) R = 1;
    else mt = 4;
  }
  if (mt == 8 && knob("ADAMAH_GEMM_MT", 8) == 4) { mt = 4; NW = 4; R = 1; }
  R = (uint32_t)knob("ADAMAH_GEMM_R", (int)R);
  NW = (uint32_t)knob("ADAMAH_GEMM_NW", (int)NW) >= 8 ? 8 : 4;
  R = R >= 4 && mt == 4 ? 4 : R >= 2 ? 2 : 1;
  if (mt == 4 && NW == 8 && R == 1) R = 2;
  dim3 grid(cdiv(N, 16 * NW * R), cdiv(M, 16 * mt), n_ops);
#define GTF(T, RR, W, F) k_gemm_q4_f16_tiled<T, RR, W, F><<<grid, 64 * W, 0, g.stream>>>(mw->buf, mw->d16, (const u4q_t*)xh, form, K, N, M, b_val, c_val, by_val, act, lb, lc, g_scale_buf, sg, 1, K >> 5, nullptr)
#define GT(RR, W) do { if (form.tiles) GTF(4, RR, W, true); else GTF(4, RR, W, false); } while (0)
  if (mt == 4 && NW == 8) { if (R == 4) GT(4, 8); else GT(2, 8); }
  else if (mt == 4) { if (R == 4) GT(4, 4); else if (R == 2) GT(2, 4); else GT(1, 4); }
  else if (NW == 8) { if (R == 2) GTF(8, 2, 8, false); else GTF(8, 1, 8, false); }
  else { if (R == 2) GTF(8, 2, 4, false); else GTF(8, 1, 4, false); }
#undef GT
#undef GTF
  count_launch();
  keep();
  return check_launch();
}

void gemm_q4_mfma_release() {
  if (g_scale_buf) hipFree(g_scale_buf);
  g_scale_buf = nullptr;
  g_scale_cap = 0;
  if (g_xh_buf) hipFree(g_xh_buf);
  g_xh_buf = nullptr;
  g_xh_cap = 0;
  g_xh_key.valid = false;
  if (g_part_buf) hipFree(g_part_buf);
  g_part_buf = nullptr;
  g_part_cap = 0;
}

}  // namespace adamah

using namespace adamah;
extern "C" int adamah_hip_matmul_plan(uint32_t rows, uint32_t k, uint32_t n, uint64_t base, uint32_t* tile, uint32_t* shares) {
  if (g.n_cu <= 0 || rows <= 64u || k == 0u || (k & 127u) || n == 0u || (base & 31u) || !tile || !shares) return ADAMAH_ERR_INVALID;
  const GemmPlan p = gemm_plan(rows, k, n, (int64_t)base);
  const uint32_t units = p.ma ? k >> 6 : cdiv(k, 128), per = cdiv(units, p.shares);      // (of the ring 64 columns, of the tiled kernel 128)
  *tile = 32u * (uint32_t)p.ma;
  *shares = cdiv(units, per);
  return ADAMAH_OK;
}
