// What the sequence mixers with a matrix state share: sizes, and the short convolution ahead of the recurrence.
//
// The convolution's inputs of the last `taps` tokens live in a ring of `taps` places per sequence, token p at place
// p % taps: a step reads the places of the taps - 1 tokens before its own and writes its own, so workgroups need no order.
#pragma once
#include "linear_common.h"

namespace adamah {

#define CH 16u            // tokens of a chunk
#define MAX_TAPS 16       // of the short convolution
#define VC 32u            // value columns of a decode workgroup
#define NO_MEMORY 110.0f  // exp(-110) is zero in float32: a stronger decay per token changes nothing, and the sums stay small

// Forms of the walk over a portion's chunks (a workgroup: 16 value columns of a head).  FEW and DEEP have four waves of state rows and
// a fifth that adds up and stores the outputs; FEW asks for a chunk's operands when it needs them, DEEP two chunks ahead.  TURNS: as
// DEEP without the fifth wave, the four take turns with the outputs.
enum { SCAN_FEW = 0, SCAN_DEEP = 1, SCAN_TURNS = 2 };
#define SCAN_T(form) ((form) == SCAN_TURNS ? 256u : 320u)
// nt: tiles of 16 state rows a wave; two: a second workgroup of DEEP fits a CU (128 registers a lane, 4 waves a SIMD; its five do not go
// twice into 3); turns: there is such a form.  Up to a workgroup a CU a chunk's latency is all: DEEP, but for one or two chunks, whose operands
// would arrive no sooner.  Beyond, workgroups hide each other's latency: FEW, of which most fit, while the first loads count, TURNS for
// longer walks.  us, four waves of which the first has the outputs / FEW / DEEP / TURNS, delta rule, dim 128, 2048 value columns
// (256 workgroups): 1 chunk 5.8 / 4.8 / 5.4 / 5.9, 4 8.9 / 9.0 / 8.4 / 8.8, 64 71 / 78 / 60 / 68; 8192 columns: 1 12.7 / 9.7 / 15.2 / 11.4, 8 35 / 33 / 41 / 36,
// 64 219 / 238 / 247 / 221; 192 state rows, 8192 columns: 4 31 / 32 / 38 / 30, 16 78 / 95 / 91 / 77, 64 300 / 389 / 336 / 292; state space, 256 rows,
// 16384 columns: 4 27 / 29 / 33 / 28, 16 67 / 86 / 83 / 68.  DEEP twice on a CU: state space, 64 rows, 8192 columns, 64 chunks 55 / 55 / 47 / 53.
static inline int scan_form(uint64_t workgroups, uint32_t chunks, int nt, bool two, bool turns) {
  const uint64_t cu = (uint64_t)g.n_cu;
  if (workgroups <= cu) return chunks <= 2u ? SCAN_FEW : SCAN_DEEP;
  if (two && workgroups <= 2u * cu) return chunks <= 4u ? SCAN_FEW : SCAN_DEEP;
  return chunks <= (nt <= 2 ? 8u : nt == 3 || !turns ? 4u : 2u) ? SCAN_FEW : turns ? SCAN_TURNS : SCAN_DEEP;
}

__device__ __forceinline__ float softplus_f(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }
// silu of the causal convolution at token position p for channel ch, older inputs from the ring only.  The taps' loads do
// not depend on each other: up to TM of them are asked for at once (TM >= taps).
template <int TM>
__device__ __forceinline__ float conv_silu_ring(const float* x, const float* ring, uint32_t n_ch, uint32_t ch, uint32_t p,
                                                const float* w, uint32_t taps, float bias = 0.f) {
  float in[TM], wt[TM];
#pragma unroll
  for (int j = 0; j < TM; j++) {
    const bool on = (uint32_t)j < taps && (uint32_t)j <= p;
    in[j] = !on ? 0.f : j == 0 ? x[ch] : ring[(uint64_t)((p - (uint32_t)j) % taps) * n_ch + ch];
    wt[j] = on ? w[taps - 1u - (uint32_t)j] : 0.f;
  }
  float a = bias;
#pragma unroll
  for (int j = 0; j < TM; j++) a = fmaf(wt[j], in[j], a);
  return silu_f(a);
}
// The same for CH consecutive tokens of a portion: rows r0 .. r0 + CH - 1 of x (zero results from row m on), row 0 at
// position pos; put(t, value).
template <int TM, class Put>
__device__ __forceinline__ void conv_silu_rows(const float* x, uint32_t x_stride, uint32_t r0, uint32_t m, const float* ring, uint32_t n_ch,
                                               uint32_t ch, uint32_t pos, const float* w, uint32_t taps, Put put, float bias = 0.f) {
  // Every load on every path, rows beyond the portion's end read its last one: a condition around a load made each of the
  // sixteen wait for the one before (delta_prep of 2048 tokens in 32 heads of 128: 221 us, now 173).
  float in[CH + TM - 1], wt[TM], y[CH];
#pragma unroll
  for (int i = 0; i < (int)CH + TM - 1; i++) {
    const int32_t r = (int32_t)r0 + i - (TM - 1);
    in[i] = x[(uint64_t)min((uint32_t)max(r, 0), m - 1u) * x_stride + ch];
  }
#pragma unroll
  for (int j = 0; j < TM; j++) wt[j] = w[taps - 1u - min((uint32_t)j, taps - 1u)];
  if (r0 < (uint32_t)TM - 1u) {
#pragma unroll
    for (int i = 0; i < TM - 1; i++) {
      const uint32_t back = (uint32_t)(TM - 1 - i) - r0;      // rows before the portion
      if (r0 + i < (uint32_t)TM - 1u) in[i] = back < taps && back <= pos ? ring[(uint64_t)((pos - back) % taps) * n_ch + ch] : 0.f;
    }
  }
#pragma unroll
  for (int j = 0; j < TM; j++) wt[j] = (uint32_t)j < taps ? wt[j] : 0.f;
  const auto row = [&](int t) {
    float a = bias;
#pragma unroll
    for (int j = 0; j < TM; j++) a = fmaf(wt[j], in[t + TM - 1 - j], a);
    return silu_f(a);
  };
  // a whole chunk without a condition among its sixteen chains; of a shorter one only its rows (delta rule of 2 rows, 4 heads of
  // 64: 29.0 us with all sixteen, 25.2 so)
  if (m - r0 >= CH) {
#pragma unroll
    for (int t = 0; t < (int)CH; t++) y[t] = row(t);
  } else {
#pragma unroll
    for (int t = 0; t < (int)CH; t++) {
      y[t] = 0.f;
      if (r0 + (uint32_t)t < m) y[t] = row(t);
    }
  }
#pragma unroll
  for (int t = 0; t < (int)CH; t++) put(t, y[t]);
}

// Operands of the walk over the chunks: tiles of 16 x 16 in the order in which a wave's lanes take them, four consecutive floats a
// lane, so that a load is 1 KB in one piece.  In rows (element (t, d) by t) a quad of lanes lay in four rows, each a request of its
// own to the L1: a chunk's operands were 2200 clocks of requests of a compute unit, more than the chain they feed.
//   rows of tokens by d (left operand, tokens its rows):  d / 16, d / 4 % 4, t, d % 4
//   rows of d by tokens (left operand, d its rows; also a right operand, d its columns):  d / 16, t / 4, d % 16, t % 4
__device__ __forceinline__ uint32_t place16(uint32_t row, uint32_t k) { return (k >> 2) * 64u + row * 4u + (k & 3u); }   // of one tile
// A thread has the CH tokens of its d; the quad's four lanes turn theirs over four by four.  Whole quads, d % 4 a lane's place in its own.
__device__ __forceinline__ void store_rows(float* o, uint32_t d, const float (&y)[CH]) {
  const bool odd = d & 1u, high = d & 2u;
  float* to = o + (d >> 4) * 256u + ((d >> 2) & 3u) * 64u;
#pragma unroll
  for (uint32_t b = 0; b < CH; b += 4u) {
    float r[4] = {y[b], y[b + 1], y[b + 2], y[b + 3]};
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
      const float got = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(odd ? r[i] : r[i + 1]), 0xB1, 0xF, 0xF, false));
      r[i] = odd ? got : r[i];
      r[i + 1] = odd ? r[i + 1] : got;
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const float got = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(high ? r[i] : r[i + 2]), 0x4E, 0xF, 0xF, false));
      r[i] = high ? got : r[i];
      r[i + 2] = high ? r[i + 2] : got;
    }
    *(f4_t*)(to + (b + (d & 3u)) * 4u) = (f4_t){r[0], r[1], r[2], r[3]};
  }
}
__device__ __forceinline__ void store_cols(float* o, uint32_t d, const float (&y)[CH]) {
  float* to = o + (d >> 4) * 256u + (d & 15u) * 4u;
#pragma unroll
  for (uint32_t b = 0; b < CH; b += 4u) *(f4_t*)(to + b * 16u) = (f4_t){y[b], y[b + 1], y[b + 2], y[b + 3]};
}

}  // namespace adamah
