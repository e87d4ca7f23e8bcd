// Where a matmul's results in registers go: a lane holds single columns of one or many rows.
//
// What hangs on the column is worked out once a column, ahead of the stores, from arguments that scalar loads bring: which of the
// stacked matrices it belongs to, its first element, its rows' distance.  Looked up by result, from the arguments in memory, each would wait for
// three loads and, since loads and stores are counted together, for the store before it: 512 x 28672 x 4096 into two matrices on the
// ring 217 us, 245 with that; 512 x 13824 x 1152 42 and 59; five shares of 512 x 6144 x 4096, raw sums, 57 and 64.
#pragma once
#include "gemv_common.h"

namespace adamah {

// column n of the result: row r lies at col[r * step]
struct ColumnPlace { float* col; uint32_t step; };
__device__ __forceinline__ ColumnPlace column_place(uint32_t n, uint32_t N, uint64_t c_off, float* out, const GemmSegs& segs) {
  if (!segs.count) return {out + c_off + n, N};
  uint64_t c = segs.c[0];
  uint32_t step = segs.n[0], first = 0u;
#pragma unroll
  for (uint32_t q = 1; q < 4; q++)
    if (q < segs.count && n >= segs.begin[q]) { c = segs.c[q]; step = segs.n[q]; first = segs.begin[q]; }
  return {out + c + (n - first), step};
}

// value(t, i, w) is the result of row(t, i), i < I, and column n[w]; rows from M and columns from N on have no place.  part: raw sums of
// share kz; else the places that `segs` names, or element c_off on.  ADDS: such launches may also store the add behind a single matrix.
template <int T, int I, int W, bool ADDS = true, class V, class R>
__device__ __forceinline__ void store_columns(const V& value, const R& row, const uint32_t (&n)[W], uint32_t M, uint32_t N, uint32_t kz, uint64_t c_off,
                                              float* out, float* part, const GemmSegs& segs) {
  // (a branch for each: one matrix by way of the stacked ones' places, 2 x 13824 x 1152 of Q8 5.1 us, 4.9 so)
  if (!part && segs.count) {
    ColumnPlace to[W];
#pragma unroll
    for (int w = 0; w < W; w++) to[w] = column_place(n[w], N, c_off, out, segs);
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
      for (int i = 0; i < I; i++) {
        if (row(t, i) >= M) continue;
#pragma unroll
        for (int w = 0; w < W; w++)
          if (n[w] < N) to[w].col[(uint64_t)row(t, i) * to[w].step] = value(t, i, w);
      }
    return;
  }
  float* const at = part ? part + (uint64_t)kz * M * N : out + c_off;
  if (ADDS && !part && segs.add) {                           // the add behind it: a tile's rows are asked for at once
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
      for (int w = 0; w < W; w++) {
        if (n[w] >= N) continue;
        const float* res = out + segs.res + n[w];
        float* dst = out + segs.dst + n[w];
        float old[I];
#pragma unroll
        for (int i = 0; i < I; i++) old[i] = res[(uint64_t)min(row(t, i), M - 1u) * N];
#pragma unroll
        for (int i = 0; i < I; i++) {
          if (row(t, i) >= M) continue;
          at[(uint64_t)row(t, i) * N + n[w]] = value(t, i, w);
          dst[(uint64_t)row(t, i) * N] = old[i] + value(t, i, w);
        }
      }
    return;
  }
#pragma unroll
  for (int t = 0; t < T; t++)
#pragma unroll
    for (int i = 0; i < I; i++) {
      if (row(t, i) >= M) continue;
#pragma unroll
      for (int w = 0; w < W; w++)
        if (n[w] < N) at[(uint64_t)row(t, i) * N + n[w]] = value(t, i, w);
    }
}

}  // namespace adamah
