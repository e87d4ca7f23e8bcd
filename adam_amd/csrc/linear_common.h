// Products with bfloat16 weight maps: the operand structs shared by the launchers and the ops built on them.
#pragma once
#include "lanes.h"
#include "lds_ring.h"
#include "../../include/adamah_hip.h"

namespace adamah {

typedef AdamahLinearSpec LinSpec;
typedef __bf16 bf16_t;
typedef bf16_t bf8_t __attribute__((ext_vector_type(8)));
typedef bf16_t bf4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float sigmoid_f(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float silu_f(float z) { return z / (1.0f + expf(-z)); }
__device__ __forceinline__ float bf_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf_hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }

// sum over a row of 16 lanes, in all of them (lane permutations of the vector unit, no LDS)
__device__ __forceinline__ float row16_sum(float v) {
#define ROW16_ADD(ctrl) v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, 0xF, 0xF, false))
  ROW16_ADD(0xB1); ROW16_ADD(0x4E); ROW16_ADD(0x141); ROW16_ADD(0x140);   // quads, then the row's halves and the row mirrored
#undef ROW16_ADD
  return v;
}

// ---- tiles of the many-row products ---------------------------------------------------------------------------------
// R rows of 64 columns (128 bytes, a cache line) a step, loaded by NW waves, eight rows an instruction; chunk j (16 bytes)
// of a row sits at slot j ^ (row & 7), which spreads the 16-byte reads of neighbouring rows over the banks (no conflict
// counted; runs of 32 columns, whose rows are half a line, loaded 15 % slower).  Where a lane's rows start is settled once,
// so they may lie anywhere.
template <int R, int NW, bool ONCE = false> struct TileRows {
  static constexpr int N = R / (8 * NW);                     // loads a step and lane
  static_assert(N * 8 * NW == R, "whole loads");
  const bf16_t* p[N];
  template <class Row>
  __device__ __forceinline__ TileRows(uint32_t wave, uint32_t lane, Row row) {
#pragma unroll
    for (int i = 0; i < N; i++) {
      const uint32_t r = ((uint32_t)i * NW + wave) * 8u + (lane >> 3);
      p[i] = row(r) + (((lane & 7u) ^ (r & 7u)) << 3);
    }
  }
  __device__ __forceinline__ void load(int i, uint32_t k, uint32_t lds, uint32_t wave) const {      // from column k on
    if (ONCE) load_to_lds_once(p[i] + k, lds + ((uint32_t)i * NW + wave) * 1024u);
    else load_to_lds(p[i] + k, lds + ((uint32_t)i * NW + wave) * 1024u);
  }
};
// BM tokens x BN matrix rows by WM x WN waves; acc[i][j]: matrix rows wn + 16 i, tokens wm + 16 j of a wave's part; la: ST
// BN 64, lb: STX BM 64 elements.  A ring of ST buffers of 64 columns (STX of the tokens'): a step's loads are asked for ST - 1 steps ahead.  A
// step is two halves of 32 columns; a half's operands are read from LDS under the products of the half before, on both
// sides of the step's one barrier.  on: this wave has tokens.  What bounds it (256 x 256, two buffers): of the 1.7 us a step takes on all CUs the
// products need 1.0 (matrix pipe 55 .. 62 % busy over a launch of 2048 rows), its loads come out of the L2s at 8.8 TB/s, reads
// of LDS run beside both; loads and reads in a run ahead of the products instead of among them: 1.95 us.  Columns k0 .. k1 of
// the tokens; column k of them meets column k mod kp of the matrix (k1 at most PL kp).  PL = 3, tokens in pieces, the largest last: an infinite weight and a lower piece
// of 0 make no number where the whole product is infinite, so the lower pieces' sum counts only where it is finite (the
// highest one's is infinite, or no number, exactly where the whole one is).
template <int BM, int BN, int WM, int WN, int ST, int PL = 1, int STX = ST, bool ONCE = false>
__device__ __forceinline__ void tile_product(f4_t (&acc)[BN / WN / 16][BM / WM / 16], const TileRows<BN, WM * WN, ONCE>& w, const TileRows<BM, WM * WN>& x,
                                             uint32_t kp, uint32_t k0, uint32_t k1, bf16_t* la, bf16_t* lb, uint32_t wave, uint32_t lane, bool on = true) {
  constexpr int NTN = BN / WN / 16, NTM = BM / WM / 16, LW = TileRows<BN, WM * WN>::N, LX = TileRows<BM, WM * WN>::N, LOADS = LW + LX;
  constexpr int LESS = STX < ST ? STX : ST, MORE = STX < ST ? ST : STX, LF = STX < ST ? LX : LW;       // stages; loads of the operand with fewer, which go first
  static_assert(MORE - LESS <= 1, "what may be on its way at a wait");
  constexpr int FLY = (LESS - 2) * LOADS + (MORE > LESS ? LOADS - LF : 0);                  // on their way when the next step's tiles must be there
  const uint32_t c = lane & 15u, kg = lane >> 4, wn = (wave % WN) * (BN / WN), wm = (wave / WN) * (BM / WM);
  const uint32_t ba = lds_byte(la), bb = lds_byte(lb);
#pragma unroll
  for (int i = 0; i < NTN; i++)
#pragma unroll
    for (int j = 0; j < NTM; j++) acc[i][j] = (f4_t){0, 0, 0, 0};
  // load i of a step that is t steps behind the one from column k on, whose buffers are bw and bx
  const auto load_w = [&](int i, uint32_t k, uint32_t into) {     // (steps past the end re-read the last: the count in flight stays)
    const uint32_t kc = min(k, k1 - 64u), kw = PL == 1 ? kc : kc >= 2u * kp ? kc - 2u * kp : kc >= kp ? kc - kp : kc;
    w.load(i, kw, ba + into * (BN * 128u), wave);
  };
  const auto load_x = [&](int i, uint32_t k, uint32_t into) { x.load(i, min(k, k1 - 64u), bb + into * (BM * 128u), wave); };
  const auto load = [&](int i, uint32_t k, uint32_t bw, uint32_t bx) {      // of what step k has made room for
    if (STX < ST ? i < LX : i >= LW) load_x(STX < ST ? i : i - LW, k + STX * 64u, bx);
    else load_w(STX < ST ? i - LX : i, k + ST * 64u, bw);
  };
  bf8_t a[2][NTN], b[2][NTM];
  const auto read = [&](int i, uint32_t bw, uint32_t bx, int h) {
    const uint32_t at = ((4u * h + kg) ^ (c & 7u)) << 3;
    if (i < NTM) b[h][i] = *(const bf8_t*)(lb + bx * (BM * 64) + (wm + 16u * i + c) * 64u + at);
    else a[h][i - NTM] = *(const bf8_t*)(la + bw * (BN * 64) + (wn + 16u * (i - NTM) + c) * 64u + at);
  };
  // four products, then a few of the next half's reads and (second half) some of the loads, and so on: the matrix pipe is never
  // behind a run of either
  constexpr int NP = NTN * NTM / 4, READS = NP > 1 ? (NTN + NTM + NP - 2) / (NP - 1) : NTN + NTM, LOADS_EACH = (LOADS + NP - 1) / NP;
  const auto half = [&](int h, uint32_t fw, uint32_t fx, uint32_t k, uint32_t bw, uint32_t bx) {
#pragma unroll
    for (int q = 0; q < NP; q++) {
#pragma unroll
      for (int i = 0; i < READS; i++) if (q * READS + i < NTN + NTM) read(q * READS + i, fw, fx, 1 - h);
      if (h == 1) {
#pragma unroll
        for (int i = 0; i < LOADS_EACH; i++) if (q * LOADS_EACH + i < LOADS) load(q * LOADS_EACH + i, k, bw, bx);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int i = (4 * q + u) / NTM, j = (4 * q + u) % NTM;
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[h][i], b[h][j], acc[i][j], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int t = 0; t < MORE; t++) {
#pragma unroll
    for (int i = 0; i < LW; i++) if (t < ST) load_w(i, k0 + (uint32_t)t * 64u, t);
#pragma unroll
    for (int i = 0; i < LX; i++) if (t < STX) load_x(i, k0 + (uint32_t)t * 64u, t);
  }
  ring_wait<STX * LX + ST * LW - LOADS>();
  uint32_t bw = 0, bx = 0, k = k0;
  if (PL == 1 && !on) {                            // a wave without tokens: its share of the loads, and the barriers
    for (; k < k1; k += 64u, bw = bw + 1 == ST ? 0 : bw + 1, bx = bx + 1 == STX ? 0 : bx + 1) {
      ring_wait<FLY>();
#pragma unroll
      for (int i = 0; i < LOADS; i++) load(i, k, bw, bx);
    }
    ring_wait<0>();
    return;
  }
#pragma unroll
  for (int i = 0; i < NTN + NTM; i++) read(i, 0, 0, 0);
  const auto walk = [&](uint32_t end) {
    for (; k < end; k += 64u) {
      const uint32_t nw = bw + 1 == ST ? 0 : bw + 1, nx = STX == ST ? nw : bx + 1 == STX ? 0 : bx + 1;
      half(0, bw, bx, 0, 0, 0);
      ring_wait<FLY>();                            // the next step's tiles have arrived, this step's are no longer read
      half(1, nw, nx, k, bw, bx);
      bw = nw; bx = nx;
    }
  };
  if (PL == 3) {                                   // (a walk of its own: a condition in the steps cost 2 of 10 us at 16 x 512 x 512)
    walk(min(k1, 2u * kp));
    if (k0 < 2u * kp)
#pragma unroll
      for (int i = 0; i < NTN; i++)
#pragma unroll
        for (int j = 0; j < NTM; j++)
#pragma unroll
          for (int e = 0; e < 4; e++) acc[i][j][e] = __builtin_isfinite(acc[i][j][e]) ? acc[i][j][e] : 0.f;
  }
  walk(k1);
  ring_wait<0>();                                  // nothing is on its way to LDS when the workgroup ends
}
// The same in float32: 64 tokens x 64 matrix rows, 32 columns a step, on the float32 matrix instruction.  Within a run of
// 16 columns, instruction i takes column 4 g + i from lane group g on both sides, so a lane's operands are one 16-byte
// read.  wsrc, xsrc: this thread's row (tid / 4 of the tile) from column (tid % 4) 8 on.
__device__ __forceinline__ void tile_product_f32(f4_t (&acc)[2][2], const bf16_t* wsrc, const float* xsrc, uint32_t kp, float (*la)[36],
                                                 float (*lb)[36]) {
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, c = lane & 15u, kg = lane >> 4;
  const uint32_t wn = (wave & 1u) * 32u, wm = (wave >> 1) * 32u, lr = tid >> 2, lc = (tid & 3u) * 8u;
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = (f4_t){0, 0, 0, 0};
  for (uint32_t k = 0; k < kp; k += 32u) {
    const uint4 w = *(const uint4*)(wsrc + k);
    const float4 x0 = *(const float4*)(xsrc + k), x1 = *(const float4*)(xsrc + k + 4);
    __syncthreads();
    *(float4*)&la[lr][lc] = make_float4(bf_lo(w.x), bf_hi(w.x), bf_lo(w.y), bf_hi(w.y));
    *(float4*)&la[lr][lc + 4] = make_float4(bf_lo(w.z), bf_hi(w.z), bf_lo(w.w), bf_hi(w.w));
    *(float4*)&lb[lr][lc] = x0;
    *(float4*)&lb[lr][lc + 4] = x1;
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; h++) {
      f4_t a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; i++) {
        a[i] = *(const f4_t*)&la[wn + 16u * i + c][16u * h + 4u * kg];
        b[i] = *(const f4_t*)&lb[wm + 16u * i + c][16u * h + 4u * kg];
      }
#pragma unroll
      for (int t = 0; t < 4; t++)
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][t], b[j][t], acc[i][j], 0, 0, 0);
    }
  }
}

// The host copy of a spec handle, or nullptr when the handle is missing, too short or written by the device.
template <class S> inline const S* spec_of(uint32_t h) { return (const S*)res_host(h, sizeof(S) / 4); }

// Device-side growable scratch of one user; contents are only valid between launches of one op.
struct Scratch { uint8_t* p = nullptr; size_t cap = 0; };
int scratch_need(Scratch& s, size_t bytes);      // linear_bf16.hip: ADAMAH_OK or an error; never shrinks
void scratch_free(Scratch& s);

// linear_bf16.hip
int run_linear(Map* ma, Map* mo, Map* mw, const LinSpec& s, const uint32_t* row_idx, uint32_t rows);

}  // namespace adamah
