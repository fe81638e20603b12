// Buffer offsets of the many-row and several-row GEMMs (rows_gemm.hip, codes_gemm.hip), shared
// verbatim between the kernels and a CPU check that walks whole launches and asserts that every
// offset lies inside its buffer.  Plain C++: under hipcc the functions are
// __host__ __device__, under g++ plain inline.
//
// A buffer load adds two offsets: one per lane, which its range check compares, and a wave-uniform
// one, which the check leaves out.  So a load that must read nothing carries kOOB as its lane offset
// (past every descriptor), the uniform offset never leaves the buffer, and no load relies on
// the two together being out of range.
#pragma once

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define GO_HD __host__ __device__ __forceinline__
#else
#define GO_HD inline
#endif

namespace go {

constexpr int kOOB = 0x7FFFFFF0;
constexpr int kStage = 128;     // columns per stage
constexpr int kQ2kBlock = 84;   // bytes of a GGUF Q2_K block of 256 columns

GO_HD int min_i(int a, int b) { return a < b ? a : b; }
GO_HD int max_i(int a, int b) { return a > b ? a : b; }

// ---------------------------------------------------------------------------
// Activations: a workgroup's 16 MB rows (`rows` of them in the matrix, >= 1) as pieces of 16 rows, a
// stage of 128 columns at a time.  Wave w's lane (l16, kq) takes row 4 w + kq of a piece.
// ---------------------------------------------------------------------------
GO_HD int x_last(int rows) { return (rows - 1) >> 4; }  // the last piece that holds a row

// The 16 bytes p = l16 ^ row of a stage go to LDS position l16 of the row.
GO_HD int x_lane(int row, int l16, int ldx) { return row * ldx * 2 + (l16 ^ row) * 16; }
GO_HD bool x_lane_hi(int row, int l16) { return (l16 ^ row) >= 8; }  // columns 64.. of the stage

// MARLIN order, a row per request: lane's word of row `row`.
GO_HD int x_marlin_piece(int row, int lane) { return (lane >> 2) ^ row; }
GO_HD int x_marlin_lane(int row, int lane, int ldx) {
  const int p = x_marlin_piece(row, lane);
  return row * ldx * 2 + 4 * (32 * (p >> 3) + 16 * (p & 1) + 4 * (lane & 3) + ((p >> 1) & 3));
}
GO_HD bool x_marlin_hi(int row, int lane) { return x_marlin_piece(row, lane) >= 8; }

// Lane offset of piece i: `off` where the row exists and its columns lie inside K (the last stage
// of K % 128 == 64 ends after 64).  row_in_last: the lane's row exists in piece x_last, which
// pieces past it read again (one select fewer; nothing uses them).
GO_HD int x_voff(int off, int i, int last, bool row_in_last, bool past_k) {
  const int full = past_k ? kOOB : off, ragged = row_in_last ? full : kOOB;
  return i < last ? full : ragged;
}
GO_HD int x_soff(int stage, int i, int last, int ldx) { return stage * (kStage * 2) + min_i(i, last) * 32 * ldx; }
GO_HD bool x_half_stage(int stage, int K) { return stage * kStage + 64 >= K; }

// ---------------------------------------------------------------------------
// Weights stored by rows (codes_gemm.hip).  rows: rows in memory (MARLIN: whole 8-row tiles), per
// half of a gate / up pair.  The last 16-row tile starts early enough to end with the matrix (its
// first rows repeat the tile before it and are not stored); fewer than 16 rows repeat the last.
// ---------------------------------------------------------------------------
GO_HD int w_row0(int unit, int n_units, int rows) {
  return max_i(min_i(min_i(unit, n_units - 1) * 16, rows - 16), 0);
}
GO_HD int w_lane_row(int l16, int rows) { return min_i(l16, rows - 1); }

// Codes of one group of 64 columns: RB bytes per row (MARLIN: 256 per 8-row tile and group), KG
// groups per row, a lane quarter's share RB / 4 (MARLIN: two words of the row pair's four).
GO_HD int w_lane(bool marlin, int lr, int kq, int KG, int RB) {
  return marlin ? (lr >> 3) * KG * 256 + 8 * ((kq >> 1) * 16 + (lr & 4) * 2 + (kq & 1) * 4 + (lr & 1) * 2 + ((lr >> 1) & 1))
                : lr * KG * RB + kq * (RB / 4);
}
GO_HD int w_soff(bool marlin, int row0, int g, int KG, int RB) { return row0 * KG * RB + g * (marlin ? 256 : RB); }

// Scales (SB bytes per row and group) of group g past the split's first stage kbA.
GO_HD int s_lane(bool marlin, int lr, int g, int KG, int SB) {
  return marlin ? (lr >> 3) * KG * 32 + (lr & 7) * SB + g * 32 : (lr * KG + g) * SB;
}
GO_HD int s_soff(bool marlin, int row0, int kbA, int KG, int SB) { return row0 * KG * SB + 2 * kbA * (marlin ? 32 : SB); }

// GGUF Q2_K: half block hb of row row0 + lane row.
GO_HD int q2k_lane(int lr, int NB) { return lr * NB * kQ2kBlock; }
GO_HD int q2k_soff(int row0, int hb, int NB) { return (row0 * NB + (hb >> 1)) * kQ2kBlock; }

}  // namespace go
