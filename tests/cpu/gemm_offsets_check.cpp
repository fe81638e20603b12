// CPU enumeration check of the many-row and several-row GEMMs' buffer offsets
// (axiomlm_amd/csrc/gemm_offsets.h, the same functions the kernels call).
//
// For each shape it walks every workgroup, wave, lane, piece, stage and weight tile of a launch and
// asserts, for each load, that its wave-uniform offset lies inside the buffer and that either the
// lane carries the out-of-range sentinel or both offsets together lie inside the buffer: no load
// may count on the uniform offset taking part in the range check.  Every byte of a valid row's
// columns below K must be requested exactly once per stage, and every output row stored by exactly
// one tile.  Exit status 0 and one "ok" line per group of shapes on success.
#include <cstdio>
#include <cstdlib>
#include <set>
#include <vector>

#include "gemm_offsets.h"

static int g_fail = 0;
#define CHECK(cond, ...)                                        \
  do {                                                          \
    if (!(cond)) {                                              \
      std::fprintf(stderr, "FAIL %s:%d: ", __FILE__, __LINE__); \
      std::fprintf(stderr, __VA_ARGS__);                        \
      std::fprintf(stderr, "\n");                               \
      if (++g_fail > 20) std::exit(1);                          \
    }                                                           \
  } while (0)

static bool load(const char* what, long bytes, long voff, long soff, long len) {
  CHECK(soff >= 0 && soff <= bytes, "%s: uniform offset %ld of %ld bytes", what, soff, bytes);
  if (voff == go::kOOB) return false;
  CHECK(voff >= 0 && voff + soff + len <= bytes, "%s: bytes [%ld, +%ld) of %ld", what, voff + soff, len, bytes);
  return true;
}

// Activations of all workgroups of M rows with tiles of 16 mb rows.
static void walk_x(int M, int K, int mb, bool marlin) {
  const int ldx = K, tok = 16 * mb, KB = (K + 127) / 128;
  for (int m0 = 0; m0 < M; m0 += tok) {
    const int rows = go::min_i(M - m0, tok), last = go::x_last(rows);
    const long bytes = (long)rows * ldx * 2;
    for (int st = 0; st < KB; ++st) {
      std::vector<int> seen(rows * 256);
      for (int i = 0; i < mb; ++i)
        for (int w = 0; w < 4; ++w)
          for (int n = 0; n < (marlin ? 4 : 1); ++n)
            for (int lane = 0; lane < 64; ++lane) {
              const int l16 = lane & 15, row = marlin ? 4 * w + n : 4 * w + (lane >> 4);
              const int off = marlin ? go::x_marlin_lane(row, lane, ldx) : go::x_lane(row, l16, ldx);
              const bool hi = marlin ? go::x_marlin_hi(row, lane) : go::x_lane_hi(row, l16);
              const int v = go::x_voff(off, i, last, 16 * last + row < rows, go::x_half_stage(st, K) && hi);
              const int len = marlin ? 4 : 16;
              if (!load("x", bytes, v, go::x_soff(st, i, last, ldx), len)) continue;
              const long at = v + (long)go::x_soff(st, i, last, ldx);
              CHECK(at / (2 * ldx) == 16 * go::min_i(i, last) + row, "x: row %ld for %d", at / (2 * ldx), 16 * i + row);
              if (i > last) continue;  // LDS rows that nothing uses
              for (int b = 0; b < len; ++b) ++seen[(16 * i + row) * 256 + (int)(at % (2 * ldx)) - st * 256 + b];
            }
      for (int r = 0; r < rows; ++r)
        for (int b = 0; b < 256; ++b)
          CHECK(seen[r * 256 + b] == (st * 256 + b < 2 * K ? 1 : 0), "x: row %d byte %d of stage %d seen %d times", r, b,
                st, seen[r * 256 + b]);
    }
  }
}

// Weights of format (code bytes per row and group, scale bytes, MARLIN), N rows (pair: gate and up).
static void walk_w(int N, int K, int nt, int RB, int SB, bool marlin, bool pair, bool two_bit) {
  const int KG = K / 64, KB = (K + 127) / 128, units = (N + 15) / 16, upw = pair ? nt / 2 : nt;
  const int rows = marlin ? (N + 7) & ~7 : N;
  const long wbytes = (long)(pair ? 2 * N : rows) * KG * RB, sbytes = (long)(pair ? 2 * N : rows) * KG * SB;
  std::multiset<int> stored;
  for (int blk = 0; blk < (units + 4 * upw - 1) / (4 * upw); ++blk)
    for (int w = 0; w < 4; ++w)
      for (int t = 0; t < nt; ++t) {
        const int u = (blk * 4 + w) * upw + t % upw;
        const int r0 = go::w_row0(u, units, rows), row0 = r0 + (pair && t >= upw ? N : 0);
        for (int l16 = 0; l16 < 16; ++l16) {
          const int lr = go::w_lane_row(l16, rows), row = r0 + l16;
          if (u < units && row >= u * 16 && row < N) {
            if (t < upw) stored.insert(row);
            CHECK(lr == l16, "stored row %d read by lane row %d", row, lr);
          }
          for (int kbA = 0; kbA < KB; kbA += go::max_i(1, KB / 3)) {
            const int n_grp = go::min_i(2 * (KB - kbA), KG - 2 * kbA);
            for (int kq = 0; kq < 4; ++kq)
              for (int gi = 0; gi < n_grp; ++gi) {
                if (two_bit)
                  load("2-bit codes", wbytes, (lr * KG + gi) * RB, (row0 * KG + 2 * kbA) * RB, 16);
                else
                  load("codes", wbytes, go::w_lane(marlin, lr, kq, KG, RB), go::w_soff(marlin, row0, 2 * kbA + gi, KG, RB),
                       marlin ? 8 : RB / 4);
                if (SB) load("scales", sbytes, go::s_lane(marlin, lr, gi, KG, SB), go::s_soff(marlin, row0, kbA, KG, SB), SB);
              }
          }
        }
      }
  for (int r = 0; r < N; ++r) CHECK(stored.count(r) == 1, "row %d stored %d times", r, (int)stored.count(r));
}

static void walk_q2k(int N, int K, int nt) {
  const int NB = K / 256, units = (N + 15) / 16;
  const long bytes = (long)N * NB * go::kQ2kBlock;
  for (int unit = 0; unit < units + 4 * nt; ++unit)
    for (int l16 = 0; l16 < 16; ++l16)
      for (int hb = 0; hb < 2 * NB; ++hb) {
        const int v = go::q2k_lane(go::w_lane_row(l16, N), NB), s = go::q2k_soff(go::w_row0(unit, units, N), hb, NB);
        for (int kq = 0; kq < 4; ++kq) load("q2k codes", bytes, v + 8 * kq, s + 16 + 32 * (hb & 1), 8);
        load("q2k scales", bytes, v, s + 8 * (hb & 1), 8);
        load("q2k d", bytes, v, s + 80, 4);
      }
}

int main() {
  for (int M : {1, 5, 15, 16, 17, 31, 33, 48, 63, 64, 65, 70, 75, 127, 129, 130})
    for (int K : {64, 128, 192, 320, 704, 4096})
      for (int mb : {1, 2, 3, 4, 8})
        for (bool marlin : {false, true}) walk_x(M, K, mb, marlin && mb <= 4);
  std::printf("ok activations\n");
  for (int N : {1, 4, 8, 9, 15, 16, 17, 24, 31, 33, 72, 100, 130, 136, 264, 1000})
    for (int K : {64, 128, 192, 320, 704})
      for (int nt : {2, 4}) {
        for (bool pair : {false, true}) {
          walk_w(N, K, nt, 64, 4, false, pair, false);   // Q8_G64
          walk_w(N, K, nt, 128, 0, false, pair, false);  // fp16
        }
        walk_w(N, K, nt, 16, 4, false, false, true);   // affine 2-bit
        walk_w(N, K, nt, 16, 2, false, false, true);   // ternary
        walk_w(N, K, nt, 32, 4, true, false, false);   // MARLIN
      }
  std::printf("ok weights\n");
  for (int N : {1, 15, 16, 17, 72, 130})
    for (int K : {256, 768})
      for (int nt : {2, 4}) walk_q2k(N, K, nt);
  std::printf("ok q2k\n");
  return g_fail ? 1 : 0;
}
