// Several-row GEMM over code matrices with 64-column groups and over fp16 rows (codes_gemm.hip).
#pragma once
#include "q4_tile16.h"

enum { kCodesQ8 = 0, kCodesQ2 = 1, kCodesTernary = 2, kCodesQ2kGguf = 3, kCodesMarlin = 4,
       kCodesF16 = 5 };

// a.w16 / a.sb16: the codes (uint8 [rows][K], or 2-bit [rows][K / 4]) and scales (fp16 (scale,
// bias) [rows][K / 64][2], ternary [rows][K / 64]), or the MARLIN tiles' (q4_marlin.hip);
// kCodesF16: plain fp16 weights [rows][K].  SwiGLU and residual epilogues: Q8 and fp16.
// a.x 16-byte aligned with ldx % 8 == 0; K % 64 == 0; a.N output rows (SwiGLU: gate rows [0, N),
// up rows [N, 2 N)).  Epilogues, residual norm and split_info as t16_gemm_launch.  K is split as far as
// ws_bytes allows.
bool codes_gemm_takes(const void* x, const void* w, const void* sb, int K, int rows, int fmt);
size_t codes_gemm_ws_bytes(int M, int K, int N, int epi);
int codes_gemm_launch(int fmt, T16Args a, int M, int epi, float* ws, size_t ws_bytes, hipStream_t s);
// Rows from which Q8 uses it: its GEMV takes four rows a launch (12288 x 4096: four rows 16.6 us
// against 20; five 29.8 against 20, sixteen 67 against 21, 64 rows 244 against 28; 4096 x 4096: five
// 14.5 against 11.9).
constexpr int kCodesQ8MinRows = 5;
// The fp16 GEMV takes four rows a launch too (7B-shape prompts over fp16 weights, three layers: 8 tokens
// 892 us by it, 405 here; 37 tokens 4380 / 463; 297 tokens 31.3 ms / 1.02 ms).
constexpr int kCodesF16MinRows = 5;
// The MARLIN GEMV also takes four a launch, and each of its rows costs vector work (4096 x 4096:
// three rows 10.1 us against 10.9 here, four 12.0 / 10.9, five 18.5 / 10.9; 12288 x 4096: one row 12.2 / 14.6,
// two 18.2 / 13.9, four 24.8 / 14.3; 4096 x 11008: two 17.5 / 15.8, four 36.4 / 16.1).
inline bool marlin_rows_use_codes(int M, int K, int N) {
  return M > 4 || (M > 1 && (size_t)N * K >= (size_t)32 << 20);
}
