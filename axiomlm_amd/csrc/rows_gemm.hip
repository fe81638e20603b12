// Many-row GEMM (prompts): y[M][N] = x W^T for M > 64 activation rows over the tile16
// copy of a MARLIN Q4 matrix, on v_mfma_f32_16x16x32_f16.
//
// Workgroup: four waves, 16 MB activation rows x (4 NT) weight tiles of 16 rows.  A wave
// owns NT weight tiles (64 weight rows at NT = 4, or two gate / up pairs) and all of the
// workgroup's activation rows, so
//  * a weight word is expanded once per wave straight from its register to the B operand
//    (the tile16 lane order) and serves MB tiles: no weight passes through LDS and none is
//    expanded twice in a workgroup;
//  * an A fragment read from LDS (1 KB) serves NT MFMAs (64 cycles at NT = 4): the four
//    SIMDs of a CU together read 64 B per cycle, half of what LDS gives.
// The activations of a 128-column stage are copied to LDS by the loads themselves
// (buffer_load ... lds, 16 bytes per lane, no registers), one stage ahead in the other
// buffer; the 16-byte pieces of a row are stored XOR-ed with the row's low bits so that 16
// rows read at one column fall into different banks.  Weights and scales come one stage
// ahead into the other register set.  Two workgroups share a CU: one wave's expansion, LDS
// reads and barriers run while the other's MFMAs do (230 VGPRs).
//
// Measured (us per call, 7B shapes, against 64-row passes of t16g_kernel): 1000 rows, QKV
// 12288 x 4096 310 -> 100 (1005 TFLOP/s), gate / up + SwiGLU 22016 x 4096 168 (1076), down
// 4096 x 11008 100 (906), O 4096 x 4096 45 (751: 256 workgroups of 64 rows, one per CU); 2048
// rows QKV 177 (1164).  A large fp16 library product reaches 1340-1410 TFLOP/s on this card.
#include <type_traits>

#include "gemm_offsets.h"
#include "kernels.h"
#include "q4_tile16.h"
#include "t16_device.h"

namespace {

constexpr int kRThreads = 256;
constexpr int kRWaves = kRThreads / 64;
constexpr int kRStage = go::kStage;  // columns per stage (one tile16 chunk)

typedef __attribute__((address_space(3))) void lds_void;

template <int EPI, int MB, int NT, bool G128>
__global__ void __launch_bounds__(kRThreads, 2) rows_gemm_kernel(T16Args a, int n_mblk, int n_split, int n_tile) {
  constexpr bool kPair = EPI == Q4_EPI_SWIGLU;
  constexpr int TOK = 16 * MB;
  constexpr int UPW = kPair ? NT / 2 : NT;  // units per wave
  __shared__ __align__(16) f16 xs[2][TOK * kRStage];

  // Workgroup i runs on XCD i % 8: each XCD takes a contiguous range of tiles, rows
  // fastest, so that the row blocks that share weights meet in one L2.
  const int per = gridDim.x / 8;
  const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (tile >= n_tile) return;
  const int m0 = (tile % n_mblk) * TOK;
  const int sp = (tile / n_mblk) % n_split;
  const int nblk = tile / (n_mblk * n_split);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, kq = lane >> 4;
  const int unit = (nblk * kRWaves + wave) * UPW;
  const int kbA = sp * a.kb_per_split;
  const int n_st = min(a.KB, kbA + a.kb_per_split) - kbA;  // stages of this split (>= 1)
  const Unpack U{to_vgpr(a.unpack[0]), to_vgpr(a.unpack[1]), a.unpack[2], a.unpack[3]};
  const __amdgpu_buffer_rsrc_t rw =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.w16, (short)0, (int)a.w16_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.sb16, (short)0, (int)a.sb16_bytes, 0x00020000);

  // Weight tile t of the wave: unit + t, or gate tiles then their up tiles.  Tiles past
  // the matrix read its last one (never stored).  All offsets are wave-uniform but the
  // lane's own.
  int chunk0[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int u = min(kPair ? unit + (t % UPW) : unit + t, a.n_units - 1);
    chunk0[t] = (u + (kPair && t >= UPW ? a.pair_offset : 0)) * a.KB + kbA;
  }
  u32x4 wr[2][NT];
  u32x2 sr[2][NT];
  auto load_w = [&](int s, auto bc) {
    constexpr int b = decltype(bc)::value;
    // A stage past the split reads the split's last chunk again (never used).
    const int so = min(s, n_st - 1);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int ch = chunk0[t] + so;
      wr[b][t] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, lane * 16, ch * 1024, 0));
      if (G128) {
        const uint32_t v = __builtin_bit_cast(uint32_t, __builtin_amdgcn_raw_buffer_load_b32(rs, l16 * 4, ch * 64, 0));
        sr[b][t] = u32x2{v, v};
      } else {
        sr[b][t] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, l16 * 8, ch * 128, 0));
      }
    }
  };

  // Activations of stage s into buffer b: load i of wave w covers rows 16 i + 4 w .. + 3,
  // lane l the piece (l % 16) ^ (row % 16) of row l / 16 of them, which lands at LDS
  // position l % 16 of that row.  Rows past M, and columns past K, are requested out of the
  // descriptor's range; whatever the LDS rows of the former hold, their results are never stored.
  const int x_rows = min(a.M_tokens - m0, TOK), x_last = go::x_last(x_rows);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.x + (size_t)m0 * a.ldx), (short)0, x_rows * a.ldx * (int)sizeof(f16), 0x00020000);
  const int xrow = 4 * wave + kq;
  const int xoff = go::x_lane(xrow, l16, a.ldx);
  auto load_x = [&](int s, auto bc) {
    constexpr int b = decltype(bc)::value;
    const int st = kbA + min(s, n_st - 1);
    const bool half = go::x_half_stage(st, a.K);
#pragma unroll
    for (int i = 0; i < MB; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rx, (lds_void*)(&xs[b][(16 * i + 4 * wave) * kRStage]), 16,
          go::x_voff(xoff, i, x_last, 16 * x_last + xrow < x_rows, half && go::x_lane_hi(xrow, l16)),
          go::x_soff(st, i, x_last, a.ldx), 0, 0);
  };

  f32x4 acc[NT][MB];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[t][mb] = f32x4{0.f, 0.f, 0.f, 0.f};

  // K % 128 == 64: the second half of the row's last stage is past the row and must read
  // zeros whatever follows the row in memory.
  const int s_tail = a.K % kRStage != 0 && kbA + n_st == a.KB ? n_st - 1 : -1;
  using B0 = std::integral_constant<int, 0>;
  using B1 = std::integral_constant<int, 1>;
  auto stage = [&](int s, auto bc, auto bn) {
    constexpr int b = decltype(bc)::value;
    if (s == s_tail) {
      for (int i = tid; i < TOK * 8; i += kRThreads) {
        const int r = i >> 3, c = 8 + (i & 7);
        *reinterpret_cast<u32x4*>(&xs[b][r * kRStage + ((c ^ (r & 15)) * 8)]) = u32x4{0, 0, 0, 0};
      }
      __syncthreads();
    }
    load_x(s + 1, bn);
    load_w(s + 1, bn);
    const f16* xa = &xs[b][l16 * kRStage];
    const f16x8 magic = {(f16)1024.f, (f16)1024.f, (f16)64.f, (f16)64.f,
                         (f16)1024.f, (f16)1024.f, (f16)64.f, (f16)64.f};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      __builtin_amdgcn_sched_barrier(0);
      f16x8 A[MB];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        A[mb] = *reinterpret_cast<const f16x8*>(xa + mb * 16 * kRStage + (((4 * c + kq) ^ l16) * 8));
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const uint32_t word = wr[b][t][c];
        const uint32_t sbw = sr[b][t][c >> 1];
        const f16x2 sb = as_h2(sbw);
        const f16x8 sc = {sb.x, sb.x, sb.x, sb.x, sb.x, sb.x, sb.x, sb.x};
        const f16x8 bi = {sb.y, sb.y, sb.y, sb.y, sb.y, sb.y, sb.y, sb.y};
        const f16x8 B = __builtin_elementwise_fma(unpack_word(word, U) - magic, sc, bi);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[t][mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(B, A[mb], acc[t][mb], 0, 0, 0);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };

  load_x(0, B0{});
  load_w(0, B0{});
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (int s = 0;;) {
    stage(s, B0{}, B1{});
    if (++s >= n_st) break;
    stage(s, B1{}, B0{});
    if (++s >= n_st) break;
  }

  // Lane: weight rows 4 kq .. + 3 of each tile, token l16 of each 16.
  if (n_split == 1) {
    const bool vec = t16g_vec4<EPI>(a);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int tok = m0 + 16 * mb + l16;
      if (tok >= a.M_tokens) continue;
#pragma unroll
      for (int t = 0; t < UPW; ++t) {
        const int row = (unit + t) * 16 + 4 * kq;
        if (unit + t < a.n_units && row < a.N)
          t16g_store4<EPI>(a, tok, row, acc[t][mb], acc[kPair ? t + UPW : t][mb], vec);
      }
    }
  } else {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int tok = m0 + 16 * mb + l16;
      if (tok >= a.M_tokens) continue;
      float* pr = a.part_ws + ((size_t)sp * a.M_tokens + tok) * a.part_cols;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int u = kPair ? unit + (t % UPW) : unit + t;
        if (u < a.n_units)
          *reinterpret_cast<f32x4*>(pr + (u + (kPair && t >= UPW ? a.pair_offset : 0)) * 16 + 4 * kq) = acc[t][mb];
      }
    }
  }
}

constexpr int kRNT = 4;  // weight tiles per wave

int rows_units_per_block(int epi) { return kRWaves * (epi == Q4_EPI_SWIGLU ? kRNT / 2 : kRNT); }

struct RowsPlan {
  int mb, splits;
};
// Row tiles and K splits of a launch by the time each choice is expected to take: a
// workgroup's stage takes 1.8 us with 128 rows, and 1.25 us (alone on its CU) or 1.0 us (in
// company) with 64; partial tiles of split K are written and read back at about 4 TB/s and cost
// a launch.  Fitted to a sweep of 64 / 128 rows x 1-16 splits over 75-2048 rows of the four 7B
// matrices; the choice is within 8 % of the sweep's best at each (e.g. 1000 x 4096 x 4096: 64
// rows unsplit 45 us, 128 rows unsplit 63, from two splits 52; 75 x 4096 x 11008: 64 rows from
// eight splits 24 us, unsplit 103).
RowsPlan rows_plan(int M, int KB, int n_units, int epi) {
  RowsPlan best{8, 1};
  float best_us = 1e30f;
  const int nb = axm_ceil_div(n_units, rows_units_per_block(epi)), cus = axm_num_cus();
  const float cols = (float)n_units * (epi == Q4_EPI_SWIGLU ? 32.f : 16.f);
  for (int mb = 4; mb <= 8; mb += 4)
    for (int s = 1; s <= 8 && (s == 1 || s <= KB / 4); ++s) {
      const int load = axm_ceil_div(nb * axm_ceil_div(M, 16 * mb) * s, cus);  // workgroups per CU
      const float stage = mb == 8 ? 1.8f * (float)load : 0.25f + (float)load;
      const float us = (float)axm_ceil_div(KB, s) * stage + (s == 1 ? 0.f : 4.f + (float)s * (float)M * cols * 2e-6f);
      if (us < best_us) best_us = us, best = {mb, s};
    }
  return best;
}

template <int EPI, int MB>
void rows_launch(const T16Args& a, int M, int splits, hipStream_t s) {
  const int n_mblk = axm_ceil_div(M, 16 * MB);
  const int n_tile = n_mblk * splits * axm_ceil_div(a.n_units, rows_units_per_block(EPI));
  const dim3 grid(8 * axm_ceil_div(n_tile, 8));
  if (a.g128)
    hipLaunchKernelGGL((rows_gemm_kernel<EPI, MB, kRNT, true>), grid, dim3(kRThreads), 0, s, a, n_mblk, splits, n_tile);
  else
    hipLaunchKernelGGL((rows_gemm_kernel<EPI, MB, kRNT, false>), grid, dim3(kRThreads), 0, s, a, n_mblk, splits, n_tile);
}

template <int MB>
void rows_launch_epi(const T16Args& a, int M, int epi, int splits, hipStream_t s) {
  if (epi == Q4_EPI_STORE) rows_launch<Q4_EPI_STORE, MB>(a, M, splits, s);
  else if (epi == Q4_EPI_RESID) rows_launch<Q4_EPI_RESID, MB>(a, M, splits, s);
  else rows_launch<Q4_EPI_SWIGLU, MB>(a, M, splits, s);
}

}  // namespace

size_t t16_rows_gemm_ws_bytes(int M, int K, int n_units, int epi) {
  const int splits = rows_plan(M, (K + 127) / 128, n_units, epi).splits;
  return splits <= 1 ? 0 : (size_t)splits * M * n_units * (epi == Q4_EPI_SWIGLU ? 32 : 16) * sizeof(float);
}

int t16_rows_gemm_launch(T16Args a, int M, int epi, float* ws, size_t ws_bytes, hipStream_t s) {
  if (M < 1 || a.ln_w != nullptr || a.argmax_keys != nullptr || a.x_parts != nullptr ||
      (epi != Q4_EPI_STORE && epi != Q4_EPI_RESID && epi != Q4_EPI_SWIGLU) || a.K <= 0 || a.K % 64 != 0 ||
      a.ldx % 8 != 0 || ((uintptr_t)a.x & 15) != 0 ||
      (a.post_ln_w != nullptr && (epi != Q4_EPI_RESID || a.post_norm_out == nullptr || a.ldr != a.N))) {
    axm_set_error("tile16 rows gemm: M=%d, epi=%d, K=%d unsupported (normalized 16-byte aligned activations, store / "
                  "residual / SwiGLU epilogues)", M, epi, a.K);
    return -2;
  }
  a.KB = (a.K + 127) / 128;
  const RowsPlan plan = rows_plan(M, a.KB, a.n_units, epi);
  a.M_tokens = M;
  a.part_ws = ws;
  a.part_cols = a.n_units * (epi == Q4_EPI_SWIGLU ? 32 : 16);
  int splits = plan.splits;
  const size_t one = (size_t)M * a.part_cols * sizeof(float);
  if (ws == nullptr || ws_bytes < 2 * one) splits = 1;
  else if (ws_bytes < splits * one) splits = (int)(ws_bytes / one);
  a.kb_per_split = axm_ceil_div(a.KB, splits);
  splits = axm_ceil_div(a.KB, a.kb_per_split);
  a.w16_bytes = t16_weight_bytes(a.N_rows_alloc, a.K);
  a.sb16_bytes = t16_sb_bytes(a.N_rows_alloc, a.K, a.g128);
  a.unpack[0] = 0x000F000Fu;
  a.unpack[1] = 0x00F000F0u;
  a.unpack[2] = 0x64006400u;
  a.unpack[3] = 0x54005400u;
  if (plan.mb == 4) rows_launch_epi<4>(a, M, epi, splits, s);
  else rows_launch_epi<8>(a, M, epi, splits, s);
  return t16_gemm_finish(a, M, epi, splits, M, true, s);
}
