// Several-row GEMM over code matrices with a scale (and bias) per 64 columns -- row-major Q8_G64,
// ternary and affine 2-bit, and the MARLIN Q4 tiles -- on v_mfma_f32_16x16x32_f16, with exact code
// products (and over plain fp16 rows, without the scales):
//
//   y[m][n] = sum_g s_ng (sum_k q_nk x_mk) + b_ng (sum_k x_mk)       (g: 64 columns)
//
// The codes enter the MFMA as the integers themselves (fp16 holds them exactly), a group's two
// MFMAs start from zero and its fp32 sum is scaled into the accumulator, so nothing is rounded
// before fp32 (rounding each weight to fp16 first would add as much error as the fp16 result
// has).  The bias term is one bf16 MFMA per four groups on the activations' group sums: a sum
// is three bf16 parts (24 bits, cut exactly), a bias two (11 bits), and the six products fill
// one lane's eight k slots; two multiply-adds per group and element on the vector units would
// take as long as the code products.
//
// Workgroup: four waves, 16 MB rows of x, NT weight tiles of 16 rows per wave.  Lane (row r of a
// tile, quarter q) holds columns 16 q .. + 15 of a group, so its codes of a group are 16 (Q8) or
// 4 contiguous bytes; the MFMA's k order is that order of columns, also for the x fragments.
// Activations are requested to LDS one 128-column stage ahead as in the many-row tile16 GEMM
// (rows_gemm.hip), Q8 codes to registers a stage ahead (64-row tiles: a group), scales and 2-bit
// codes two stages at a time (load_pair).  Only ternary and fp16 weights multiply while those
// activations are under way: in the forms with a bias term the group sums are a second LDS array (sx), and
// the compiler, which cannot tell the two apart, waits for the requests before the stage's first
// LDS read (vmcnt(6) after three LDS and six register loads, 48 rows).
//
// Measured (us, graph of back-to-back calls, against the GEMVs of up to 4 / 16 rows a launch):
// Q8 12288 x 4096, 16 rows 67 -> 21, 64 rows 244 -> 28, 1000 rows -> 177 (569 TFLOP/s); ternary 64
// rows 91 -> 25.5, 1000 rows 150 (671); MARLIN, whose GEMV takes 4, 16 rows 98 -> 15.5, 64 rows 373 -> 27.5,
// 1000 rows 5703 -> 186 (541).  (Scales and codes loaded group by group: Q8 16 rows 25, 1000 rows
// 227; ternary 1000 rows 202.)  Large launches are bound by the vector units: per group
// and 16 x 16 tile four multiply-adds (16 cycles) and a share of the code expansion stand beside
// 32 MFMA cycles.
#include <type_traits>

#include "axm.h"
#include "codes_gemm.h"
#include "gemm_offsets.h"
#include "kernels.h"
#include "t16_device.h"

namespace {

constexpr int kCThreads = 256;
constexpr int kCWaves = kCThreads / 64;
constexpr int kCStage = go::kStage;

typedef __attribute__((address_space(3))) void lds_void;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Lane row i (lanes 16 i .. + 15) of v, in every lane row: i = 0, 1 in the first result pair
// (v_permlane32_swap of two copies gives rows 0 1 0 1 and 2 3 2 3, v_permlane16_swap of two
// copies of those one row each).
template <int HALF>
__device__ __forceinline__ u32x2 lane_rows(uint32_t v) {
  const auto p = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  const uint32_t h = HALF == 0 ? p[0] : p[1];
  const auto q = __builtin_amdgcn_permlane16_swap(h, h, false, false);
  return u32x2{q[0], q[1]};
}
// 4 x 4 transpose of words between a lane's four registers and the four lane rows.
__device__ __forceinline__ u32x4 lane_transpose(u32x4 w) {
  const auto a = __builtin_amdgcn_permlane32_swap(w.x, w.z, false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(w.y, w.w, false, false);
  const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  return u32x4{c[0], c[1], d[0], d[1]};
}

// One lane's codes of one group (16 columns) and their two MFMA operands (8 columns each).
template <int F>
struct Codes;
template <>
struct Codes<kCodesQ8> {
  static constexpr int kRowBytes64 = 64;  // code bytes of a row per group
  u32x4 w;
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    w = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
  }
  // Bytes to halves 1024 + q by one permute per pair with the exponent byte 0x64, then the
  // exact difference.
  __device__ __forceinline__ f16x8 operand(int c) const {
    const f16x2 off = {(f16)1024.f, (f16)1024.f};
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t d = w[2 * c + i];
      o[2 * i] = as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, d, 0x04010400u)) - off);
      o[2 * i + 1] = as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, d, 0x04030402u)) - off);
    }
    return __builtin_bit_cast(f16x8, o);
  }
};
// MARLIN tiles (q4_marlin.hip): a word of a row pair holds four columns 8 apart of both rows.
// The pair's lanes load two of its four words of quarter kq each and swap halves (own_rows), which
// leaves a lane word j with columns 32 j + 8 s + 2 kq (low half, nibble s) and + 1 (high half) of its row:
// operand j is those eight in pairs, and x is staged in that order.
template <>
struct Codes<kCodesMarlin> {
  static constexpr int kRowBytes64 = 32;
  u32x2 w;
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    w = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
  }
  __device__ __forceinline__ void own_rows(uint32_t sel) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint32_t other = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w[j], 0xB1, 0xF, 0xF, true);  // lane ^ 1
      w[j] = __builtin_amdgcn_perm(other, w[j], sel);
    }
  }
  __device__ __forceinline__ f16x8 operand(int c) const {
    const uint32_t v = w[c], v8 = v >> 8;
    const u32x4 u = {(v & 0x000F000Fu) | 0x64006400u, (v & 0x00F000F0u) | 0x54005400u,
                     (v8 & 0x000F000Fu) | 0x64006400u, (v8 & 0x00F000F0u) | 0x54005400u};
    const f16 lo = (f16)1024.f, hi = (f16)64.f;
    const f16x8 m = {lo, lo, hi, hi, lo, lo, hi, hi};
    return __builtin_bit_cast(f16x8, u) - m;
  }
};
// Plain fp16 weights: a group's MFMAs add to the accumulator directly.
template <>
struct Codes<kCodesF16> {
  static constexpr int kRowBytes64 = 128;
  u32x4 w[2];
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
      w[c] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff + 16 * c, soff, 0));
  }
  __device__ __forceinline__ f16x8 operand(int c) const { return __builtin_bit_cast(f16x8, w[c]); }
};
// Sixteen 2-bit fields, element i at bits 2 i.
struct Codes2 {
  static constexpr int kRowBytes64 = 16;
  uint32_t w;
  // Fields 8 c .. 8 c + 7 minus sub: the fields in the low half and, one field on, in the high
  // half, so that a mask yields neighbours as a pair (1024 + q or 64 + q, as unpack_word).
  __device__ __forceinline__ static f16x8 fields(uint32_t w, int c, float sub) {
    const uint32_t h = c == 0 ? w : w >> 16;
    const uint32_t v = (h & 0xFFFFu) | ((c == 0 ? w << 14 : w >> 2) & 0xFFFF0000u);
    const uint32_t v8 = v >> 8;
    const u32x4 u = {(v & 0x00030003u) | 0x64006400u, (v & 0x00300030u) | 0x54005400u,
                     (v8 & 0x00030003u) | 0x64006400u, (v8 & 0x00300030u) | 0x54005400u};
    const f16 lo = (f16)(1024.f + sub), hi = (f16)(64.f + sub);
    const f16x8 m = {lo, lo, hi, hi, lo, lo, hi, hi};
    return __builtin_bit_cast(f16x8, u) - m;
  }
};
template <>
struct Codes<kCodesQ2> : Codes2 {
  __device__ __forceinline__ f16x8 operand(int c) const { return fields(w, c, 0.f); }
};
template <>
struct Codes<kCodesTernary> : Codes2 {
  // Codes 0, 1, 2, 3 stand for 0, 1, -1, 0: the fields become value + 1.
  __device__ __forceinline__ f16x8 operand(int c) const {
    const uint32_t lo = w & 0x55555555u, hi = (w >> 1) & 0x55555555u;
    return fields(((lo & ~hi) << 1) | (~(lo ^ hi) & 0x55555555u), c, 1.f);
  }
};

// Waits until all but the wave's last N loads are done.  (Loads complete in issue order.)
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <int F, int EPI, int MB, int NT>
__global__ void __launch_bounds__(kCThreads, 2) codes_gemm_kernel(T16Args a, int n_mblk, int n_split, int n_tile) {
  constexpr bool kPair = EPI == Q4_EPI_SWIGLU;
  constexpr bool kPlain = F == kCodesF16;
  constexpr bool kBias = F != kCodesTernary && !kPlain;
  constexpr int TOK = 16 * MB;
  constexpr int UPW = kPair ? NT / 2 : NT;  // units per wave
  constexpr bool kMarlin = F == kCodesMarlin;
  constexpr bool kRing = F == kCodesQ8 || kMarlin || kPlain;  // codes requested by the group
  constexpr int RING = (F == kCodesQ8 && MB > 3) || (kPlain && NT > 2) ? 2 : 4;
  __shared__ __align__(16) f16 xs[2][TOK * kCStage];
  // Group sums of four groups (a pair of stages) as bf16 parts (s0, s1, s2, s0, s1, s2, 0, 0).
  __shared__ __align__(16) u32x4 sx[kBias ? 2 : 1][kBias ? TOK * 4 : 1];

  const int per = gridDim.x / 8;  // XCD-contiguous tiles, rows fastest (rows_gemm.hip)
  const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (tile >= n_tile) return;
  const int m0 = (tile % n_mblk) * TOK;
  const int sp = (tile / n_mblk) % n_split;
  const int nblk = tile / (n_mblk * n_split);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, kq = lane >> 4;
  const int unit = (nblk * kCWaves + wave) * UPW;
  const int kbA = sp * a.kb_per_split;
  const int n_st = min(a.KB, kbA + a.kb_per_split) - kbA;  // stages of this split (>= 1)
  const int KG = a.K / 64;
  constexpr int RB = Codes<F>::kRowBytes64;
  constexpr int SB = kBias ? 4 : 2;  // scale bytes of a row per group
  const __amdgpu_buffer_rsrc_t rw =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.w16, (short)0, (int)a.w16_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.sb16, (short)0, (int)a.sb16_bytes, 0x00020000);

  // This lane's codes of tile 0, and the (wave-uniform) first row of tile t: an up tile starts
  // a.N rows after its gate tile.  Tiles past the matrix read the last one and are not stored.
  const int w_rows = kMarlin ? (a.N + 7) & ~7 : a.N;
  const int lrow = go::w_lane_row(l16, w_rows);
  const int wlane = go::w_lane(kMarlin, lrow, kq, KG, RB);
  const uint32_t row_sel = l16 & 1 ? 0x03020706u : 0x05040100u;   // Codes<kCodesMarlin>
  int row0[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
    row0[t] = go::w_row0(unit + t % UPW, a.n_units, w_rows) + (kPair && t >= UPW ? a.N : 0);
  // The row's last stage has one group only if K % 128 == 64: its second one reads that group
  // again, and zeros of x.
  const int s_tail = a.K % kCStage != 0 && kbA + n_st == a.KB ? n_st - 1 : -1;
  const int n_grp = 2 * n_st - (s_tail >= 0 ? 1 : 0);

  // Scales (and biases), and 2-bit codes, are requested for two stages at a time, lane quarter kq
  // taking group kq of the four: 16 (64) contiguous bytes per row and request.  Group by group each
  // request touched 16 cache lines for 4 bytes each, and those requests, not bytes or latency,
  // bound the launch (Q8, 22016 x 4096, 75 rows: 87 us, 59 with constant scales, 68.5 this way).
  uint32_t sv[NT], sn[NT];
  u32x4 cv[kRing ? 1 : NT], cn[kRing ? 1 : NT];
  auto load_pair = [&](int p) {
    if constexpr (kPlain) return;
    const int g = min(4 * p + kq, n_grp - 1);  // past the split: its last group again
    const int so = go::s_lane(kMarlin, lrow, g, KG, SB);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int ch = go::s_soff(kMarlin, row0[t], kbA, KG, SB);
      if (kBias) sn[t] = __builtin_amdgcn_raw_buffer_load_b32(rs, so, ch, 0);
      else sn[t] = __builtin_amdgcn_raw_buffer_load_b16(rs, so, ch, 0);
      if constexpr (!kRing)
        cn[t] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                              rw, (lrow * KG + g) * RB, (row0[t] * KG + 2 * kbA) * RB, 0));
    }
  };
  // Codes of RING groups: a stage ahead, or (Q8's 64-row tiles, for their registers) a group ahead.
  Codes<F> wr[kRing ? RING : 1][kRing ? NT : 1];
  auto load_w = [&](int gi, auto bc) {
    if constexpr (kRing) {
      constexpr int b = decltype(bc)::value;
      const int g = 2 * kbA + min(gi, n_grp - 1);
#pragma unroll
      for (int t = 0; t < NT; ++t) wr[b][t].load(rw, wlane, go::w_soff(kMarlin, row0[t], g, KG, RB));
    }
  };

  // Activations to LDS as in rows_gemm.hip: row r's 16-byte piece p at position p ^ (r % 16).
  const int x_rows = min(a.M_tokens - m0, TOK), x_last = go::x_last(x_rows);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.x + (size_t)m0 * a.ldx), (short)0, x_rows * a.ldx * (int)sizeof(f16), 0x00020000);
  const int xrow = 4 * wave + kq;
  const int xoff = go::x_lane(xrow, l16, a.ldx);
  // MARLIN: a row per request, word s of piece (g, quarter, c) from word 32 g + 16 c + 4 s + quarter.
  int xm[kMarlin ? 4 : 1];
  if constexpr (kMarlin)
#pragma unroll
    for (int n = 0; n < 4; ++n) xm[n] = go::x_marlin_lane(4 * wave + n, lane, a.ldx);
  auto load_x = [&](int s, auto bc) {
    constexpr int b = decltype(bc)::value;
    const int st = kbA + min(s, n_st - 1);
    const bool half = go::x_half_stage(st, a.K);
    if constexpr (!kMarlin) {
#pragma unroll
      for (int i = 0; i < MB; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rx, (lds_void*)(&xs[b][(16 * i + 4 * wave) * kCStage]), 16,
            go::x_voff(xoff, i, x_last, 16 * x_last + xrow < x_rows, half && go::x_lane_hi(xrow, l16)),
            go::x_soff(st, i, x_last, a.ldx), 0, 0);
    } else {
      auto request = [&](auto checked) {
        constexpr bool C = decltype(checked)::value;
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int n = 0; n < 4; ++n) {
            const int r = 4 * wave + n;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rx, (lds_void*)(&xs[b][(16 * i + r) * kCStage]), 4,
                C ? go::x_voff(xm[n], i, x_last, 16 * x_last + r < x_rows, half && go::x_marlin_hi(r, lane)) : xm[n],
                C ? go::x_soff(st, i, x_last, a.ldx) : st * (kCStage * 2) + i * 32 * a.ldx, 0, 0);
          }
      };
      // Four requests per piece: whole tiles and stages skip their selects (1024 rows of 12288 x
      // 4096 179 -> 173 us; the other formats, with one, lost more to the branch).
      if (x_rows == TOK && !half) request(std::false_type{});
      else request(std::true_type{});
    }
  };

  f32x4 acc[NT][MB];
  uint32_t bb[NT];  // fp16 bias of group kq of the pair of stages
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    bb[t] = 0;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[t][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  using B0 = std::integral_constant<int, 0>;
  using B1 = std::integral_constant<int, 1>;
  auto stage = [&](int s, auto bc, auto bn) {
    constexpr int b = decltype(bc)::value;
    if (s == s_tail) {
      for (int i = tid; i < TOK * 8; i += kCThreads) {
        const int r = i >> 3, c = 8 + (i & 7);
        *reinterpret_cast<u32x4*>(&xs[b][r * kCStage + ((c ^ (r & 15)) * 8)]) = u32x4{0, 0, 0, 0};
      }
      __syncthreads();
    }
    load_x(s + 1, bn);
    // The wait at the stage's end counts the loads requested after these: none may move before them.
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kRing && RING == 4) {
      load_w(2 * s + 2, std::integral_constant<int, 2 - 2 * b>{});
      load_w(2 * s + 3, std::integral_constant<int, 3 - 2 * b>{});
    }
    if constexpr (b == 0 && !kPlain) {
      // A pair of stages begins: its scales and codes are there, the next pair's are requested.  Past
      // K the scale is zero, not the last group's again, which may be infinite.
      const uint32_t in_k = 2 * s + kq < n_grp ? ~0u : 0u;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        sv[t] = sn[t] & in_k;
        if constexpr (!kRing) cv[t] = lane_transpose(cn[t]);
        if (kBias) bb[t] = sv[t] >> 16;
      }
      load_pair((s >> 1) + 1);
    }
    u32x2 sc2[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) sc2[t] = kPlain ? u32x2{0, 0} : lane_rows<b>(sv[t]);
    if (kBias) {
      // Sums of the stage's two groups per row, TPP threads each.
      constexpr int TPP = MB == 1 ? 8 : (MB == 2 ? 4 : 2);
      const f16x2 one = {(f16)1.f, (f16)1.f};
      // An opaque copy of the thread index: the addresses below are then formed here, in a few
      // operations, and not kept in registers across the loop (25 of them spilled with Q8's
      // 64-row tiles).
      int tq = tid;
      asm volatile("" : "+v"(tq));
      for (int p = tq / TPP; p < 2 * TOK; p += kCThreads / TPP) {
        const int r = p >> 1, g = p & 1;
        float v = 0.f;
#pragma unroll
        for (int i = 0; i < 8 / TPP; ++i) {
          const int c = 8 * g + (tq % TPP) * (8 / TPP) + i;
          const u32x4 x = *reinterpret_cast<const u32x4*>(&xs[b][r * kCStage + ((c ^ (r & 15)) * 8)]);
#pragma unroll
          for (int e = 0; e < 4; ++e) v = __builtin_amdgcn_fdot2(as_h2(x[e]), one, v, false);
        }
        v += dpp_move<0xB1>(v);                    // lane ^ 1
        if (TPP >= 4) v += dpp_move<0x4E>(v);      // lane ^ 2
        if (TPP >= 8) v += dpp_move<0x141>(v);     // the other quad of eight
        if (tq % TPP == 0) {
          const uint32_t s0 = __builtin_bit_cast(uint32_t, v) & 0xFFFF0000u;
          const float r1 = v - __builtin_bit_cast(float, s0);
          const uint32_t s1 = __builtin_bit_cast(uint32_t, r1) & 0xFFFF0000u;
          const uint32_t s2 = __builtin_bit_cast(uint32_t, r1 - __builtin_bit_cast(float, s1));
          u32x4 w = {(s0 >> 16) | s1, (s2 >> 16) | s0, (s1 >> 16) | (s2 & 0xFFFF0000u), 0u};
          // An infinite sum has no rest, and meets the bias's first part only: its product is infinite
          // as in the 2-bit GEMV (that of Q8 and MARLIN, whose codes carry an offset there, is not).
          // (With a wave-uniform branch 0.8 % of a 64-row launch, 1.5 % with selects alone.)
          if constexpr (F == kCodesQ2) {
            const bool inf = __builtin_amdgcn_classf(v, 0x204);
            if (__builtin_amdgcn_ballot_w64(inf) != 0)
              if (inf) w = u32x4{s0 >> 16, 0u, 0u, 0u};
          }
          sx[(s >> 1) & 1][r * 4 + 2 * b + g] = w;
        }
      }
    }
    const f16* xa = &xs[b][l16 * kCStage];
    auto group = [&](auto gc) {
      constexpr int g = decltype(gc)::value;
      __builtin_amdgcn_sched_barrier(0);
      constexpr int w = kRing ? (2 * b + g) % RING : 0;  // a pair starts at an even stage
      if constexpr (kRing && RING == 2) load_w(2 * s + g + 1, std::integral_constant<int, 1 - g>{});
      f16x8 A[2][MB];
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          A[c][mb] = *reinterpret_cast<const f16x8*>(xa + mb * 16 * kCStage + (((8 * g + 2 * kq + c) ^ l16) * 8));
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        __builtin_amdgcn_sched_barrier(0);
        Codes<F> q;
        if constexpr (kRing) q = wr[w][t];
        else q.w = cv[t][2 * b + g];
        if constexpr (kMarlin) q.own_rows(row_sel);
        const f16x8 q0 = q.operand(0), q1 = q.operand(1);
        if constexpr (kPlain) {
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
            acc[t][mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[0][mb], q0, acc[t][mb], 0, 0, 0);
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
            acc[t][mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[1][mb], q1, acc[t][mb], 0, 0, 0);
          continue;
        }
        const float sc = h2f(u16_as_h((uint16_t)sc2[t][g]));
        f32x4 d[MB];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          d[mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[0][mb], q0, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) d[mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[1][mb], q1, d[mb], 0, 0, 0);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int v = 0; v < 4; ++v) acc[t][mb][v] = __builtin_fmaf(sc, d[mb][v], acc[t][mb][v]);
      }
    };
    group(B0{});
    if (!kPlain || s != s_tail) group(B1{});  // (plain weights may be infinite: not even times zero)
    // The next stage's x (requested first in this one) is in LDS; of the loads after it some may
    // still be under way.
    wait_loads<kPlain ? 2 * NT : kRing || b == 0 ? NT : 0>();
    __syncthreads();
  };
  // The bias term of the pair of stages that holds stage s (after its barrier).
  auto flush = [&](int s) {
    if constexpr (kBias) {
      const u32x4* sp4 = sx[(s >> 1) & 1];
      bf16x8 S[MB];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) S[mb] = __builtin_bit_cast(bf16x8, sp4[(16 * mb + l16) * 4 + kq]);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const float bf = h2f(u16_as_h((uint16_t)bb[t]));
        const uint32_t b0 = __builtin_bit_cast(uint32_t, bf) & 0xFFFF0000u;
        const uint32_t b1 = __builtin_bit_cast(uint32_t, bf - __builtin_bit_cast(float, b0));
        const u32x4 bw = {(b0 >> 16) | b0, (b0 >> 16) | (b1 & 0xFFFF0000u), (b1 >> 16) | (b1 & 0xFFFF0000u), 0u};
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          acc[t][mb] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(S[mb], __builtin_bit_cast(bf16x8, bw), acc[t][mb], 0, 0, 0);
      }
    }
  };

  if (kBias)
    for (int i = tid; i < TOK * 4; i += kCThreads) sx[0][i] = sx[kBias ? 1 : 0][i] = u32x4{0, 0, 0, 0};
  load_x(0, B0{});
  load_pair(0);
  load_w(0, B0{});
  if constexpr (RING == 4) load_w(1, B1{});
  wait_loads<0>();
  __syncthreads();
  for (int s = 0;;) {
    stage(s, B0{}, B1{});
    if (++s >= n_st) break;
    stage(s, B1{}, B0{});
    flush(s);
    if (++s >= n_st) break;
  }
  if (n_st & 1) flush(n_st - 1);

  // Lane: weight row l16 of each tile, tokens 4 kq .. + 3 of each 16.
#pragma unroll
  for (int t = 0; t < (n_split == 1 ? UPW : NT); ++t) {
    const int u = unit + t % UPW, row = go::w_row0(u, a.n_units, w_rows) + l16;
    if (u >= a.n_units || row < u * 16 || row >= a.N) continue;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int tok = m0 + 16 * mb + 4 * kq + v;
        if (tok >= a.M_tokens) continue;
        if (n_split == 1)
          t16g_store<EPI>(a, tok, row, acc[t][mb][v], acc[kPair ? t + UPW : t][mb][v]);
        else
          a.part_ws[((size_t)sp * a.M_tokens + tok) * a.part_cols + row + (kPair && t >= UPW ? a.n_units * 16 : 0)] =
              acc[t][mb][v];
      }
  }
}

// The same over GGUF Q2_K blocks (84 bytes per 256 columns: 16 x (scale | min << 4), 64 bytes of
// codes, d, dmin): y = sum_blocks d (sum_k sc q x) - dmin sum_s m_s (sum_k x), s: 16 columns.  A
// stage is half a block, 32 code bytes per row of which lane quarter kq holds 8 kq .. + 7: column
// 32 j + 8 kq + i of the half sits at bits 2 j of byte 8 kq + i, so k-step j of the MFMA takes the
// columns in order.  sc q (at most 45) comes from a four-entry byte table of multiples of sc by one byte
// permute and enters the MFMA as an exact half; the min term is one bf16 MFMA per half block
// whose A holds the sixteen-column sums in three parts and whose B the integers m.
// Against the GEMV's launches of 4-16 rows (us): 4096 x 11008, 16 rows 25.5 -> 17, 40 rows 53 -> 25.5, 64
// rows 87.5 -> 30; 12288 x 4096, 64 rows 90.5 -> 30, 1000 rows 204 here.  Few rows are bound by the
// latency of the few stages of a split, many by the vector units, as above.
template <int MB, int NT>
__global__ void __launch_bounds__(kCThreads, 2) q2k_gemm_kernel(T16Args a, int n_mblk, int n_split, int n_tile) {
  constexpr int TOK = 16 * MB;
  __shared__ __align__(16) f16 xs[2][TOK * kCStage];
  __shared__ __align__(16) u32x2 sx[2][TOK * 8];  // bf16 parts (s0, s1, s2, 0) of each sub-block's sum

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
  const int unit = (nblk * kCWaves + wave) * NT;
  const int kbA = sp * a.kb_per_split;
  const int n_st = min(a.KB, kbA + a.kb_per_split) - kbA;  // half blocks of this split (>= 1)
  const int NB = a.K / 256;
  const __amdgpu_buffer_rsrc_t rw =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.w16, (short)0, (int)a.w16_bytes, 0x00020000);
  const int wlane = go::q2k_lane(go::w_lane_row(l16, a.N), NB);

  u32x2 cw[2][NT], sw[2][NT];
  uint32_t dw[2][NT];
  auto load_w = [&](int s, auto bc) {
    constexpr int b = decltype(bc)::value;
    const int hb = kbA + min(s, n_st - 1);  // past the split: its last half block again (never used)
    const int h = hb & 1;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int base = go::q2k_soff(go::w_row0(unit + t, a.n_units, a.N), hb, NB);  // wave-uniform
      cw[b][t] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rw, wlane + 8 * kq, base + 16 + 32 * h, 0));
      sw[b][t] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rw, wlane, base + 8 * h, 0));
      dw[b][t] = __builtin_amdgcn_raw_buffer_load_b32(rw, wlane, base + 80, 0);
    }
  };
  const int x_rows = min(a.M_tokens - m0, TOK), x_last = go::x_last(x_rows);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.x + (size_t)m0 * a.ldx), (short)0, x_rows * a.ldx * (int)sizeof(f16), 0x00020000);
  const int xrow = 4 * wave + kq;
  const int xoff = go::x_lane(xrow, l16, a.ldx);
  auto load_x = [&](int s, auto bc) {
    constexpr int b = decltype(bc)::value;
    const int st = kbA + min(s, n_st - 1);
#pragma unroll
    for (int i = 0; i < MB; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void*)(&xs[b][(16 * i + 4 * wave) * kCStage]), 16,
                                               go::x_voff(xoff, i, x_last, 16 * x_last + xrow < x_rows, false),
                                               go::x_soff(st, i, x_last, a.ldx), 0, 0);
  };

  f32x4 acc[NT][MB];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[t][mb] = f32x4{0.f, 0.f, 0.f, 0.f};

  using B0 = std::integral_constant<int, 0>;
  using B1 = std::integral_constant<int, 1>;
  auto stage = [&](int s, auto bc, auto bn) {
    constexpr int b = decltype(bc)::value;
    load_x(s + 1, bn);
    load_w(s + 1, bn);
    {
      const f16x2 one = {(f16)1.f, (f16)1.f};
      int tq = tid;
      asm volatile("" : "+v"(tq));  // addresses formed here (see codes_gemm_kernel)
      for (int p = tq; p < 8 * TOK; p += kCThreads) {
        const int r = p >> 3, g = p & 7;
        float v = 0.f;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const u32x4 x = *reinterpret_cast<const u32x4*>(&xs[b][r * kCStage + (((2 * g + i) ^ (r & 15)) * 8)]);
#pragma unroll
          for (int e = 0; e < 4; ++e) v = __builtin_amdgcn_fdot2(as_h2(x[e]), one, v, false);
        }
        const uint32_t s0 = __builtin_bit_cast(uint32_t, v) & 0xFFFF0000u;
        // (At most 2^13; an infinite sum's rest, a NaN, becomes any number: the sum's products with the
        // mins are infinite, as in the few-row kernel.  A branch as in codes_gemm_kernel cost 2 %.)
        const float r1 = __builtin_fminf(v - __builtin_bit_cast(float, s0), 0x1p20f);
        const uint32_t s1 = __builtin_bit_cast(uint32_t, r1) & 0xFFFF0000u;
        const uint32_t s2 = __builtin_bit_cast(uint32_t, r1 - __builtin_bit_cast(float, s1));
        sx[b][p] = u32x2{(s0 >> 16) | s1, s2 >> 16};
      }
    }
    const f16* xa = &xs[b][l16 * kCStage];
    // Two passes of NT / 2 tiles bound the sums in flight.
    constexpr int NH = NT / 2;
#pragma unroll
    for (int th = 0; th < 2; ++th) {
      f32x4 d[NH][MB];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        __builtin_amdgcn_sched_barrier(0);
        f16x8 A[MB];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          A[mb] = *reinterpret_cast<const f16x8*>(xa + mb * 16 * kCStage + (((4 * j + kq) ^ l16) * 8));
#pragma unroll
        for (int u = 0; u < NH; ++u) {
          const int t = th * NH + u;
          const uint32_t sc = (sw[b][t][j >> 1] >> (16 * (j & 1) + 8 * (kq >> 1))) & 15u;
          const uint32_t lut = sc * 0x03020100u;  // bytes 0, sc, 2 sc, 3 sc
          const f16x2 off = {(f16)1024.f, (f16)1024.f};
          u32x4 o;
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const uint32_t v = __builtin_amdgcn_perm(0u, lut, (cw[b][t][i] >> (2 * j)) & 0x03030303u);
            o[2 * i] = as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, v, 0x04010400u)) - off);
            o[2 * i + 1] = as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, v, 0x04030402u)) - off);
          }
          const f16x8 q = __builtin_bit_cast(f16x8, o);
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
            d[u][mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[mb], q, j == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : d[u][mb], 0,
                                                              0, 0);
        }
      }
#pragma unroll
      for (int u = 0; u < NH; ++u) {
        const float dd = h2f(u16_as_h((uint16_t)dw[b][th * NH + u]));
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            acc[th * NH + u][mb][v] = __builtin_fmaf(dd, d[u][mb][v], acc[th * NH + u][mb][v]);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    // The half block's min term: its sums are all written now; scales stay in buffer b.
    bf16x8 S[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      S[mb] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&sx[b][(16 * mb + l16) * 8 + 2 * kq]));
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      // Sub-blocks 2 kq and 2 kq + 1 of the half: their bytes, mins in the high nibbles.
      const uint32_t by = (kq & 2 ? sw[b][t].y : sw[b][t].x) >> (16 * (kq & 1));
      const uint32_t ma = __builtin_bit_cast(uint32_t, (float)((by >> 4) & 15u)) & 0xFFFF0000u;
      const uint32_t mc = __builtin_bit_cast(uint32_t, (float)((by >> 12) & 15u)) & 0xFFFF0000u;
      const u32x4 bw = {(ma >> 16) | ma, ma >> 16, (mc >> 16) | mc, mc >> 16};
      const float dm = -h2f(u16_as_h((uint16_t)(dw[b][t] >> 16)));
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const f32x4 e = __builtin_amdgcn_mfma_f32_16x16x32_bf16(S[mb], __builtin_bit_cast(bf16x8, bw),
                                                                f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[t][mb][v] = __builtin_fmaf(dm, e[v], acc[t][mb][v]);
      }
    }
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

#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int row = go::w_row0(unit + t, a.n_units, a.N) + l16;
    if (unit + t >= a.n_units || row < (unit + t) * 16 || row >= a.N) continue;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int tok = m0 + 16 * mb + 4 * kq + v;
        if (tok >= a.M_tokens) continue;
        if (n_split == 1) t16g_store<Q4_EPI_STORE>(a, tok, row, acc[t][mb][v], 0.f);
        else a.part_ws[((size_t)sp * a.M_tokens + tok) * a.part_cols + row] = acc[t][mb][v];
      }
  }
}

struct CodesPlan {
  int mb, nt, splits;
};
// Row tile: the fewest row blocks of up to 64 rows, evenly filled.  Weight tiles per wave (two, or
// four with 64 rows; 48 rows with four were always slower) and K splits by the time each choice is
// expected to take: a round of the workgroups that fit a CU (four of up to 32 rows, three with two
// tiles per wave, two with four) (or part of one past the first) costs kStage[0] us per stage,
// each workgroup of a CU kStage[1]; partial tiles are written and read back at about 5 TB/s.
// Fitted to a sweep of 1-16 splits and both tile counts over 8-1000 rows, six matrices (1024-22016
// rows) and five formats: the choice is within 1-2 % of the sweep's best on average and 14 % at
// worst but for one (27 %), four tiles per wave with two workgroups a CU had been 15-35 % off on
// average (Q8 4096 x 4096, 40 rows: four tiles 20.3 us, two from eight splits 15.1; 12288 x 4096,
// 75 rows 41.0 / 34.7; 1000 rows: four tiles unsplit 155, two 167).
CodesPlan codes_plan(int M, int KB, int n_units, int epi) {
  static const float kStage[5][2] = {{.18f, .41f}, {.26f, .51f}, {.38f, .51f}, {.53f, .54f},  // 16-64 rows, two tiles
                                     {1.f, .9f}};                                             // 64, four
  const int nb = axm_ceil_div(M, 64), mb = axm_ceil_div(M, 16 * nb), cus = axm_num_cus();
  const float part_us = 1.5e-6f * (float)M * (float)n_units * (epi == Q4_EPI_SWIGLU ? 32.f : 16.f);
  CodesPlan best{mb, 2, 1};
  float best_us = 1e30f;
  for (int nt = 2; nt <= (mb == 4 ? 4 : 2); nt += 2) {
    const float* st = kStage[nt == 2 ? mb - 1 : 4];
    const int per_cu = mb <= 2 ? 4 : nt == 2 ? 3 : 2;
    const int tiles = axm_ceil_div(n_units, kCWaves * (epi == Q4_EPI_SWIGLU ? nt / 2 : nt)) * axm_ceil_div(M, 16 * mb);
    for (int s = 1; s <= 16 && (s == 1 || s <= KB / 2); ++s) {
      const int stages = axm_ceil_div(KB, s), splits = axm_ceil_div(KB, stages);
      const int load = axm_ceil_div(tiles * splits, cus);  // workgroups per CU
      const float rounds = load > per_cu ? (float)load / (float)per_cu : 1.f;
      const float us = (float)stages * (st[0] * rounds + st[1] * (float)load) +
                       (splits == 1 ? 0.f : 1.3f + (float)splits * part_us);
      if (us < best_us) best_us = us, best = {mb, nt, splits};
    }
  }
  return best;
}

template <int F, int EPI, int MB, int NT>
void codes_launch(const T16Args& a, int M, int splits, hipStream_t s) {
  constexpr int kUnits = kCWaves * (EPI == Q4_EPI_SWIGLU ? NT / 2 : NT);
  const int n_mblk = axm_ceil_div(M, 16 * MB);
  const int n_tile = n_mblk * splits * axm_ceil_div(a.n_units, kUnits);
  hipLaunchKernelGGL((codes_gemm_kernel<F, EPI, MB, NT>), dim3(8 * axm_ceil_div(n_tile, 8)), dim3(kCThreads), 0, s, a,
                     n_mblk, splits, n_tile);
}
template <int MB, int NT>
void q2k_launch(const T16Args& a, int M, int splits, hipStream_t s) {
  const int n_mblk = axm_ceil_div(M, 16 * MB);
  const int n_tile = n_mblk * splits * axm_ceil_div(a.n_units, kCWaves * NT);
  hipLaunchKernelGGL((q2k_gemm_kernel<MB, NT>), dim3(8 * axm_ceil_div(n_tile, 8)), dim3(kCThreads), 0, s, a, n_mblk,
                     splits, n_tile);
}
void q2k_launch_shape(const T16Args& a, int M, const CodesPlan& p, hipStream_t s) {
  switch (p.mb) {
    case 1: return q2k_launch<1, 2>(a, M, p.splits, s);
    case 2: return q2k_launch<2, 2>(a, M, p.splits, s);
    case 3: return q2k_launch<3, 2>(a, M, p.splits, s);
    default: return p.nt == 2 ? q2k_launch<4, 2>(a, M, p.splits, s) : q2k_launch<4, 4>(a, M, p.splits, s);
  }
}

template <int F, int EPI>
void codes_launch_shape(const T16Args& a, int M, const CodesPlan& p, hipStream_t s) {
  switch (p.mb) {
    case 1: return codes_launch<F, EPI, 1, 2>(a, M, p.splits, s);
    case 2: return codes_launch<F, EPI, 2, 2>(a, M, p.splits, s);
    case 3: return codes_launch<F, EPI, 3, 2>(a, M, p.splits, s);
    default: return p.nt == 2 ? codes_launch<F, EPI, 4, 2>(a, M, p.splits, s) : codes_launch<F, EPI, 4, 4>(a, M, p.splits, s);
  }
}

template <int F>
void codes_launch_epi(const T16Args& a, int M, int epi, const CodesPlan& p, hipStream_t s) {
  if (epi == Q4_EPI_STORE) codes_launch_shape<F, Q4_EPI_STORE>(a, M, p, s);
  else if (epi == Q4_EPI_RESID) codes_launch_shape<F, Q4_EPI_RESID>(a, M, p, s);
  else codes_launch_shape<F, Q4_EPI_SWIGLU>(a, M, p, s);
}

}  // namespace

// Code / scale bytes of a matrix.
static size_t codes_bytes(int fmt, int rows, int K) {
  if (fmt == kCodesMarlin) return (size_t)((rows + 7) / 8) * (K / 64) * 256;
  return (size_t)rows * (fmt == kCodesF16 ? 2 * K : fmt == kCodesQ2kGguf ? K / 256 * 84 : fmt == kCodesQ8 ? K : K / 4);
}
static size_t scale_bytes(int fmt, int rows, int K) {
  const size_t r = fmt == kCodesMarlin ? (size_t)(rows + 7) / 8 * 8 : rows;
  return r * (K / 64) * (fmt == kCodesTernary ? 2 : 4);
}

bool codes_gemm_takes(const void* x, const void* w, const void* sb, int K, int rows, int fmt) {
  if (fmt == kCodesQ2kGguf)
    return K > 0 && K % 256 == 0 && K <= 16384 && (size_t)rows * (K / 256) * 84 < (size_t)0x7FFFFFF0 &&
           ((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 3) == 0;
  const size_t code_bytes = codes_bytes(fmt, rows, K);
  const uintptr_t wa = fmt == kCodesQ8 || fmt == kCodesF16 ? 15 : fmt == kCodesMarlin ? 7 : 3, sa = fmt == kCodesTernary ? 1 : 3;
  return K > 0 && K % 64 == 0 && K <= 32768 && code_bytes < (size_t)0x7FFFFFF0 && ((uintptr_t)x & 15) == 0 &&
         ((uintptr_t)w & wa) == 0 && ((uintptr_t)sb & sa) == 0;
}

size_t codes_gemm_ws_bytes(int M, int K, int N, int epi) {
  const int n_units = (N + 15) / 16;
  const int splits = codes_plan(M, (K + 127) / 128, n_units, epi).splits;
  return splits <= 1 ? 0 : (size_t)splits * M * n_units * (epi == Q4_EPI_SWIGLU ? 32 : 16) * sizeof(float);
}

int codes_gemm_launch(int fmt, T16Args a, int M, int epi, float* ws, size_t ws_bytes, hipStream_t s) {
  const int rows = epi == Q4_EPI_SWIGLU ? 2 * a.N : a.N;
  if (M < 1 || !codes_gemm_takes(a.x, a.w16, a.sb16, a.K, rows, fmt) || a.ldx % 8 != 0 || a.ln_w != nullptr ||
      (epi != Q4_EPI_STORE && epi != Q4_EPI_RESID && epi != Q4_EPI_SWIGLU) ||
      (fmt != kCodesQ8 && fmt != kCodesF16 && epi != Q4_EPI_STORE) ||
      (a.post_ln_w != nullptr && (epi != Q4_EPI_RESID || a.post_norm_out == nullptr || a.ldr != a.N))) {
    axm_set_error("codes gemm: format %d, M=%d, epi=%d, K=%d unsupported", fmt, M, epi, a.K);
    return -2;
  }
  a.KB = (a.K + 127) / 128;
  a.n_units = (a.N + 15) / 16;
  a.M_tokens = M;
  a.part_ws = ws;
  a.part_cols = a.n_units * (epi == Q4_EPI_SWIGLU ? 32 : 16);
  a.pair_offset = a.n_units;  // of the partial tiles' columns
  CodesPlan p = codes_plan(M, a.KB, a.n_units, epi);
  const size_t one = (size_t)M * a.part_cols * sizeof(float);
  if (ws == nullptr || ws_bytes < 2 * one) p.splits = 1;
  else if (ws_bytes < p.splits * one) p.splits = (int)(ws_bytes / one);
  a.kb_per_split = axm_ceil_div(a.KB, p.splits);
  p.splits = axm_ceil_div(a.KB, a.kb_per_split);
  a.w16_bytes = codes_bytes(fmt, rows, a.K);
  a.sb16_bytes = scale_bytes(fmt, rows, a.K);
  if (fmt == kCodesQ2kGguf) q2k_launch_shape(a, M, p, s);
  else if (fmt == kCodesQ2) codes_launch_shape<kCodesQ2, Q4_EPI_STORE>(a, M, p, s);
  else if (fmt == kCodesMarlin) codes_launch_shape<kCodesMarlin, Q4_EPI_STORE>(a, M, p, s);
  else if (fmt == kCodesTernary) codes_launch_shape<kCodesTernary, Q4_EPI_STORE>(a, M, p, s);
  else if (fmt == kCodesF16) codes_launch_epi<kCodesF16>(a, M, epi, p, s);
  else codes_launch_epi<kCodesQ8>(a, M, epi, p, s);
  return t16_gemm_finish(a, M, epi, p.splits, M, true, s);
}

// ---------------------------------------------------------------------------
// C ABI: products of several rows with a workspace for split K.
// ---------------------------------------------------------------------------
// The 2-bit GEMVs' own matrix-core launches take up to 16 rows each (fewer at large K, whose rows
// fill LDS); this kernel takes over where they need four, and for a large matrix (32 Mi weights)
// where they need two, or one of ternary or affine codes with more than eight rows and a K that
// splits well (us, ternary, 12288 x 4096: eight rows in one launch 13.3, ten 20.6 against 15.8 here,
// sixteen 23.2 / 16.4, 17 in two 28.7 / 17.7, 64 in four 90.7 / 25.7; 32000 x 2048 affine: ten 17.8 / 18.7;
// 4096 x 4096: 32 in two 13.6 / 14, 40 in three 19.1 / 13.2, 64 in four 26.4 / 16.2;
// 4096 x 11008: six in one 11.5 / 14.4, eight in two 20.2 / 14.9; GGUF 4096 x 11008: eight in two
// 16.2 / 16.5, twelve 17.8 / 16.9, sixteen in three 25.5 / 17, 64 in ten 87.5 / 30; 4096 x 4096: 48 in
// three 19.3 / 16.4).
static bool lowbit_rows_use_codes(int fmt, int M, int K, int N) {
  const bool gguf = fmt == kCodesQ2kGguf;
  const int per = gguf ? q2k_gguf_mfma_rows(K) : lowbit_mfma_rows(N, K);
  const int launches = per > 0 ? axm_ceil_div(M, per) : M;
  if (launches >= 3) return true;
  if ((size_t)N * K < (size_t)32 << 20) return false;
  return gguf ? launches >= 2 && M >= 12 : launches >= 2 || (M > 8 && K >= 4096);
}

// Whether M rows of a format go through this kernel (shapes and alignment apart).  Q8 products of five or six
// rows and few weight rows stay with the GEMV's two launches where K is too short to pay for split K and
// its reduction (us, GEMV / here, 1000 weight rows: K = 256 five rows 6.3 / 4.9; 512 6.2 / 6.4; 1024 five 6.4 / 7.0,
// six 6.7 / 7.1, seven 7.0 / 7.0; 2048 five 7.0 / 7.4, six 7.5 / 7.4; 4096 five 9.0 / 8.2; 2048 weight rows: never).
static bool rows_use_codes(int fmt, int M, int K, int N) {
  if (fmt == kCodesMarlin) return marlin_rows_use_codes(M, K, N);
  if (fmt == kCodesQ8) return M >= 7 || (M >= kCodesQ8MinRows && (N > 1024 || K < 512 || K > 2048));
  return M > 4 && lowbit_rows_use_codes(fmt, M, K, N);
}

extern "C" size_t axm_qmm_codes_workspace_bytes(int format, int M, int K, int N) {
  if (format < kCodesQ8 || format > kCodesMarlin || M <= 0 || K <= 0 || N <= 0) return 0;
  return rows_use_codes(format, M, K, N) ? codes_gemm_ws_bytes(M, K, N, Q4_EPI_STORE) : 0;
}

static int qmm_codes(int fmt, const char* who, const void* x, const void* w, const void* sb, const void* bias, void* y,
                     int M, int K, int N, void* ws, size_t ws_bytes, hipStream_t s) {
  T16Args a{};
  a.x = (const f16*)x;
  a.ldx = K;
  a.w16 = (const u32x4*)w;
  a.sb16 = (const u32x2*)sb;
  a.K = K;
  a.N = N;
  a.y = (f16*)y;
  a.ldy = N;
  a.bias = (const f16*)bias;
  a.bias_f32 = fmt != kCodesQ8 && fmt != kCodesMarlin;  // as the formats' GEMVs
  const int rc = codes_gemm_launch(fmt, a, M, Q4_EPI_STORE, (float*)ws, ws_bytes, s);
  if (rc) return rc;
  AXM_LAUNCH_CHECK(who);
  return 0;
}

extern "C" int axm_qmm_q8_g64(const void* x, const void* w_packed, const void* sb, const void* bias, void* y, int M,
                              int K, int N, void* workspace, size_t workspace_bytes, void* stream) {
  if (!rows_use_codes(kCodesQ8, M, K, N) || !codes_gemm_takes(x, w_packed, sb, K, N, kCodesQ8))
    return axm_qmv_q8_g64(x, w_packed, sb, bias, y, M, K, N, stream);
  AXM_CHECK_ARG(w_packed && sb && x && y && N > 0, -1, "qmm_q8_g64: bad arguments");
  return qmm_codes(kCodesQ8, "qmm_q8_g64", x, w_packed, sb, bias, y, M, K, N, workspace, workspace_bytes,
                   (hipStream_t)stream);
}

extern "C" int axm_qmm_q4_marlin(const void* x, const void* w_marlin, const void* sb_marlin, const void* bias, void* y,
                                 int M, int K, int N, void* workspace, size_t workspace_bytes, void* stream) {
  if (N <= 0 || !rows_use_codes(kCodesMarlin, M, K, N) || !codes_gemm_takes(x, w_marlin, sb_marlin, K, N, kCodesMarlin))
    return axm_qmv_q4_marlin(x, w_marlin, sb_marlin, bias, y, M, K, N, stream);
  AXM_CHECK_ARG(w_marlin && sb_marlin && x && y, -1, "qmm_q4_marlin: bad arguments");
  return qmm_codes(kCodesMarlin, "qmm_q4_marlin", x, w_marlin, sb_marlin, bias, y, M, K, N, workspace, workspace_bytes,
                   (hipStream_t)stream);
}

extern "C" int axm_qmm_ternary(const void* x, const void* w_packed, const void* scales, const void* bias, void* y,
                               int M, int K, int N, void* workspace, size_t workspace_bytes, void* stream) {
  if (!rows_use_codes(kCodesTernary, M, K, N) || !codes_gemm_takes(x, w_packed, scales, K, N, kCodesTernary))
    return axm_qmv_ternary(x, w_packed, scales, bias, y, M, K, N, stream);
  AXM_CHECK_ARG(x && w_packed && scales && y && N > 0, -1, "qmm_ternary: bad arguments");
  return qmm_codes(kCodesTernary, "qmm_ternary", x, w_packed, scales, bias, y, M, K, N, workspace, workspace_bytes,
                   (hipStream_t)stream);
}

extern "C" int axm_qmm_q2_k(const void* x, const void* w_packed, const void* scales_biases, const void* bias, void* y,
                            int M, int K, int N, void* workspace, size_t workspace_bytes, void* stream) {
  if (!rows_use_codes(kCodesQ2, M, K, N) || !codes_gemm_takes(x, w_packed, scales_biases, K, N, kCodesQ2))
    return axm_qmv_q2_k(x, w_packed, scales_biases, bias, y, M, K, N, stream);
  AXM_CHECK_ARG(x && w_packed && scales_biases && y && N > 0, -1, "qmm_q2_k: bad arguments");
  return qmm_codes(kCodesQ2, "qmm_q2_k", x, w_packed, scales_biases, bias, y, M, K, N, workspace, workspace_bytes,
                   (hipStream_t)stream);
}

extern "C" int axm_qmm_q2_k_gguf(const void* x, const void* blocks, const void* bias, void* y, int M, int K, int N,
                                 void* workspace, size_t workspace_bytes, void* stream) {
  if (K <= 0 || !rows_use_codes(kCodesQ2kGguf, M, K, N) || !codes_gemm_takes(x, blocks, nullptr, K, N, kCodesQ2kGguf))
    return axm_qmv_q2_k_gguf(x, blocks, bias, y, M, K, N, stream);
  AXM_CHECK_ARG(x && blocks && y && N > 0, -1, "qmm_q2_k_gguf: bad arguments");
  return qmm_codes(kCodesQ2kGguf, "qmm_q2_k_gguf", x, blocks, nullptr, bias, y, M, K, N, workspace, workspace_bytes,
                   (hipStream_t)stream);
}
