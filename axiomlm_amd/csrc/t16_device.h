// Device helpers shared by the tile16 GEMV kernels (stand-alone launches and
// the persistent decode-step kernel).
#pragma once
#include "axm_common.h"
#include "q4_tile16.h"

// Nibble expansion: (w & mask) | magic as one v_and_or_b32.  gfx950 VOP3 takes
// neither literals nor two scalar operands, so the masks must sit in VGPRs and
// the magic exponents in SGPRs for instruction selection to fuse the pair.
// The masks are moved into VGPRs once, through an opaque move the compiler
// cannot fold back into a constant; the AND-OR itself stays compiler-generated
// so the MFMA hazard recognizer sees every VALU write that feeds a B operand
// (a VALU write read by an MFMA source needs two wait states, and the
// recognizer does not model inline-asm producers).
struct Unpack {
  uint32_t m_lo, m_hi, g_lo, g_hi;  // 0x000F000F, 0x00F000F0, 0x64006400, 0x54005400
};

__device__ __forceinline__ uint32_t to_vgpr(uint32_t s) {
  uint32_t v;
  asm volatile("v_mov_b32 %0, %1" : "=v"(v) : "s"(s));
  return v;
}

// A VGPR copy the compiler cannot see through (keeps a loaded uniform value out of
// SGPRs until here, so the wait for it lands here).
__device__ __forceinline__ uint32_t t16_vgpr(uint32_t v) {
  uint32_t r;
  asm volatile("v_mov_b32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}

// A value the compiler cannot fold into a literal operand, kept in an SGPR.
__device__ __forceinline__ uint32_t to_sgpr(uint32_t s) {
  uint32_t v;
  asm volatile("s_mov_b32 %0, %1" : "=s"(v) : "s"(s));
  return v;
}

__device__ __forceinline__ uint32_t and_or(uint32_t w, uint32_t mask_v, uint32_t magic_s) {
  return (w & mask_v) | magic_s;
}

__device__ __forceinline__ f16x8 unpack_word(uint32_t w, const Unpack& u) {
  const uint32_t w8 = w >> 8;
  const u32x4 h = {and_or(w, u.m_lo, u.g_lo), and_or(w, u.m_hi, u.g_hi), and_or(w8, u.m_lo, u.g_lo),
                   and_or(w8, u.m_hi, u.g_hi)};
  return __builtin_bit_cast(f16x8, h);
}

__device__ __forceinline__ float t16_silu(float g) { return g / (1.0f + expf(-g)); }

// One output element of the epilogue (identical arithmetic to the GEMV's):
// v0 the gate / plain accumulator, v1 the up accumulator (SwiGLU).
template <int EPI>
__device__ __forceinline__ void t16g_store(const T16Args& a, int tok, int row, float v0, float v1) {
  if (EPI == Q4_EPI_SWIGLU) {
    const f16 g = f2h(v0);
    const f16 u = f2h(v1);
    const f16 sg = f2h(t16_silu(h2f(g)));
    a.y[(size_t)tok * a.ldy + row] = f2h(h2f(sg) * h2f(u));
  } else {
    if (a.bias_f32 && a.bias != nullptr) v0 += h2f(a.bias[row]);
    f16 h = f2h(v0);
    if (!a.bias_f32 && a.bias != nullptr) h = f2h(h2f(h) + h2f(a.bias[row]));
    if (EPI == Q4_EPI_STORE) {
      a.y[(size_t)tok * a.ldy + row] = h;
    } else {
      f16* xr = a.resid + (size_t)tok * a.ldr + row;
      *xr = f2h(h2f(*xr) + h2f(h));
    }
  }
}

// The same for four consecutive output rows of one token (the accumulators of a lane when
// the weights are the MFMA's row operand): one 8-byte access each of the residual / output
// row and the bias where t16g_vec4 allows it, else element by element up to row N.
template <int EPI>
__device__ __forceinline__ void t16g_store4(const T16Args& a, int tok, int row, f32x4 v0, f32x4 v1, bool vec) {
  if (!vec) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (row + e < a.N) t16g_store<EPI>(a, tok, row + e, v0[e], v1[e]);
    return;
  }
  f16x4 h;
  if (EPI == Q4_EPI_SWIGLU) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const f16 g = f2h(v0[e]);
      const f16 u = f2h(v1[e]);
      h[e] = f2h(h2f(f2h(t16_silu(h2f(g)))) * h2f(u));
    }
  } else {
    f16x4 b = {};
    if (a.bias != nullptr) b = *reinterpret_cast<const f16x4*>(a.bias + row);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (a.bias_f32) v0[e] += h2f(b[e]);
      h[e] = f2h(v0[e]);
      if (!a.bias_f32 && a.bias != nullptr) h[e] = f2h(h2f(h[e]) + h2f(b[e]));
    }
  }
  if (EPI == Q4_EPI_RESID) {
    f16x4* xr = reinterpret_cast<f16x4*>(a.resid + (size_t)tok * a.ldr + row);
    f16x4 x = *xr;
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = f2h(h2f(x[e]) + h2f(h[e]));
    *xr = x;
  } else {
    *reinterpret_cast<f16x4*>(a.y + (size_t)tok * a.ldy + row) = h;
  }
}
// Whether every 4-row access of t16g_store4 is whole and 8-byte aligned.
template <int EPI>
__device__ __forceinline__ bool t16g_vec4(const T16Args& a) {
  const int ld = EPI == Q4_EPI_RESID ? a.ldr : a.ldy;
  const uintptr_t p = EPI == Q4_EPI_RESID ? (uintptr_t)a.resid : (uintptr_t)a.y;
  return a.N % 4 == 0 && ld % 4 == 0 && ((p | (uintptr_t)a.bias) & 7) == 0;
}
