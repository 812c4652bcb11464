// Device pieces of a register radix-16 FFT stage, shared by the vector passes
// (fft.hip) and the low layers of the matrix passes (fft_matrix.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "field.hpp"

namespace stwo_hip {

// `t2` is the twiddle doubled (the passes read the doubled trees).
template <bool INV>
__device__ __forceinline__ void bfly(uint32_t &a, uint32_t &b, uint32_t t2) {
  if (INV) {
    uint32_t s = m31_add(a, b);
    b = m31_mul_dbl(m31_sub(a, b), t2);
    a = s;
  } else {
    uint32_t tmp = m31_mul_dbl(b, t2);
    b = m31_sub(a, tmp);
    a = m31_add(a, tmp);
  }
}

// Twiddles of one stage: for register bit r, 8 >> r consecutive words of
// tree level s = sh + r starting at gb >> (s + 1); the circle layer (s = 0)
// is expanded from two (x, y) pairs of line layer 0 into [y, -y, -x, x].
struct StageTw {
  uint32_t t0[8], t1[4], t2[2], t3[1];
};

// Word `byte_off / 4` of a table whose base is wave-uniform: the base stays
// in SGPRs and the lane part is a 32-bit offset (global_load ... saddr).
__device__ __forceinline__ uint32_t gld(const uint32_t *base, uint32_t byte_off) {
  return *(gconst_u32 *)((gconst_u8 *)as_global(base) + byte_off);
}
__device__ __forceinline__ void gst(uint32_t *base, uint32_t byte_off, uint32_t v) {
  *(g_u32 *)((g_u8 *)as_global(base) + byte_off) = v;
}
__device__ __forceinline__ u32x4 gld4(const uint32_t *base, uint32_t byte_off) {
  return *(gconst_u4 *)((gconst_u8 *)as_global(base) + byte_off);
}
__device__ __forceinline__ void gst4(uint32_t *base, uint32_t byte_off, u32x4 v) {
  *(g_u4 *)((g_u8 *)as_global(base) + byte_off) = v;
}
// The same for words that the launch touches once.
__device__ __forceinline__ u32x4 gld4_once(const uint32_t *base, uint32_t byte_off) {
  return __builtin_nontemporal_load((gconst_u4 *)((gconst_u8 *)as_global(base) + byte_off));
}
__device__ __forceinline__ void gst4_once(uint32_t *base, uint32_t byte_off, u32x4 v) {
  __builtin_nontemporal_store(v, (g_u4 *)((g_u8 *)as_global(base) + byte_off));
}

__device__ __forceinline__ void load_level(uint32_t *dst, int cnt, const uint32_t *tw_end, uint32_t N, uint32_t s,
                                           uint32_t gb) {
  const uint32_t hs = gb >> (s + 1);
  if (s == 0) {
    const uint32_t *l0 = tw_end - ((size_t)1 << (N - 1));
    const uint32_t o = (hs >> 1) << 2;
    uint32_t w4[4];
#pragma unroll
    for (int k = 0; k < 4; k++) w4[k] = gld(l0, o + 4 * k);
#pragma unroll
    for (int u = 0; u < 8; u++) {
      uint32_t xx = w4[2 * (u >> 2)], yy = w4[2 * (u >> 2) + 1];
      uint32_t v = (u & 2) ? xx : yy;
      // doubled negation: 2 (P - v / 2) = 2P - v < 2^32 (for v = 0 it is 2P, still 0 mod P)
      dst[u] = ((u & 3) == 1 || (u & 3) == 2) ? 2u * P - v : v;
    }
    return;
  }
  const uint32_t *lv = tw_end - ((size_t)1 << (N - s));
  const uint32_t o = hs << 2;
#pragma unroll
  for (int u = 0; u < 8; u++)
    if (u < cnt) dst[u] = gld(lv, o + 4 * u);
}

// Loads only the levels of the stage's active register bits [r_lo, r_hi).
__device__ __forceinline__ void load_stage_twiddles(StageTw &t, const uint32_t *tw_end, uint32_t N, uint32_t sh,
                                                    uint32_t gb, uint32_t r_lo, uint32_t r_hi) {
  if (r_lo <= 0 && 0 < r_hi) load_level(t.t0, 8, tw_end, N, sh + 0, gb);
  if (r_lo <= 1 && 1 < r_hi) load_level(t.t1, 4, tw_end, N, sh + 1, gb);
  if (r_lo <= 2 && 2 < r_hi) load_level(t.t2, 2, tw_end, N, sh + 2, gb);
  if (r_lo <= 3 && 3 < r_hi) load_level(t.t3, 1, tw_end, N, sh + 3, gb);
}

template <int R>
__device__ __forceinline__ uint32_t stage_tw(const StageTw &t, int u) {
  return R == 0 ? t.t0[u] : R == 1 ? t.t1[u] : R == 2 ? t.t2[u] : t.t3[u];
}

// Layers at register bits [RLO, RHI) of the group (forward: high to low).
template <bool INV, int RLO, int RHI>
__device__ __forceinline__ void stage_layers(uint32_t (&x)[16], const StageTw &t) {
#pragma unroll
  for (int rr = 0; rr < RHI - RLO; rr++) {
    const int r = INV ? RLO + rr : RHI - 1 - rr;
#pragma unroll
    for (int j0 = 0; j0 < 16; j0++)
      if (!((j0 >> r) & 1)) {
        const int u = j0 >> (r + 1);
        const uint32_t tw = r == 0 ? stage_tw<0>(t, u) : r == 1 ? stage_tw<1>(t, u) : r == 2 ? stage_tw<2>(t, u)
                                                                                           : stage_tw<3>(t, u);
        bfly<INV>(x[j0], x[j0 | (1 << r)], tw);
      }
  }
}

}  // namespace stwo_hip
