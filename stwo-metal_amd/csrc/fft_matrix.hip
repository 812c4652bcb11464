// Circle FFT passes whose butterflies run on the matrix cores.
//
// Four consecutive layers s .. s+3 (s >= 4) of a column act on 16 elements
// that differ in index bits [s, s+4) as one 16 x 16 matrix over the field; the
// matrix depends only on the index bits above, so every position below (and
// every column) shares it.  v_mfma_i32_16x16x64_i8 contracts 64 signed bytes:
// exactly 16 elements of 4 bytes.  So
//   y_j = sum_i M[j][i] x_i,  x_i = sum_l 256^l byte_l(x_i)
//       = sum_{i,l} (M[j][i] 256^l mod P) byte_l(x_i)
// and the constants (M[j][i] 256^l mod P) are split into 4 signed bytes of
// weight 1, 2^8, 2^15 and 2^23, one operand per byte m: four MFMAs give a_m =
// sum (byte m of the constant) * byte, |a_m| <= 64 * 128 * 128 = 2^20, and
// y = a_0 + 2^8 a_1 + 2^15 (a_2 + 2^8 a_3) exactly.  (2^15: then 2^15 d splits
// into d's 16-bit halves, d >> 16 and (d & 0xffff) 2^15, which one instruction
// each adds up.)  The element words are the operand as they lie in
// registers (their bytes, made signed by x ^ 0x80808080), the accumulator
// layout equals the operand layout (lane g * 16 + n, register q: element
// 4 g + q of vector n), so a stage is in place and two lane bits and two
// register bits carry the 16 elements.
//
// Cost per 64 words and 4 layers: one MFMA (16 cycles, 8 of them blocking
// issue) and 5 VALU instructions, about 29 cycles by a register-only loop,
// against 22 VALU instructions (95 cycles) of four butterfly layers.
#include <algorithm>
#include <vector>

#include "common.hpp"
#include "fft_dev.hpp"
#include "field.hpp"
#include "fft_matrix.hpp"
#include "internal.hpp"

namespace stwo_hip {

typedef int i32x4 __attribute__((ext_vector_type(4)));

namespace {

// The four operands of one stage (byte m of every constant) and the
// accumulators' start values.
struct MxMat {
  i32x4 a[4];
  i32x4 c0, c2;
};

// Accumulators: c = a_0 + 256 a_1 and d = a_2 + 256 a_3 are at most 2^28 +
// 2^20 in magnitude, so kMxOff keeps both positive; y = c + 2^15 d.  The start
// values carry the offsets' negation mod P and the correction for the signed
// bytes: sum_i M[j][i] * 0x80808080.
constexpr uint32_t kMxOff = (1u << 28) + (1u << 21);
constexpr uint32_t kMxOffSum = (uint32_t)(((uint64_t)kMxOff * 32769u) % P);
constexpr uint32_t kMxSign = 0x80808080u;
constexpr uint32_t kMxSignP = kMxSign - P;

__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) {
  return __builtin_amdgcn_perm(hi, lo, sel);
}

// The matrix of the low `layers` (1..4) of the four layers whose lowest is
// line layer N - D of a domain of log size N, for the block of index h (the
// element index's bits above the four): with e the index on the evaluation
// side, c on the coefficient side,
//   forward  M[e][c] = prod_{r < layers, c_r = 1} (e_r ? -t_r : t_r),
//   inverse  M[c][e] likewise with inverse twiddles (the transposed network),
// t_r = tree level D - r at (h << (3 - r)) | (e >> (r + 1)); bits r >= layers
// pass through (M = 0 where e_r != c_r).  `tw_end`: the end of the plain tree
// (inverse tree when INV).  Every lane of the wave takes part.
//
// v_0 .. v_3: a lane's four constants, M[row][4 g + q].  Four products each
// way: the factors of bits 3 and 2 (inverse: 1 too) do not depend on q but for
// their sign.
template <bool INV>
__device__ __forceinline__ void mx_consts(const uint32_t *tw_end, uint32_t D, uint32_t h, uint32_t layers,
                                          uint32_t scale, uint32_t v[4]) {
  const uint32_t lane = threadIdx.x & 63, row = lane & 15, g = lane >> 4;
  auto tw = [&](uint32_t r, uint32_t k) {  // t_r at (h << (3 - r)) | k
    return gld(tw_end - ((size_t)1 << (D - r)), ((h << (3 - r)) | k) << 2);
  };
  // factor of bit r: (e_r ? -t : t) where c_r, else 1; pass-through bits: 1 or 0
  auto fac = [&](uint32_t r, uint32_t t, bool er, bool cr) {
    const uint32_t s = er ? P - t : t;
    return r < layers ? (cr ? s : 1u) : (er == cr ? 1u : 0u);
  };
  if (!INV) {
    const uint32_t t3 = tw(3, 0), t2 = tw(2, row >> 3), t1 = tw(1, row >> 2), t0 = tw(0, row >> 1);
    const bool e0 = row & 1, e1 = row & 2, e2 = row & 4, e3 = row & 8;
    const uint32_t base = m31_mul(m31_mul(fac(3, t3, e3, g & 2), fac(2, t2, e2, g & 1)), scale);
    const uint32_t a = m31_mul(base, fac(1, t1, e1, false)), b = m31_mul(base, fac(1, t1, e1, true));
    const uint32_t f0 = fac(0, t0, e0, false), f1 = fac(0, t0, e0, true);
    v[0] = m31_mul(a, f0);
    v[1] = m31_mul(a, f1);
    v[2] = m31_mul(b, f0);
    v[3] = m31_mul(b, f1);
  } else {
    const uint32_t t3 = tw(3, 0), t2 = tw(2, g >> 1), t1 = tw(1, g), t0a = tw(0, 2 * g), t0b = tw(0, 2 * g + 1);
    const bool c0 = row & 1, c1 = row & 2, c2 = row & 4, c3 = row & 8;
    const uint32_t base = m31_mul(m31_mul(fac(3, t3, g & 2, c3), fac(2, t2, g & 1, c2)), scale);
    const uint32_t a = m31_mul(base, fac(1, t1, false, c1)), b = m31_mul(base, fac(1, t1, true, c1));
    v[0] = m31_mul(a, fac(0, t0a, false, c0));
    v[1] = m31_mul(a, fac(0, t0a, true, c0));
    v[2] = m31_mul(b, fac(0, t0b, false, c0));
    v[3] = m31_mul(b, fac(0, t0b, true, c0));
  }
}

// A constant as signed bytes d_0..d_3 of weight 1, 2^8, 2^15, 2^23.  With
// c = d_0 + 256 d_1 in [-2^14, 2^14) and d = d_2 + 256 d_3 in [-32896, 32640),
// w = v (less P where that is needed for d's range) + 2^14 + 32896 * 2^15 is in
// [0, 2^31) and holds c + 2^14 in its low 15 bits and d + 32896 above; both
// halves are then spread to 16 bits, c's brought to + 32896, and each byte
// taken less 128.
__device__ __forceinline__ uint32_t mx_digits(uint32_t v) {
  const uint32_t u = v + 0x40404000u, w = umin32(u, u - P);
  return (w + (w & 0xffff8000u) + 0x4080u) ^ kMxSign;
}
__device__ __forceinline__ uint32_t m31_rot8(uint32_t v) { return ((v & 0x7fffffu) << 8) | (v >> 23); }  // 256 v

// The start values of a row whose constants sum to `sum`.
__device__ __forceinline__ void mx_starts(uint32_t sum, uint32_t &c0, uint32_t &c2) {
  const uint32_t k = m31_sub(m31_mul(sum, kMxSignP), kMxOffSum);
  c0 = (k & 0x7fffu) + kMxOff;
  c2 = (k >> 15) + kMxOff;
}

template <bool INV>
__device__ __forceinline__ MxMat mx_build(const uint32_t *tw_end, uint32_t D, uint32_t h, uint32_t layers,
                                          uint32_t scale) {
  const uint32_t g = (threadIdx.x >> 4) & 3;
  uint32_t v[4];
  mx_consts<INV>(tw_end, D, h, layers, scale, v);
  MxMat M;
  uint32_t sum = m31_add(m31_add(v[0], v[1]), m31_add(v[2], v[3]));
#pragma unroll
  for (uint32_t q = 0; q < 4; q++) {
    uint32_t pk[4], vl = v[q];
#pragma unroll
    for (int l = 0; l < 4; l++) {  // v * 256^l
      pk[l] = mx_digits(vl);
      vl = m31_rot8(vl);
    }
    const uint32_t l01 = perm(pk[1], pk[0], 0x05010400u), h01 = perm(pk[1], pk[0], 0x07030602u);
    const uint32_t l23 = perm(pk[3], pk[2], 0x05010400u), h23 = perm(pk[3], pk[2], 0x07030602u);
    M.a[0][q] = (int)perm(l23, l01, 0x05040100u);
    M.a[1][q] = (int)perm(l23, l01, 0x07060302u);
    M.a[2][q] = (int)perm(h23, h01, 0x05040100u);
    M.a[3][q] = (int)perm(h23, h01, 0x07060302u);
  }
  sum = m31_add(sum, (uint32_t)__shfl_xor((int)sum, 16));
  sum = m31_add(sum, (uint32_t)__shfl_xor((int)sum, 32));
#pragma unroll
  for (uint32_t r = 0; r < 4; r++) {
    uint32_t c0, c2;
    mx_starts((uint32_t)__shfl((int)sum, (int)(4 * g + r)), c0, c2);
    M.c0[r] = (int)c0;
    M.c2[r] = (int)c2;
  }
  return M;
}

// The same matrix built by the 16 waves of a workgroup into LDS, one constant
// times one power of 256 per lane: wave w holds power l = w / 4 and rows 4 (w % 4) + lane / 16, its
// lanes % 16 the columns.  `m`: 1,024 operand words (operand, lane, register)
// and 2 x 16 start values, as in the table.
template <bool INV>
__device__ __forceinline__ void mx_build_wg(const uint32_t *tw_end, uint32_t D, uint32_t h, uint32_t layers,
                                            uint32_t scale, uint32_t *m) {
  const uint32_t l = threadIdx.x >> 8, row = (threadIdx.x >> 4) & 15, col = threadIdx.x & 15;
  const uint32_t e = INV ? col : row, c = INV ? row : col;
  uint32_t v = scale;
#pragma unroll
  for (uint32_t r = 0; r < 4; r++) {
    const uint32_t t = gld(tw_end - ((size_t)1 << (D - r)), ((h << (3 - r)) | (e >> (r + 1))) << 2);
    const bool er = (e >> r) & 1, cr = (c >> r) & 1;
    const uint32_t p = m31_mul(v, er ? P - t : t);
    v = r < layers ? (cr ? p : v) : (er == cr ? v : 0);
  }
  uint32_t sum = v;
#pragma unroll
  for (int k = 1; k < 16; k <<= 1) sum = m31_add(sum, (uint32_t)__shfl_xor((int)sum, k));
  for (uint32_t k = 0; k < l; k++) v = m31_rot8(v);
  const uint32_t d = mx_digits(v);
  uint8_t *mb = reinterpret_cast<uint8_t *>(m);
  const uint32_t word = ((col >> 2) * 16 + row) * 4 + (col & 3);  // (lane, register) of [row][col]
#pragma unroll
  for (uint32_t k = 0; k < 4; k++) mb[(k * 256 + word) * 4 + l] = (uint8_t)(d >> (8 * k));
  if (l == 0 && col == 0) mx_starts(sum, m[1024 + row], m[1040 + row]);
}

// Four words of a lane (elements 4 g .. 4 g + 3 of one vector, as signed
// bytes: word ^ kMxSign) -> the products, congruent mod P and below
// 2^31 + 2^29 + 2^23 (m31_reduce1 makes them canonical).
__device__ __forceinline__ void mx_apply(const MxMat &M, const uint32_t x[4], uint32_t u[4]) {
  const i32x4 b = {(int)x[0], (int)x[1], (int)x[2], (int)x[3]}, z = {0, 0, 0, 0};
  const i32x4 a0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(M.a[0], b, M.c0, 0, 0, 0);
  const i32x4 a1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(M.a[1], b, z, 0, 0, 0);
  const i32x4 a2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(M.a[2], b, M.c2, 0, 0, 0);
  const i32x4 a3 = __builtin_amdgcn_mfma_i32_16x16x64_i8(M.a[3], b, z, 0, 0, 0);
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const uint32_t c = ((uint32_t)a1[r] << 8) + (uint32_t)a0[r];
    const uint32_t d = ((uint32_t)a3[r] << 8) + (uint32_t)a2[r];
    // u = c + (d >> 16) + (d & 0xffff) * 2^15: one multiply-add of 16-bit halves
    // each (the compiler takes four instructions).
    uint32_t t;
    asm("v_mad_u32_u16 %0, %1, 1, %2 op_sel:[1,0,0,0]" : "=v"(t) : "v"(d), "v"(c));
    asm("v_mad_u32_u16 %0, %1, %2, %3" : "=v"(u[r]) : "v"(d), "s"(0x8000u), "v"(t));
  }
}
__device__ __forceinline__ uint32_t m31_reduce1(uint32_t u) { return umin32(u, u - P); }

// ---- the matrix table of the strided top passes -----------------------------
//
// Kept with the twiddle tree: per matrix 4 x 64 x 4 words of operands
// (operand m, lane, register) and 2 x 16 start values.
constexpr uint32_t kMxWords = 1024 + 32;
constexpr uint32_t kMxInvTop = 0;                       // [29]: layers n-4..n-1 inverse, scaled by 2^-n
constexpr uint32_t kMxInv8 = kMxInvTop + 29;            // [16]: layers n-8..n-5 inverse
constexpr uint32_t kMxFwd4 = kMxInv8 + 16;              // [b][2^b]
constexpr uint32_t kMxFwd8 = kMxFwd4 + (2u << kMxMaxBlowup) - 1;  // [b][16 * 2^b]
constexpr uint32_t kMxCount = kMxFwd8 + 16 * ((2u << kMxMaxBlowup) - 1);

__device__ __forceinline__ uint32_t mx_fwd4(uint32_t b, uint32_t k) { return kMxFwd4 + (1u << b) - 1 + k; }
__device__ __forceinline__ uint32_t mx_fwd8(uint32_t b, uint32_t k) { return kMxFwd8 + 16 * ((1u << b) - 1) + k; }

__device__ __forceinline__ void mx_store(uint32_t *m, const MxMat &M) {
  const uint32_t lane = threadIdx.x & 63, row = lane & 15, g = lane >> 4;
#pragma unroll
  for (uint32_t k = 0; k < 4; k++)
    *(g_u4 *)as_global(m + (k * 64 + lane) * 4) = u32x4{(uint32_t)M.a[k][0], (uint32_t)M.a[k][1], (uint32_t)M.a[k][2],
                                                        (uint32_t)M.a[k][3]};
  if (row == 0) {
    *(g_u4 *)as_global(m + 1024 + 4 * g) = u32x4{(uint32_t)M.c0[0], (uint32_t)M.c0[1], (uint32_t)M.c0[2], (uint32_t)M.c0[3]};
    *(g_u4 *)as_global(m + 1040 + 4 * g) = u32x4{(uint32_t)M.c2[0], (uint32_t)M.c2[1], (uint32_t)M.c2[2], (uint32_t)M.c2[3]};
  }
}
__device__ __forceinline__ i32x4 ld_i4(const uint32_t *p, uint32_t byte_off) {
  const u32x4 v = gld4(p, byte_off);
  return i32x4{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
}
__device__ __forceinline__ MxMat mx_load(const uint32_t *table, uint32_t id) {
  const uint32_t lane = threadIdx.x & 63, g = lane >> 4;
  const uint32_t *m = table + (size_t)id * kMxWords;
  MxMat M;
#pragma unroll
  for (uint32_t k = 0; k < 4; k++) M.a[k] = ld_i4(m, (k * 64 + lane) * 16);
  M.c0 = ld_i4(m, (1024 + 4 * g) * 4);
  M.c2 = ld_i4(m, (1040 + 4 * g) * 4);
  return M;
}

// A matrix laid out like the table's in LDS.
__device__ __forceinline__ MxMat mx_lds(const uint32_t *m) {
  const uint32_t lane = threadIdx.x & 63, g = lane >> 4;
  MxMat M;
#pragma unroll
  for (uint32_t k = 0; k < 4; k++) M.a[k] = *reinterpret_cast<const i32x4 *>(m + (k * 64 + lane) * 4);
  M.c0 = *reinterpret_cast<const i32x4 *>(m + 1024 + 4 * g);
  M.c2 = *reinterpret_cast<const i32x4 *>(m + 1040 + 4 * g);
  return M;
}

// One wave per matrix.
__global__ void __launch_bounds__(64) mx_table_kernel(const uint32_t *tw_end, const uint32_t *itw_end, uint32_t *table) {
  const uint32_t id = blockIdx.x;
  uint32_t *m = table + (size_t)id * kMxWords;
  if (id < kMxInv8) {
    // 2^-n = 2^(31 k - n): a power of two (2^31 = 1)
    const uint32_t n = id - kMxInvTop;
    mx_store(m, mx_build<true>(itw_end, 4, 0, 4, n ? 1u << (31 - n) : 1u));
  } else if (id < kMxFwd4) {
    mx_store(m, mx_build<true>(itw_end, 8, id - kMxInv8, 4, 1));
  } else if (id < kMxFwd8) {
    const uint32_t j = id - kMxFwd4 + 1, b = 31 - __clz(j);
    mx_store(m, mx_build<false>(tw_end, 4 + b, j - (1u << b), 4, 1));
  } else {
    const uint32_t j = id - kMxFwd8 + 16, b = 31 - __clz(j >> 4);
    mx_store(m, mx_build<false>(tw_end, 8 + b, j - (16u << b), 4, 1));
  }
}

// ---- strided top passes ------------------------------------------------------
//
// The top 4 or 8 layers of a column of 2^n coefficients.  INV: the inverse
// layers (scaled by 1/2^n, so they end an interpolation); FWD: the forward
// layers of each of the 2^b output blocks (they start an evaluation); both:
// the coefficients stay in registers between the two, and are stored only
// when p.store.  A lane's 16 words are rows 4 g + q (q = 0..3) at 4
// consecutive positions 4 n' + k: 16-byte accesses in runs of 256 bytes, and
// each k is one MFMA vector group.

struct Words16 {
  uint32_t w[4][4];  // [q][k]
};

// Words of 4 rows `step` words apart (uniform) from lane offset `off` words.
//
// ONCE: non-temporal, for the words between the fused pass's reads and the
// evaluations: the intermediates that a pass hands on and the low pass's
// output.  Each is touched once per launch, and kept in the caches they push
// out the matrices (0.7 MB, read by every wave for every tile) and each other.
// With either side alone the gain is lost where a set fits the 256 MB cache
// (100 x 2^17 at blowup 2: stores only 95 us, both 87, neither 91); both: 256 x
// 2^20 at blowup 4 commit 6.10 -> 5.96 ms, 1,024 uneven columns 1,666 -> 1,600
// us, a 256 x 2^18 prove 2.07 -> 2.01 ms; sets that stay in the cache either way
// are within 3% (20 x 2^18 at 2 46 -> 45 us, 40 x 2^17 at 4 70 -> 72).  A branch
// on the size inside the kernels cost the prove 35 us and gave those nothing
// back.  The caller's own columns (an
// inverse's input, the coefficients of a forward pass alone) are read the
// ordinary way: they may well be in the cache (forward-only reads as ONCE: 91
// -> 98 us).
template <bool ONCE = false>
__device__ __forceinline__ void mx_ld(const uint32_t *col, uint32_t step, uint32_t off, Words16 &x) {
#pragma unroll
  for (uint32_t q = 0; q < 4; q++) {
    const uint32_t *r = col + (size_t)q * step;
    const u32x4 v = ONCE ? gld4_once(r, off << 2) : gld4(r, off << 2);
    x.w[q][0] = v.x;
    x.w[q][1] = v.y;
    x.w[q][2] = v.z;
    x.w[q][3] = v.w;
  }
}
template <bool ONCE = false>
__device__ __forceinline__ void mx_st(uint32_t *col, uint32_t step, uint32_t off, const Words16 &x) {
#pragma unroll
  for (uint32_t q = 0; q < 4; q++) {
    const u32x4 v{x.w[q][0], x.w[q][1], x.w[q][2], x.w[q][3]};
    uint32_t *r = col + (size_t)q * step;
    if (ONCE) gst4_once(r, off << 2, v); else gst4(r, off << 2, v);
  }
}

// Applies M to each of the 4 vector groups.  SIGN: the input words still have
// plain bytes.  The output is canonical when CANON, else congruent words.
// GROUPS: how many groups' accumulators may be in flight (16 registers each).
template <bool SIGN, bool CANON, int GROUPS = 2>
__device__ __forceinline__ void mx_stage(const MxMat &M, const Words16 &x, Words16 &y) {
#pragma unroll
  for (int k = 0; k < 4; k++) {
    uint32_t b[4], u[4];
#pragma unroll
    for (int q = 0; q < 4; q++) b[q] = SIGN ? x.w[q][k] ^ kMxSign : x.w[q][k];
    mx_apply(M, b, u);
#pragma unroll
    for (int q = 0; q < 4; q++) {
      y.w[q][k] = CANON ? m31_reduce1(u[q]) : u[q];
      // Combined here, not where a conditional store uses it: sunk there, all
      // four groups' accumulators would be live at once.
      asm volatile("" : "+v"(y.w[q][k]));
    }
    if (k % GROUPS == GROUPS - 1) __builtin_amdgcn_sched_barrier(0);
  }
}

// 8 layers: a workgroup of 16 waves owns 256 rows x 64 positions.  With the
// row index split as U (upper 4 bits) and e (lower 4), wave w first holds
// U = w with its lanes on e, or e = w with its lanes on U; the tile changes
// between the two through LDS, whose 64-word rows are rotated by 16 words per
// 4 rows of U and of e so that the lanes g = 0..3 of an access start on
// different banks.
//
// LDS word of row (U, e) = (w, 4 g) (UWAVE) or (4 g, w); the lane's rows q
// follow at 64 or 1,024 words.
template <bool UWAVE>
__device__ __forceinline__ uint32_t mx_row(uint32_t w, uint32_t pos) {
  const uint32_t g = (threadIdx.x >> 4) & 3;
  const uint32_t row = UWAVE ? (w << 4) | (g << 2) : (g << 6) | w;
  return (row << 6) + ((pos + ((g + (w >> 2)) << 4)) & 63);
}
template <bool UWAVE>
__device__ __forceinline__ void mx_put(uint32_t *L, const Words16 &x) {
#pragma unroll
  for (uint32_t q = 0; q < 4; q++)
    *reinterpret_cast<uint4 *>(L + q * (UWAVE ? 64 : 1024)) =
        make_uint4(x.w[q][0] ^ kMxSign, x.w[q][1] ^ kMxSign, x.w[q][2] ^ kMxSign, x.w[q][3] ^ kMxSign);
}
template <bool UWAVE>
__device__ __forceinline__ void mx_get(const uint32_t *L, Words16 &x) {
#pragma unroll
  for (uint32_t q = 0; q < 4; q++) {
    const uint4 v = *reinterpret_cast<const uint4 *>(L + q * (UWAVE ? 64 : 1024));
    x.w[q][0] = v.x;
    x.w[q][1] = v.y;
    x.w[q][2] = v.z;
    x.w[q][3] = v.w;
  }
}

// Exchanges alternate between two tile buffers, so each needs one barrier: a
// buffer is written again only after the barrier of the exchange in between,
// which every wave reaches after its reads.  Waves drift by up to an exchange
// and overlap each other's loads, products and stores (one workgroup fills a
// CU).  The matrices that all waves share are copied to LDS once; the next tile's rows and the wave's next matrix are
// loaded ahead, before the stores that a wait for them would otherwise include.
// 256 x 2^20 at blowup 4: 1.18 ms for 5.5 GB, 4.7 TB/s (a large copy: 4.9;
// 1.38 ms with ordinary loads and stores), where the butterfly form of the fused
// pass (lde_pass_kernel<9, 2>) takes 2.04 ms; the accesses are 256-byte runs 16
// KB apart.
constexpr uint32_t kMxTopLds = 1 + (1u << kMxMaxBlowup);  // the inverse one, one per output block
struct MxTopLds {
  uint32_t t[2][256 * 64];
  uint32_t m[kMxTopLds][kMxWords];
};

template <bool INV, bool FWD>
__device__ __forceinline__ void mx_top8_body(const MxTop &p, uint32_t wg, MxTopLds &S) {
  uint32_t *lds = S.t[0];
  const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t n = p.n, row_log = n - 8, blk_log = row_log - 6;
  const uint32_t n_tiles = p.n_cols << blk_log;
  // A workgroup's tiles are p.wgs apart, so that those running together cover
  // consecutive 256-byte runs of a row (all channels) and not every eighth.
  const uint32_t tile0 = wg, tile1 = n_tiles, step = p.wgs;
  const uint32_t g = (threadIdx.x >> 4) & 3, lane_pos = (threadIdx.x & 15) << 2;
  const uint32_t *table = p.mats;
  const FftCol *icols = INV ? p.icols : p.fcols;
  constexpr int G = INV && FWD ? 1 : 2;  // the fused pass has 16 more words live
  // rows (U, e) = (w, 4 g + q): first row and step in words; (4 g + q, w) likewise
  const uint32_t u_row = ((w << 4) | (g << 2)) << row_log, u_step = 1u << row_log;
  const uint32_t e_row = ((g << 6) | w) << row_log, e_step = 16u << row_log;
  uint32_t *const lu = lds + mx_row<true>(w, lane_pos), *const le = lds + mx_row<false>(w, lane_pos);
  uint32_t buf = 0;
  Words16 x;
  auto load = [&](uint32_t tile) {
    const uint32_t *in = (const uint32_t *)readfirstlane_u64((uint64_t)icols[tile >> blk_log].in);
    const uint32_t pos = ((tile & ((1u << blk_log) - 1)) << 6) + lane_pos;
    mx_ld<INV && FWD>(in, INV ? u_step : e_step, (INV ? u_row : e_row) + pos, x);
  };
  load(tile0);
  MxMat M = mx_load(table, INV ? kMxInv8 + w : mx_fwd8(p.b, w));
  // shared matrices: the inverse top one, then the forward ones by block
  constexpr uint32_t F0 = INV ? 1 : 0;
  const uint32_t n_rep = FWD ? 1u << p.b : 0, n_lds = F0 + n_rep;
  for (uint32_t j = threadIdx.x; j < n_lds * (kMxWords / 4); j += 1024) {
    const uint32_t k = j / (kMxWords / 4), o = j - k * (kMxWords / 4);
    const uint32_t id = INV && k == 0 ? kMxInvTop + n : mx_fwd4(p.b, k - F0);
    const uint4 v = ld_global4(table + (size_t)id * kMxWords + 4 * o);
    *reinterpret_cast<uint4 *>(&S.m[k][4 * o]) = v;
  }
  __syncthreads();
  for (uint32_t tile = tile0; tile < tile1; tile += step) {
    const uint32_t ci = tile >> blk_log;
    const uint32_t pos = ((tile & ((1u << blk_log) - 1)) << 6) + lane_pos;
    Words16 y;
    if (INV) {
      mx_stage<true, false, G>(M, x, y);
      mx_put<true>(lu + buf, y);
      if (FWD) M = mx_load(table, mx_fwd8(p.b, w));
      if (!FWD && tile + step < tile1) load(tile + step);
      __syncthreads();
      mx_get<false>(le + buf, y);
      buf ^= 256 * 64;
      mx_stage<false, true, G>(mx_lds(S.m[0]), y, FWD ? x : y);
      if (!FWD) M = mx_load(table, kMxInv8 + w);
      if (p.store)
        mx_st((uint32_t *)readfirstlane_u64((uint64_t)p.icols[ci].out), e_step, e_row + pos, FWD ? x : y);
    }
    if (FWD) {
      uint32_t *out = (uint32_t *)readfirstlane_u64((uint64_t)p.fcols[ci].out);
      for (uint32_t rep = 0; rep < n_rep; rep++) {
        const bool last = rep + 1 == n_rep;
        mx_stage<true, false, G>(mx_lds(S.m[F0 + rep]), x, y);
        mx_put<false>(le + buf, y);
        if (last && tile + step < tile1) load(tile + step);
        __syncthreads();
        mx_get<true>(lu + buf, y);
        buf ^= 256 * 64;
        mx_stage<false, true, G>(M, y, y);
        M = mx_load(table, INV && last ? kMxInv8 + w : mx_fwd8(p.b, (last ? 0 : (rep + 1) * 16) + w));
        mx_st<true>(out + ((size_t)rep << n), u_step, u_row + pos, y);
      }
    }
  }
}

// 4 layers: one wave per 16 rows x 64 positions, no exchange.
template <bool INV, bool FWD>
__device__ __forceinline__ void mx_top4_body(const MxTop &p, uint32_t wg) {
  const uint32_t n = p.n, row_log = n - 4, blk_log = row_log - 6;
  const uint32_t unit = __builtin_amdgcn_readfirstlane((wg << 2) | (threadIdx.x >> 6));
  if (unit >= p.n_cols << blk_log) return;
  const uint32_t ci = unit >> blk_log;
  const uint32_t pos = ((unit & ((1u << blk_log) - 1)) << 6) + ((threadIdx.x & 15) << 2);
  Words16 x, y;
  const uint32_t step = 1u << row_log, off = ((threadIdx.x & 48) >> 2 << row_log) + pos;  // rows 4 g + q
  const uint32_t *in = (const uint32_t *)readfirstlane_u64((uint64_t)(INV ? p.icols[ci].in : p.fcols[ci].in));
  mx_ld<INV && FWD>(in, step, off, x);
  if (INV) {
    const MxMat T = mx_load(p.mats, kMxInvTop + n);
    mx_stage<true, true>(T, x, y);
    x = y;
    if (p.store) mx_st((uint32_t *)readfirstlane_u64((uint64_t)p.icols[ci].out), step, off, x);
  }
  if (FWD) {
    uint32_t *out = (uint32_t *)readfirstlane_u64((uint64_t)p.fcols[ci].out);
    for (uint32_t rep = 0; rep < 1u << p.b; rep++) {
      const MxMat T = mx_load(p.mats, mx_fwd4(p.b, rep));
      mx_stage<true, true>(T, x, y);
      mx_st<true>(out + ((size_t)rep << n), step, off, y);
    }
  }
}

// The group whose range of workgroups [start, next start) holds this one.
template <typename G>
__device__ __forceinline__ uint32_t find_group(const G *groups, uint32_t n_groups) {
  uint32_t g = 0, hi = n_groups;
  while (hi - g > 1) {
    const uint32_t mid = (g + hi) >> 1;
    if (groups[mid].wg_start <= blockIdx.x) g = mid; else hi = mid;
  }
  return g;
}

// One group (descriptor by value) or several.
template <bool INV, bool FWD>
__global__ void __launch_bounds__(1024) mx_top8_kernel(MxTop p) {
  __shared__ __align__(16) MxTopLds L;
  mx_top8_body<INV, FWD>(p, blockIdx.x, L);
}
template <bool INV, bool FWD>
__global__ void __launch_bounds__(1024) mx_top8_multi_kernel(const MxTop *groups, uint32_t n_groups) {
  __shared__ __align__(16) MxTopLds L;
  const uint32_t g = find_group(groups, n_groups);
  mx_top8_body<INV, FWD>(groups[g], blockIdx.x - groups[g].wg_start, L);
}
template <bool INV, bool FWD>
__global__ void __launch_bounds__(256) mx_top4_kernel(MxTop p) {
  mx_top4_body<INV, FWD>(p, blockIdx.x);
}
template <bool INV, bool FWD>
__global__ void __launch_bounds__(256) mx_top4_multi_kernel(const MxTop *groups, uint32_t n_groups) {
  const uint32_t g = find_group(groups, n_groups);
  mx_top4_body<INV, FWD>(groups[g], blockIdx.x - groups[g].wg_start);
}

// ---- the contiguous low pass ---------------------------------------------------
//
// Bound by memory: 256 x 2^22 forward in 1.89 ms and 256 x 2^20 inverse in
// 0.45 ms move 4.5 and 4.8 TB/s (a large copy: 4.9), where twelve butterfly
// layers in registers (fft_pass_kernel) took 2.85 and 0.65 ms at the VALU's
// issue rate.
//
// Layers [0, t0), 9 <= t0 <= 12, on chunks of 4,096 consecutive words: layers
// 0..3 as register butterflies (their matrices would be one per 16 words),
// layers 4..7 and 8..t0-1 on the matrix cores.  A workgroup of 16 waves takes
// one chunk of 4 columns at a time and walks over up to 4 * iters columns: the
// matrices of a chunk are the same for every column, so they are built once
// from the twiddles (about 230 instructions per wave) and kept, the chunk's
// one matrix of layers 8.. in LDS and wave w's matrix of layers 4..7 (block
// U = w of the chunk's sixteen) in registers, like the 15 butterfly twiddles.
//
// Chunk index bits: U = [8, 12), e = [4, 8), i = [0, 4).  Only layers 8..
// cross the 256-word blocks U: there wave w works on column w / 4, rows U,
// positions 64 (w % 4) + 0..63, and the words change hands through LDS once
// (layout A, a block of 256 words per column and U, one barrier).  Layers 0..7
// of block U = w of all 4 columns belong to wave w alone, which turns its
// block in place in LDS between the two forms (layout B) with no barrier.
// Two tile buffers alternate, so a wave may be an iteration ahead of others
// and one wave's loads and stores run under another's products.
//
// Banks: A permutes its 16-word rows within their group of 4, so that the
// lanes of the e groups, 64 words apart, meet different banks; columns are 16
// words apart modulo 64 for the same reason in B, which also rotates e by 4
// words per 4 i, so that a lane's 4 consecutive e are one 16-byte access and
// lanes i = 0..15 cover all banks.
__device__ __forceinline__ uint32_t mx_a_off(uint32_t e, uint32_t i) {
  return (((e & ~3u) | ((e + (e >> 2)) & 3)) << 4) + i;
}
__device__ __forceinline__ uint32_t mx_b_off(uint32_t i, uint32_t e) { return (i << 4) + ((e + (i & ~3u)) & 15); }
constexpr uint32_t kMxCol = 4096 + 16;

constexpr uint32_t kMxIters = 16;  // most groups of 4 columns per workgroup
struct MxLowLds {
  uint32_t t[2][4][kMxCol];  // [buffer][column][U * 256 + A or B offset]
  uint32_t m[1024 + 32];
  uint32_t tw[16][16][16];  // [U][e]: a butterfly lane's 15 twiddles
  uint32_t c[16][32];       // [U]: start values of the block's matrix
  FftCol col[4 * kMxIters];
};

// A wave's own LDS writes are in order with its reads; this keeps the
// compiler from moving them across the change of layout.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <bool INV>
__device__ __forceinline__ void mx_low_body(const MxLow &p, uint32_t wg, MxLowLds &S) {
  const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & 63, g = lane >> 4, nn = lane & 15;
  const uint32_t slot = w >> 2, wq = w & 3;  // layers 8..: column of the four, quarter of its positions
  // Consecutive workgroups take consecutive chunks of the same columns: the
  // columns' same offsets would share memory channels.
  const uint32_t tile = wg & ((1u << (p.N - 12)) - 1), chunk = wg >> (p.N - 12);
  const uint32_t col0 = chunk * 4 * p.iters, col1 = min(col0 + 4 * p.iters, p.n_cols);
  // The walk's column addresses: read from memory inside it, each would wait
  // for every load and store in flight (one in-order counter).
  if (threadIdx.x < col1 - col0) S.col[threadIdx.x] = p.cols[col0 + threadIdx.x];
  // butterflies of layers 0..3: lane (column g, e = nn), the 16 words at
  // U * 256 + 16 e of its column
  const uint32_t bfly0 = (w << 8) | (nn << 4);
  const uint32_t in_chunk = INV ? tile << 12 : (tile << 12) & ((1u << p.in_log) - 1);
  const uint32_t rpos = (wq << 6) + (nn << 2);
  uint32_t xin[16];
  // Forward: rows U = 4 g + q of column c0 + slot; inverse: this lane's 16
  // words of column c0 + g.
  auto load = [&](uint32_t c0, const FftCol *cols, uint32_t base) {
    const uint32_t c = c0 + (INV ? g : slot);
    if (c >= col1) return;
    const uint32_t *in = cols[c - base].in;
    if (!INV) in = (const uint32_t *)readfirstlane_u64((uint64_t)in);
#pragma unroll
    for (uint32_t q = 0; q < 4; q++) {
      const uint32_t o = INV ? in_chunk + bfly0 + 4 * q : in_chunk + ((4 * g + q) << 8) + rpos;
      const u32x4 v = INV ? gld4(in, o << 2) : gld4_once(in, o << 2);
      xin[4 * q] = v.x;
      xin[4 * q + 1] = v.y;
      xin[4 * q + 2] = v.z;
      xin[4 * q + 3] = v.w;
    }
  };
#pragma unroll
  for (int j = 0; j < 16; j++) xin[j] = 0;
  load(col0, p.cols, 0);  // under way while the matrices are built
  StageTw tw;
  load_stage_twiddles(tw, p.tw2_end, p.N, 0, (tile << 12) | bfly0, 0, 4);
  const MxMat M2 = mx_build<INV>(p.tw_end, p.N - 4, (tile << 4) | w, 4, 1);
  mx_build_wg<INV>(p.tw_end, p.N - 8, tile, p.t0 - 8, p.scale, S.m);
  // Twiddles and M2's start values are read back from LDS where they are
  // used: kept in registers for the whole walk they spilled.
  {
    if (g == 0) {
      uint4 *d = reinterpret_cast<uint4 *>(S.tw[w][nn]);
      d[0] = make_uint4(tw.t0[0], tw.t0[1], tw.t0[2], tw.t0[3]);
      d[1] = make_uint4(tw.t0[4], tw.t0[5], tw.t0[6], tw.t0[7]);
      d[2] = make_uint4(tw.t1[0], tw.t1[1], tw.t1[2], tw.t1[3]);
      d[3] = make_uint4(tw.t2[0], tw.t2[1], tw.t3[0], 0);
    }
    if (nn == 0) {
      *reinterpret_cast<i32x4 *>(&S.c[w][4 * g]) = M2.c0;
      *reinterpret_cast<i32x4 *>(&S.c[w][16 + 4 * g]) = M2.c2;
    }
  }
  auto lds_tw = [&]() {
    const uint4 *d = reinterpret_cast<const uint4 *>(S.tw[w][nn]);
    const uint4 a = d[0], b = d[1], c = d[2], e = d[3];
    StageTw t;
    t.t0[0] = a.x, t.t0[1] = a.y, t.t0[2] = a.z, t.t0[3] = a.w;
    t.t0[4] = b.x, t.t0[5] = b.y, t.t0[6] = b.z, t.t0[7] = b.w;
    t.t1[0] = c.x, t.t1[1] = c.y, t.t1[2] = c.z, t.t1[3] = c.w;
    t.t2[0] = e.x, t.t2[1] = e.y, t.t3[0] = e.z;
    return t;
  };
  auto m2 = [&]() {
    MxMat M = M2;
    M.c0 = *reinterpret_cast<const i32x4 *>(&S.c[w][4 * g]);
    M.c2 = *reinterpret_cast<const i32x4 *>(&S.c[w][16 + 4 * g]);
    return M;
  };
  const uint32_t st_off = ((lane >> 2) << 4) + ((((lane & 3) + (lane >> 4)) & 3) << 2);
  uint32_t boff[4];
#pragma unroll
  for (uint32_t k = 0; k < 4; k++) boff[k] = g * kMxCol + mx_b_off(4 * k, nn);
  // the A offset of positions rpos .. rpos + 3 (e = rpos / 16)
  const uint32_t a_rpos = mx_a_off(rpos >> 4, rpos & 15);
  __syncthreads();
  uint32_t buf = 0;
  for (uint32_t cb = col0; cb < col1; cb += 4) {
    uint32_t *T = &S.t[buf][0][0];
    uint32_t *blk = T + (w << 8);  // block U = w of column 0
    buf ^= 1;
    if (!INV) {
      {
        const MxMat M1 = mx_lds(S.m);
        Words16 x, y;
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
          for (int k = 0; k < 4; k++) x.w[q][k] = xin[4 * q + k];
        mx_stage<true, false, 1>(M1, x, y);
        load(cb + 4, S.col, col0);
#pragma unroll
        for (uint32_t q = 0; q < 4; q++)
          *reinterpret_cast<uint4 *>(&T[slot * kMxCol + (4 * g + q) * 256 + a_rpos]) =
              make_uint4(y.w[q][0] ^ kMxSign, y.w[q][1] ^ kMxSign, y.w[q][2] ^ kMxSign, y.w[q][3] ^ kMxSign);
      }
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);
      const MxMat Mb = m2();
#pragma unroll
      for (uint32_t k = 0; k < 4; k++) {
        if (cb + k >= col1) break;
        uint32_t b[4], u[4];
#pragma unroll
        for (uint32_t q = 0; q < 4; q++) b[q] = blk[k * kMxCol + mx_a_off(4 * g + q, nn)];
        mx_apply(Mb, b, u);
        *reinterpret_cast<uint4 *>(&blk[k * kMxCol + mx_b_off(nn, 4 * g)]) =
            make_uint4(m31_reduce1(u[0]), m31_reduce1(u[1]), m31_reduce1(u[2]), m31_reduce1(u[3]));
        __builtin_amdgcn_sched_barrier(0);
      }
      wave_lds_fence();
      __builtin_amdgcn_sched_barrier(0);
      uint32_t x[16];
#pragma unroll
      for (uint32_t i = 0; i < 16; i++) x[i] = blk[boff[i >> 2] + (i & 3) * 16];
      stage_layers<false, 0, 4>(x, lds_tw());
      // Back through the wave's block, so that a store writes 1 KB of one
      // column and not 16 bytes in each of 64 lines (256 x 2^22: 2.33 -> 1.89
      // ms, 4.5 TB/s read and written).  Groups of 4 words are rotated
      // within 16 by i / 4 of the lane for the banks.
#pragma unroll
      for (uint32_t q = 0; q < 4; q++)
        *reinterpret_cast<uint4 *>(&blk[g * kMxCol + (nn << 4) + (((q + (nn >> 2)) & 3) << 2)]) =
            make_uint4(x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]);
      wave_lds_fence();
#pragma unroll
      for (uint32_t k = 0; k < 4; k++) {
        if (cb + k >= col1) break;
        const uint4 v = *reinterpret_cast<const uint4 *>(&blk[k * kMxCol + st_off]);
        uint32_t *out = (uint32_t *)readfirstlane_u64((uint64_t)S.col[cb + k - col0].out);
        gst4_once(out, ((tile << 12) + (w << 8) + (lane << 2)) << 2, u32x4{v.x, v.y, v.z, v.w});
      }
    } else {
      uint32_t x[16];
#pragma unroll
      for (int i = 0; i < 16; i++) x[i] = xin[i];
      stage_layers<true, 0, 4>(x, lds_tw());
      load(cb + 4, S.col, col0);
#pragma unroll
      for (uint32_t i = 0; i < 16; i++)
        blk[boff[i >> 2] + (i & 3) * 16] = x[i] ^ kMxSign;
      wave_lds_fence();
      __builtin_amdgcn_sched_barrier(0);
      const MxMat Mb = m2();
#pragma unroll
      for (uint32_t k = 0; k < 4; k++) {
        if (cb + k >= col1) break;
        const uint4 v = *reinterpret_cast<const uint4 *>(&blk[k * kMxCol + mx_b_off(nn, 4 * g)]);
        const uint32_t b[4] = {v.x, v.y, v.z, v.w};
        uint32_t u[4];
        mx_apply(Mb, b, u);
#pragma unroll
        for (uint32_t q = 0; q < 4; q++) blk[k * kMxCol + mx_a_off(4 * g + q, nn)] = u[q] ^ kMxSign;
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);
      const MxMat M1 = mx_lds(S.m);
      Words16 xx, y;
#pragma unroll
      for (uint32_t q = 0; q < 4; q++) {
        const uint4 v = *reinterpret_cast<const uint4 *>(&T[slot * kMxCol + (4 * g + q) * 256 + a_rpos]);
        xx.w[q][0] = v.x;
        xx.w[q][1] = v.y;
        xx.w[q][2] = v.z;
        xx.w[q][3] = v.w;
      }
      mx_stage<false, true, 1>(M1, xx, y);
      if (cb + slot < col1) {
        uint32_t *out = (uint32_t *)readfirstlane_u64((uint64_t)S.col[cb + slot - col0].out);
#pragma unroll
        for (uint32_t q = 0; q < 4; q++)
          gst4(out, ((tile << 12) + ((4 * g + q) << 8) + rpos) << 2,
               u32x4{y.w[q][0], y.w[q][1], y.w[q][2], y.w[q][3]});
      }
    }
  }
}

template <bool INV>
__global__ void __launch_bounds__(1024) mx_low_kernel(MxLow p) {
  __shared__ __align__(16) MxLowLds S;
  mx_low_body<INV>(p, blockIdx.x, S);
}
template <bool INV>
__global__ void __launch_bounds__(1024) mx_low_multi_kernel(const MxLow *groups, uint32_t n_groups) {
  __shared__ __align__(16) MxLowLds S;
  const uint32_t g = find_group(groups, n_groups);
  mx_low_body<INV>(groups[g], blockIdx.x - groups[g].wg_start, S);
}

}  // namespace

constexpr uint64_t kMxBatchUnits = 32;  // kMxMinUnits, shared launch

uint64_t mx_top_units(uint32_t n_cols, uint32_t n, const MxPlan &plan) {
  return plan.top_layers == 8 ? (uint64_t)n_cols << (n - 14) : 0;
}
uint64_t mx_low_units(uint32_t n_cols, uint32_t N) { return (uint64_t)((n_cols + 3) / 4) << (N - 12); }

// The matrix passes need work for one workgroup per CU to pay for building
// their matrices.  Measured against the vector passes alone on a context (us,
// vector -> matrix, interpolation / evaluation at blowup 2): 64 low-pass units
// (2^16 x 16) 18.7 -> 22.4 / 24.8 -> 25.0; 128 (2^16 x 32) 25.9 -> 26.7 /
// 34.7 -> 33.3; 256 (2^16 x 64) 39.8 -> 35.1 / 49.1 -> 42.8; 1,024 (2^20 x 16)
// 88.3 -> 61.6 / 149 -> 115.  A batched launch shares its workgroups between
// groups, so there a group of kMxBatchUnits is taken along.  One or two columns
// would leave most of the low pass's four column slots empty; from 2^22 on, where
// three passes over memory are the time either way, three do too, and at 2^24 five
// (us, vector -> matrix, interpolation / evaluation at blowup 1, 2 and 4: 3 x 2^21 60 ->
// 56 / 58 -> 54, 88 -> 88 and 150 -> 154, 3 x 2^22 95 -> 92 / 90 -> 89, 151 -> 155 and 288 ->
// 306, 4 x 2^22 116 -> 106 / 110 -> 103, 193 -> 178 and 380 -> 351, 3 x 2^23 160 -> 167 / 153
// -> 164, 296 -> 314 and 588 -> 598, 5 x 2^24 501 -> 565 / 500 -> 551, 975 -> 989 and 1,910 ->
// 1,891, 6 x 2^24 596 -> 605 / 595 -> 591, 1,165 -> 1,086 and 2,289 -> 2,067).
bool mx_plan(const stwo_hip_ctx *ctx, const stwo_hip_twiddles *tw, uint32_t n, uint32_t b, bool inverse, size_t n_cols,
             bool aligned16, bool batched, MxPlan *plan) {
  if (!tw->d_mx || !aligned16 || n < kMxMinLog || n > kMxMaxLog || b > kMxMaxBlowup || n_cols < 3) return false;
  if ((n >= 22 && n_cols < 4) || (n >= 24 && n_cols == 5)) return false;
  const uint64_t units = mx_low_units((uint32_t)n_cols, n);
  if (units < (batched ? kMxBatchUnits : kMxMinUnits)) return false;
  // A vector plan chosen for the shape stands in a launch of its own.  It was timed
  // there: in a shared launch it would only take the group out of the others' (the
  // plan of 1,024 uneven columns 1.68 ms, 1.73 with three groups taken out; with them
  // kept in 1.60 beside 1.66).
  auto it = ctx->fft_tune.find(fft_tune_key(n, n + b, inverse));
  if (!batched && it != ctx->fft_tune.end() && it->second.chosen) return false;
  plan->top_layers = n == 12 ? 0 : n <= 16 ? 4 : 8;
  plan->t0 = n <= 20 ? n - plan->top_layers : 12;
  plan->mid = n > 20;
  return true;
}

// One workgroup fills a CU, so up to kMxIters units per CU the units are
// spread over the 256 CUs' worth of workgroups and each walks over its share
// (its matrices and the next unit's loads under the current one's products);
// past that a workgroup takes kMxIters.  100 x 2^17 -> 2^18 (1,600 units):
// 103 us, with one unit per workgroup instead 130 us.
// A launch over several groups mixes workgroups of different lengths, so there
// about four rounds of them even out the CUs' shares.
static uint32_t mx_iters(uint64_t units, bool batched) {
  const uint64_t per = batched ? 1024 : 256;
  return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(kMxIters, (units + per - 1) / per));
}

MxTop mx_top(const stwo_hip_twiddles *tw, const FftCol *icols, const FftCol *fcols, uint32_t n_cols, uint32_t n,
             uint32_t b, bool store, const MxPlan &plan, uint64_t launch_units, bool batched, uint32_t *wgs) {
  MxTop p{};
  p.icols = icols;
  p.fcols = fcols;
  p.mats = tw->d_mx;
  p.n_cols = n_cols;
  p.n = n;
  p.b = b;
  p.store = store;
  if (plan.top_layers == 8) {
    const uint32_t iters = mx_iters(launch_units, batched), units = (uint32_t)mx_top_units(n_cols, n, plan);
    p.wgs = (units + iters - 1) / iters;
  } else {
    p.wgs = ((n_cols << (n - 10)) + 3) / 4;
  }
  *wgs = p.wgs;
  return p;
}

MxLow mx_low(const stwo_hip_twiddles *tw, const FftCol *cols, uint32_t n_cols, uint32_t n, uint32_t N, bool inverse,
             const MxPlan &plan, uint64_t launch_units, bool batched, uint32_t *wgs) {
  MxLow p{};
  p.cols = cols;
  p.tw_end = (inverse ? tw->d_itw : tw->d_tw) + tw->len;
  p.tw2_end = (inverse ? tw->d_itw2 : tw->d_tw2) + tw->len;
  p.n_cols = n_cols;
  p.N = N;
  p.t0 = plan.t0;
  // after a top pass the chunks are whole; the low pass alone reads the
  // coefficients of every block
  p.in_log = plan.top_layers ? N : n;
  p.scale = inverse && !plan.top_layers ? 1u << (31 - n) : 1u;
  const uint32_t quads = (n_cols + 3) / 4;
  // an even share of the column groups for every part
  const uint32_t most = std::min(mx_iters(launch_units, batched), quads), parts = (quads + most - 1) / most;
  p.iters = (quads + parts - 1) / parts;
  *wgs = ((quads + p.iters - 1) / p.iters) << (N - 12);
  return p;
}

size_t mx_table_bytes(uint32_t root_log) { return root_log >= kMxMinLog ? (size_t)kMxCount * kMxWords * 4 : 0; }

int mx_table_build(stwo_hip_ctx *ctx, const uint32_t *tw_end, const uint32_t *itw_end, uint32_t *table) {
  return launch(ctx, "mx_table", mx_table_kernel, dim3(kMxCount), dim3(64), 0, tw_end, itw_end, table);
}

int launch_mx_top(stwo_hip_ctx *ctx, const MxTop *one, const MxTop *d_groups, uint32_t n_groups, uint32_t total_wgs,
                  uint32_t layers, bool inv, bool fwd) {
  const dim3 grid(total_wgs), block(layers == 8 ? 1024 : 256);
  const char *name = inv && fwd ? "lde_pass_mx_top" : inv ? "ifft_pass_mx_top" : "rfft_pass_mx_top";
#define STWO_MX_TOP(I, F)                                                                                       \
  if (inv == I && fwd == F) {                                                                                   \
    if (one)                                                                                                    \
      return launch(ctx, name, layers == 8 ? mx_top8_kernel<I, F> : mx_top4_kernel<I, F>, grid, block, 0, *one); \
    return launch(ctx, name, layers == 8 ? mx_top8_multi_kernel<I, F> : mx_top4_multi_kernel<I, F>, grid, block, 0, \
                  d_groups, n_groups);                                                                          \
  }
  STWO_MX_TOP(true, true) STWO_MX_TOP(true, false) STWO_MX_TOP(false, true)
#undef STWO_MX_TOP
  return set_error(ctx, STWO_HIP_EINVAL, "internal: matrix pass without a direction");
}

int launch_mx_low(stwo_hip_ctx *ctx, const MxLow *one, const MxLow *d_groups, uint32_t n_groups, uint32_t total_wgs,
                  bool inverse) {
  const dim3 grid(total_wgs), block(1024);
  const char *name = inverse ? "ifft_pass_mx_low" : "rfft_pass_mx_low";
  if (one)
    return launch(ctx, name, inverse ? mx_low_kernel<true> : mx_low_kernel<false>, grid, block, 0, *one);
  return launch(ctx, name, inverse ? mx_low_multi_kernel<true> : mx_low_multi_kernel<false>, grid, block, 0, d_groups,
                n_groups);
}

}  // namespace stwo_hip
