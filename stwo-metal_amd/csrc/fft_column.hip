// Interpolation, evaluation or both of small columns (2^4 to 2^13 words), a
// workgroup per column, for calls that leave most of the device idle: there a
// pass costs its chain of memory round trips, not its arithmetic.
//
// The register passes (fft.hip) take a table, data and a stage's twiddles one
// after another, and an interpolation and an evaluation are two launches. Here
// the column and every twiddle of its domains (2^(n-1) and 2^(N-1) words, one
// contiguous end of each tree) are read at once, the transforms run two
// layers at a time through LDS, and the coefficients pass from the last
// interpolation step to the first evaluation step, whose elements are the same
// ones, in registers.  extend_evals of 16 columns of
// 2^10 at blowup 2 took 19.5 us in two passes, 6.2 us here.
#include "fft_column.hpp"

#include <algorithm>

#include "fft_dev.hpp"
#include "field.hpp"

namespace stwo_hip {
namespace {

constexpr uint32_t kColMaxLog = 13;  // domain; 59 KB of LDS at most (coefficients up to 2^12)
constexpr uint32_t kColMaxThreads = 1024;

// Position of element i: 4 words of padding every 64 spread the strides of
// the steps over the banks and keep runs of 4 aligned.
__device__ __forceinline__ uint32_t pos(uint32_t i) { return i + ((i >> 6) << 2); }

// Level s of the twiddles of a domain of 2^M, whose 2^(M-1) words are at T.
__device__ __forceinline__ const uint32_t *level(const uint32_t *T, uint32_t M, uint32_t s) {
  return T + ((1u << (M - 1)) - (1u << (M - s)));
}

// The circle layer's twiddles of pairs 2q and 2q + 1: from [y, -y, -x, x] of
// pairs (x, y) of level 1 (doubled, as fft_dev.hpp's load_level).
__device__ __forceinline__ void circle_pair(const uint32_t *T, uint32_t q, uint32_t &t0, uint32_t &t1) {
  const uint32_t v = T[(q & ~1u) | (q & 1 ? 0u : 1u)], neg = 2u * P - v;
  t0 = q & 1 ? neg : v;
  t1 = q & 1 ? v : neg;
}

// Layers s + 1 and s of the quad whose elements are 2^s apart, the first of
// its pairs being pair h of layer s + 1.
template <bool INV>
__device__ __forceinline__ void quad_layers(uint32_t (&x)[4], uint32_t t1, uint32_t t00, uint32_t t01) {
  if (INV) {
    bfly<true>(x[0], x[1], t00);
    bfly<true>(x[2], x[3], t01);
    bfly<true>(x[0], x[2], t1);
    bfly<true>(x[1], x[3], t1);
  } else {
    bfly<false>(x[0], x[2], t1);
    bfly<false>(x[1], x[3], t1);
    bfly<false>(x[0], x[1], t00);
    bfly<false>(x[2], x[3], t01);
  }
}

// The lowest quad (4 neighbours): layers 0 and, in an even number of layers, 1.
template <bool INV>
__device__ __forceinline__ void low_layers(uint32_t (&x)[4], const uint32_t *T, uint32_t M, uint32_t q, bool two) {
  uint32_t t0, t1;
  circle_pair(T, q, t0, t1);
  const uint32_t t2 = two ? level(T, M, 1)[q] : 0;
  if (INV) {
    bfly<true>(x[0], x[1], t0);
    bfly<true>(x[2], x[3], t1);
    if (two) {
      bfly<true>(x[0], x[2], t2);
      bfly<true>(x[1], x[3], t2);
    }
  } else {
    if (two) {
      bfly<false>(x[0], x[2], t2);
      bfly<false>(x[1], x[3], t2);
    }
    bfly<false>(x[0], x[1], t0);
    bfly<false>(x[2], x[3], t1);
  }
}

// Layers s, s + 1 over the 2^M elements in D.
template <bool INV>
__device__ __forceinline__ void lds_step(uint32_t *D, const uint32_t *T, uint32_t M, uint32_t s) {
  const uint32_t *l0 = level(T, M, s), *l1 = level(T, M, s + 1);
  for (uint32_t q = threadIdx.x; q < 1u << (M - 2); q += blockDim.x) {
    const uint32_t h = q >> s, g = (h << (s + 2)) | (q & ((1u << s) - 1));
    uint32_t x[4];
#pragma unroll
    for (int k = 0; k < 4; k++) x[k] = D[pos(g + ((uint32_t)k << s))];
    quad_layers<INV>(x, l1[h], l0[2 * h], l0[2 * h + 1]);
#pragma unroll
    for (int k = 0; k < 4; k++) D[pos(g + ((uint32_t)k << s))] = x[k];
  }
  __syncthreads();
}

// Steps pair the layers from the top, so an odd count leaves layer 0 alone.
template <bool INV, bool FWD>
__device__ __forceinline__ void column_body(const ColumnFft &p, const FftCol *cols, uint32_t col, uint32_t *S) {
  const uint32_t tid = threadIdx.x, nt = blockDim.x, n = p.n, N = FWD ? p.N : n;
  const uint32_t Q = 1u << (n - 2), s_low = n & 1 ? 1 : 2;
  const bool two = !(n & 1);
  uint32_t *TI = S, *TF = TI + (INV ? 1u << (n - 1) : 0), *D = TF + (FWD ? 1u << (N - 1) : 0);
  // At least 2^(N-3) lanes: 4 twiddles a lane at most, and two quads.
  const bool has_ti = INV && 4 * tid < 1u << (n - 1), has_tf = FWD && 4 * tid < 1u << (N - 1);
  u32x4 ti = {0, 0, 0, 0}, tf = {0, 0, 0, 0};
  if (has_ti) ti = gld4(p.itw_end - ((size_t)1 << (n - 1)), 16 * tid);
  if (has_tf) tf = gld4(p.tw_end - ((size_t)1 << (N - 1)), 16 * tid);
  const FftCol c = cols[col];
  const uint32_t *in = (const uint32_t *)readfirstlane_u64((uint64_t)c.in);
  uint32_t *coeffs = (uint32_t *)in, *out = (uint32_t *)readfirstlane_u64((uint64_t)c.out);
  uint32_t x[2][4];
#pragma unroll
  for (int it = 0; it < 2; it++) {
    const uint32_t q = tid + it * nt;
    if (q >= Q) continue;
    if (!INV) {
#pragma unroll
      for (int k = 0; k < 4; k++) x[it][k] = gld(in, (q + k * Q) << 2);
    } else if (((uintptr_t)in & 15) == 0) {
      const u32x4 v = gld4(in, q << 4);
      x[it][0] = v.x;
      x[it][1] = v.y;
      x[it][2] = v.z;
      x[it][3] = v.w;
    } else {
#pragma unroll
      for (int k = 0; k < 4; k++) x[it][k] = gld(in, (4 * q + k) << 2);
    }
  }
  if (has_ti) *reinterpret_cast<u32x4 *>(TI + 4 * tid) = ti;
  if (has_tf) *reinterpret_cast<u32x4 *>(TF + 4 * tid) = tf;
  __syncthreads();
  if (INV) {
#pragma unroll
    for (int it = 0; it < 2; it++) {
      const uint32_t q = tid + it * nt;
      if (q >= Q) continue;
      low_layers<true>(x[it], TI, n, q, two);
      *reinterpret_cast<u32x4 *>(D + pos(4 * q)) = u32x4{x[it][0], x[it][1], x[it][2], x[it][3]};
    }
    __syncthreads();
    for (uint32_t s = s_low; s + 2 < n; s += 2) lds_step<true>(D, TI, n, s);
  }
  // The top two layers, of the interpolation and of the evaluation: the same
  // four elements of a lane.  An evaluation on a larger domain starts from
  // 2^(N-n) copies of the coefficients.
#pragma unroll
  for (int it = 0; it < 2; it++) {
    const uint32_t q = tid + it * nt;
    if (q >= Q) continue;
    if (INV) {
#pragma unroll
      for (int k = 0; k < 4; k++) x[it][k] = D[pos(q + k * Q)];
      const uint32_t *l0 = level(TI, n, n - 2), *l1 = level(TI, n, n - 1);
      quad_layers<true>(x[it], l1[0], l0[0], l0[1]);
#pragma unroll
      for (int k = 0; k < 4; k++) x[it][k] = m31_mul(x[it][k], p.scale);
      if (!FWD || p.store)
#pragma unroll
        for (int k = 0; k < 4; k++) gst(coeffs, (q + k * Q) << 2, x[it][k]);
    }
    if (FWD) {
      const uint32_t *l0 = level(TF, N, n - 2), *l1 = level(TF, N, n - 1);
      for (uint32_t r = 0; r < 1u << (N - n); r++) {
        uint32_t y[4] = {x[it][0], x[it][1], x[it][2], x[it][3]};
        quad_layers<false>(y, l1[r], l0[2 * r], l0[2 * r + 1]);
#pragma unroll
        for (int k = 0; k < 4; k++) D[pos((r << n) + q + k * Q)] = y[k];
      }
    }
  }
  if (!FWD) return;
  __syncthreads();
  for (uint32_t s = n - 2; s > s_low;) {
    s -= 2;
    lds_step<false>(D, TF, N, s);
  }
  const bool al = ((uintptr_t)out & 15) == 0;
  for (uint32_t q = tid; q < 1u << (N - 2); q += nt) {
    const u32x4 v = *reinterpret_cast<const u32x4 *>(D + pos(4 * q));
    uint32_t y[4] = {v.x, v.y, v.z, v.w};
    low_layers<false>(y, TF, N, q, two);
    if (al) {
      gst4(out, q << 4, u32x4{y[0], y[1], y[2], y[3]});
    } else {
#pragma unroll
      for (int k = 0; k < 4; k++) gst(out, (4 * q + k) << 2, y[k]);
    }
  }
}

// The low pass (layers 0 .. 11 of a larger domain) of few columns: a workgroup
// of 1,024 lanes per 2^12 words, four words a lane, two layers at a time through
// LDS with the chunk's twiddles read beside its words.  The register pass gives a
// lane sixteen words and a workgroup 256, and reads its twiddles stage by stage:
// a quarter of the waves, each with four times the arithmetic between barriers.
// 512 of them (16 x 2^17): 12.4 us, here 11.1.
constexpr uint32_t kChunk = 12, kChunkQuads = 1u << (kChunk - 2);
struct ChunkLds {
  uint32_t T[1u << (kChunk - 1)], D[(1u << kChunk) / 16 * 17];
};
template <bool INV>
__device__ __forceinline__ void chunk_body(const FftPass2 &p, uint32_t wg, ChunkLds &S) {
  const uint32_t q = threadIdx.x, N = p.N, chunk = wg & ((1u << (N - kChunk)) - 1), col = wg >> (N - kChunk);
  // Words 2q and 2q + 1 of the chunk's part of every level, laid out as the
  // tree of a domain of 2^12: level s has 2^(11 - s) of them from 2^11 - 2^(12 - s) on.
  uint32_t t[2];
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const uint32_t i = 2 * q + k, r = (1u << (kChunk - 1)) - i;  // the last word is no level's
    const uint32_t s = kChunk - (32 - __clz(r - 1));
    t[k] = r < 2 ? 0u
                 : gld(p.tw_end - ((size_t)1 << (N - s)),
                       ((chunk << (kChunk - 1 - s)) + i - ((1u << (kChunk - 1)) - (1u << (kChunk - s)))) << 2);
  }
  const FftCol c = p.cols[col];
  const uint32_t *in = (const uint32_t *)readfirstlane_u64((uint64_t)(c.in + ((size_t)chunk << kChunk)));
  uint32_t *out = (uint32_t *)readfirstlane_u64((uint64_t)(c.out + ((size_t)chunk << kChunk)));
  uint32_t x[4];
  if (!INV) {
#pragma unroll
    for (int k = 0; k < 4; k++) x[k] = gld(in, (q + k * kChunkQuads) << 2);
  } else if (((uintptr_t)in & 15) == 0) {
    const u32x4 v = gld4(in, q << 4);
    x[0] = v.x;
    x[1] = v.y;
    x[2] = v.z;
    x[3] = v.w;
  } else {
#pragma unroll
    for (int k = 0; k < 4; k++) x[k] = gld(in, (4 * q + k) << 2);
  }
  S.T[2 * q] = t[0];
  S.T[2 * q + 1] = t[1];
  __syncthreads();
  const uint32_t *l0 = level(S.T, kChunk, kChunk - 2), *l1 = level(S.T, kChunk, kChunk - 1);
  if (INV) {
    low_layers<true>(x, S.T, kChunk, q, true);
    *reinterpret_cast<u32x4 *>(S.D + pos(4 * q)) = u32x4{x[0], x[1], x[2], x[3]};
    __syncthreads();
#pragma unroll
    for (uint32_t s = 2; s + 2 < kChunk; s += 2) lds_step<true>(S.D, S.T, kChunk, s);
#pragma unroll
    for (int k = 0; k < 4; k++) x[k] = S.D[pos(q + k * kChunkQuads)];
    quad_layers<true>(x, l1[0], l0[0], l0[1]);
    if (p.scale)
#pragma unroll
      for (int k = 0; k < 4; k++) x[k] = m31_mul(x[k], p.scale);
#pragma unroll
    for (int k = 0; k < 4; k++) gst(out, (q + k * kChunkQuads) << 2, x[k]);
    return;
  }
  quad_layers<false>(x, l1[0], l0[0], l0[1]);
#pragma unroll
  for (int k = 0; k < 4; k++) S.D[pos(q + k * kChunkQuads)] = x[k];
  __syncthreads();
#pragma unroll
  for (uint32_t s = kChunk - 4; s >= 2; s -= 2) lds_step<false>(S.D, S.T, kChunk, s);
  const u32x4 v = *reinterpret_cast<const u32x4 *>(S.D + pos(4 * q));
  uint32_t y[4] = {v.x, v.y, v.z, v.w};
  low_layers<false>(y, S.T, kChunk, q, true);
  if (((uintptr_t)out & 15) == 0) {
    gst4(out, q << 4, u32x4{y[0], y[1], y[2], y[3]});
  } else {
#pragma unroll
    for (int k = 0; k < 4; k++) gst(out, (4 * q + k) << 2, y[k]);
  }
}
template <bool INV>
__global__ void __launch_bounds__(kColMaxThreads) fft_chunk_kernel(FftPass2 p) {
  __shared__ __align__(16) ChunkLds S;
  chunk_body<INV>(p, blockIdx.x, S);
}
template <bool INV>
__global__ void __launch_bounds__(kColMaxThreads) fft_chunk_multi_kernel(const FftPass2 *groups,
                                                                         const uint32_t *wg_start, uint32_t n_groups) {
  __shared__ __align__(16) ChunkLds S;
  uint32_t g = 0, hi = n_groups;
  while (hi - g > 1) {
    const uint32_t mid = (g + hi) / 2;
    if (wg_start[mid] <= blockIdx.x) g = mid; else hi = mid;
  }
  const FftPass2 p = groups[g];
  chunk_body<INV>(p, blockIdx.x - wg_start[g], S);
}

__device__ __forceinline__ uint32_t column_group(const ColumnFft *groups, uint32_t n) {
  uint32_t g = 0, hi = n;
  while (hi - g > 1) {
    const uint32_t mid = (g + hi) / 2;
    if (groups[mid].wg_start <= blockIdx.x) g = mid; else hi = mid;
  }
  return g;
}

template <bool INV, bool FWD>
__global__ void __launch_bounds__(kColMaxThreads) column_fft_kernel(ColumnFft p) {
  extern __shared__ __align__(16) uint32_t S[];
  column_body<INV, FWD>(p, p.cols, blockIdx.x, S);
}
// The columns among the arguments: uploading them costs as much as the launch.
struct InlineFftCols {
  FftCol c[kInlineCols];
};
template <bool INV, bool FWD>
__global__ void __launch_bounds__(kColMaxThreads) column_fft_inline_kernel(ColumnFft p, InlineFftCols cols) {
  extern __shared__ __align__(16) uint32_t S[];
  column_body<INV, FWD>(p, cols.c, blockIdx.x, S);
}
template <bool INV, bool FWD>
__global__ void __launch_bounds__(kColMaxThreads) column_fft_multi_kernel(const ColumnFft *groups, uint32_t n_groups) {
  extern __shared__ __align__(16) uint32_t S[];
  const ColumnFft p = groups[column_group(groups, n_groups)];
  column_body<INV, FWD>(p, p.cols, blockIdx.x - p.wg_start, S);
}

dim3 threads(uint32_t N) { return dim3(std::min(kColMaxThreads, std::max(64u, 1u << (N - 2)))); }
// For every group of at most n and N: the twiddles of each transform, the words.
constexpr size_t lds_bytes(uint32_t n, uint32_t N, bool inv, bool fwd) {
  return ((inv ? (size_t)1 << (n - 1) : 0) + (fwd ? (size_t)1 << (N - 1) : 0) + ((size_t)1 << N) / 16 * 17 + 4) * 4;
}
static_assert(lds_bytes(kColMaxLog - 1, kColMaxLog, true, true) <= 59 << 10, "two workgroups of the largest a CU");
const char *name(bool inv, bool fwd) { return !fwd ? "ifft_pass_column" : inv ? "lde_pass_column" : "rfft_pass_column"; }

}  // namespace

// Up to 2^21 words in a launch the arithmetic stays behind the round trips
// (us, register passes -> here, extend_evals at blowup 2 of 2^n x columns):
// 2^8 x 16 31.7 -> 20.9; 2^10 x 16 35.8 -> 22.4, x 512 45.2 -> 33.0, x 2,048
// 62.4 -> 53.5; 2^11 x 1,024 58.5 -> 51.4, x 4,096 118 -> 125; 2^12 x 16 32.7 ->
// 29.2, x 512 53.1 -> 47.7 (from 1,024 on the matrix passes). 2^13 alone, one
// workgroup's largest: 32.9 -> 34.5.
bool column_fft_takes(const stwo_hip_ctx *ctx, uint32_t n, uint32_t N, size_t n_cols, bool inv, bool fwd,
                      bool batched) {
  if (n < 4 || n > 12 || N > kColMaxLog || n_cols << n > kColumnFftWords) return false;
  // At a large blowup a column is a long chain of a few lanes: 2^(n-2) of them write
  // its 2^(N-n) blocks one after another (of 2^4 words, four lanes of 64). Where
  // there are more columns than the CUs hold at once, that is the time (us, register
  // passes -> here; the line lies between the two of each size): 2^4 at blowup 2^5 x
  // 16,384 121 -> 121, x 32,768 155 -> 199; at 2^8 x 4,096 584 -> 512, x 8,192 590 -> 966;
  // 2^5 at 2^7 x 8,192 648 -> 478, x 16,384 675 -> 913; 2^6 at 2^5 x 16,384 196 -> 182, x
  // 32,768 264 -> 331.
  if (n_cols > (n == 4 ? 4096 : 8192) && n_cols << N > (size_t)1 << (n == 4 ? 23 : 25)) return false;
  // a vector plan chosen for the shape stands in a launch of its own (as in mx_plan)
  if (batched) return true;
  auto chosen = [&](uint32_t M, int inverse) {
    auto it = ctx->fft_tune.find(fft_tune_key(n, M, inverse));
    return it != ctx->fft_tune.end() && it->second.chosen;
  };
  return !(inv && chosen(n, 1)) && !(fwd && chosen(N, 0));
}

ColumnFft column_fft(const stwo_hip_twiddles *tw, const FftCol *d_cols, uint32_t n_cols, uint32_t n, uint32_t N,
                     bool store) {
  ColumnFft p{};
  p.cols = d_cols;
  p.itw_end = tw->d_itw2 + tw->len;
  p.tw_end = tw->d_tw2 + tw->len;
  p.n = n;
  p.N = N;
  p.scale = m31_inv((uint32_t)(((uint64_t)1 << n) % P));
  p.store = store;
  p.n_cols = n_cols;
  return p;
}

int run_column_fft(stwo_hip_ctx *ctx, const stwo_hip_twiddles *tw, const std::vector<FftCol> &cols, uint32_t n,
                   uint32_t N, bool store, bool inv, bool fwd) {
  ColumnFft p = column_fft(tw, nullptr, (uint32_t)cols.size(), n, N, store);
  const dim3 grid(p.n_cols), block = threads(N);
  const size_t lds = lds_bytes(n, N, inv, fwd);
  if (cols.size() <= kInlineCols) {
    InlineFftCols in{};
    std::copy(cols.begin(), cols.end(), in.c);
    if (!fwd) return launch(ctx, name(inv, fwd), column_fft_inline_kernel<true, false>, grid, block, lds, p, in);
    if (!inv) return launch(ctx, name(inv, fwd), column_fft_inline_kernel<false, true>, grid, block, lds, p, in);
    return launch(ctx, name(inv, fwd), column_fft_inline_kernel<true, true>, grid, block, lds, p, in);
  }
  void *d = nullptr;
  int rc = upload_table(ctx, cols.data(), cols.size() * sizeof(FftCol), &d);
  if (rc) return rc;
  p.cols = (const FftCol *)d;
  if (!fwd) return launch(ctx, name(inv, fwd), column_fft_kernel<true, false>, grid, block, lds, p);
  if (!inv) return launch(ctx, name(inv, fwd), column_fft_kernel<false, true>, grid, block, lds, p);
  return launch(ctx, name(inv, fwd), column_fft_kernel<true, true>, grid, block, lds, p);
}

bool fft_chunk_takes(const FftPass2 &p, uint32_t total_wgs) {
  return p.fixed == 1 && p.rep_log == 0 && p.in_log == p.N && total_wgs <= kChunkWgs;
}
int launch_fft_chunk(stwo_hip_ctx *ctx, bool inverse, const FftPass2 &p, uint32_t wgs) {
  const dim3 grid(wgs), block(kColMaxThreads);
  return inverse ? launch(ctx, "ifft_pass_chunk", fft_chunk_kernel<true>, grid, block, 0, p)
                 : launch(ctx, "rfft_pass_chunk", fft_chunk_kernel<false>, grid, block, 0, p);
}
int launch_fft_chunk_multi(stwo_hip_ctx *ctx, bool inverse, const FftPass2 *d_groups, const uint32_t *d_wg_start,
                           uint32_t n_groups, uint32_t total_wgs) {
  const dim3 grid(total_wgs), block(kColMaxThreads);
  return inverse ? launch(ctx, "ifft_pass_chunk", fft_chunk_multi_kernel<true>, grid, block, 0, d_groups, d_wg_start,
                          n_groups)
                 : launch(ctx, "rfft_pass_chunk", fft_chunk_multi_kernel<false>, grid, block, 0, d_groups, d_wg_start,
                          n_groups);
}

int launch_column_fft_multi(stwo_hip_ctx *ctx, const ColumnFft *d_groups, uint32_t n_groups, uint32_t wgs,
                            uint32_t max_n, uint32_t max_N, bool inv, bool fwd) {
  const dim3 grid(wgs), block = threads(max_N);
  const size_t lds = lds_bytes(max_n, max_N, inv, fwd);
  if (!fwd)
    return launch(ctx, name(inv, fwd), column_fft_multi_kernel<true, false>, grid, block, lds, d_groups, n_groups);
  if (!inv)
    return launch(ctx, name(inv, fwd), column_fft_multi_kernel<false, true>, grid, block, lds, d_groups, n_groups);
  return launch(ctx, name(inv, fwd), column_fft_multi_kernel<true, true>, grid, block, lds, d_groups, n_groups);
}

}  // namespace stwo_hip
