// Evaluation of circle polynomials at a point of the secure-field circle
// (PolyOps::eval_at_point, STWO/prover/poly/circle/ops.rs; CpuBackend
// CPUB/circle.rs:82-99; Metal batch_eval_at_point, SH/eval_at_point.metal),
// the out-of-domain sampling step of the PCS.
//
// For coefficients c_0..c_{2^n - 1} (natural FFT-basis order) and the point
// (x, y), eval_at_point = fold(c, [pi^(n-2)(x), ..., pi(x), x, y])
// (STWO/core/poly/utils.rs:27-38), i.e. sum_j c_j * basis_j with
// basis_j = prod of g_k over the set bits k of j, g_0 = y, g_1 = x,
// g_k = pi^(k-1)(x), pi(x) = 2x^2 - 1.  The basis does not depend on the
// column: a workgroup of the one launch takes several 2^11-coefficient blocks of
// up to 8 columns of the same size, its lanes holding the low 2^11 basis values,
// forms the dot products (64-bit accumulation, one
// multiply-add per limb and coefficient), and multiplies by the product of
// g_k over the block index's bits; the last workgroup of a run of columns to
// finish sums the others' shares.  Sums of field elements are exact, so the
// grouping does not change the result.
#include <string.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "common.hpp"
#include "field.hpp"
#include "internal.hpp"
#include "merkle_dev.hpp"

namespace stwo_hip {

constexpr uint32_t kEvalBlockLog = 11;  // 2048 coefficients per workgroup and block

// A run of n <= kDotCols consecutive columns of one log size: the first of its
// workgroups, how many it has, and its shares' place (words).
constexpr uint32_t kDotCols = 8;
struct EvalRun {
  uint32_t col0, n, log_size, wg0, wgs, part;
};
struct EvalFactors {
  uint32_t g[32][4];  // g_0 = y, g_1 = x, g_k = pi^(k-1)(x)
};
static_assert(sizeof(EvalFactors) == 4 * kOodsFactorWords, "the device OODS point's factor layout");

__device__ __forceinline__ qm31 ld_factor(const EvalFactors *f, uint32_t k) {
  return qm31_make(f->g[k][0], f->g[k][1], f->g[k][2], f->g[k][3]);
}

// Workgroup w of its run takes blocks w, w + wgs, ... (2^B coefficients each, B =
// min(log, kEvalBlockLog)) of the run's columns.  Lane t holds
// the basis values of coefficients 4t .. 4t + 3 and 1024 above in registers and, per
// column, accumulates sum c_j * basis_j limb by limb in 64 bits
// (v_mad_u64_u32; each product is at most P^2, so four fit, also on top of a fold
// (x & P) + (x >> 31) of the four before, which is below 2^34).  The 256 lanes' sums
// are reduced through LDS, multiplied by the block's factor and added to the
// workgroup's share, while the next block's loads are on their way.
//
// Bound by the multiply-adds and the loads under them, three workgroups a CU:
// 264 columns of 2^18 (277 MB) take 78 us and 3.5 KB of tables.  In three launches
// (the basis, a workgroup per block and run, the sums) it was 7.4 + 72.7 + 5.1 us
// and the gaps between them, with a table entry per block and run (68 KB).
constexpr uint32_t kEvalFactorBlocks = 64;  // blocks whose factors are held at once
struct EvalLds {
  uint32_t red[kDotCols * 4][257];
  uint32_t sums[kDotCols * 4];
  uint32_t low[2][16][4];                 // basis of index bits 2..5 and 6..9
  uint32_t fac[kEvalFactorBlocks][4];
  uint32_t last;
};
__device__ __forceinline__ qm31 ld_qm31(const uint32_t *p) { return qm31_make(p[0], p[1], p[2], p[3]); }

__global__ void __launch_bounds__(256) eval_point_kernel(const uint32_t *const *cols, const EvalRun *runs,
                                                         uint32_t n_runs, const EvalFactors *f, uint32_t *partials,
                                                         uint32_t *counters, uint32_t *out) {
  __shared__ EvalLds S;
  const uint32_t tid = threadIdx.x;
  uint32_t ri = 0, hi = n_runs;
  while (hi - ri > 1) {
    const uint32_t mid = (ri + hi) / 2;
    if (runs[mid].wg0 <= blockIdx.x) ri = mid; else hi = mid;
  }
  const EvalRun R = runs[ri];
  const uint32_t w = blockIdx.x - R.wg0, n = R.n;
  const uint32_t B = R.log_size < kEvalBlockLog ? R.log_size : kEvalBlockLog, nb = 1u << B;
  const uint32_t n_blocks = 1u << (R.log_size - B), t0 = tid * 4, t1 = t0 + 1024;
  // 8 words per lane and column, as two 16-byte loads when the block is
  // whole and the column pointer 16-byte aligned (a wave-uniform test).
  uint32_t cv[kDotCols][8];
  auto load = [&](uint32_t block) {
#pragma unroll
    for (uint32_t j = 0; j < kDotCols; j++) {
      if (j < n) {
        const uint32_t *c = cols[R.col0 + j] + ((size_t)block << B);
        if (nb == (1u << kEvalBlockLog) && ((uintptr_t)c & 15) == 0) {
          const u32x4 lo = *(gconst_u4 *)(as_global(c) + t0), h4 = *(gconst_u4 *)(as_global(c) + t1);
          cv[j][0] = lo.x;
          cv[j][1] = lo.y;
          cv[j][2] = lo.z;
          cv[j][3] = lo.w;
          cv[j][4] = h4.x;
          cv[j][5] = h4.y;
          cv[j][6] = h4.z;
          cv[j][7] = h4.w;
        } else {
#pragma unroll
          for (int i = 0; i < 8; i++) {
            const uint32_t t = i < 4 ? t0 + i : t1 + i - 4;
            cv[j][i] = t < nb ? as_global(c)[t] : 0;
          }
        }
      }
    }
  };
  load(w);
  // Factors of blocks w + k wgs: bit i of the block index selects g_{B + i}.
  auto factors = [&](uint32_t first) {
    const uint32_t block = first + (tid & (kEvalFactorBlocks - 1)) * R.wgs;
    if (tid >= kEvalFactorBlocks || block >= n_blocks) return;
    qm31 r = qm31_make(1, 0, 0, 0);
    for (uint32_t k = B; k < R.log_size; k++)
      if ((block >> (k - B)) & 1) r = qm31_mul(r, ld_factor(f, k));
    for (int k = 0; k < 4; k++) S.fac[tid][k] = r.v[k];
  };
  // The basis: of index bits 2..5 and 6..9 by 32 lanes, their products and
  // those of bits 0, 1 and 10 in every lane.
  if (tid >= 128 && tid < 160) {
    const uint32_t half = (tid >> 4) & 1, e = tid & 15;
    qm31 r = qm31_make(1, 0, 0, 0);
    for (uint32_t k = 0; k < 4; k++)
      if ((e >> k) & 1) r = qm31_mul(r, ld_factor(f, 2 + 4 * half + k));
    for (int k = 0; k < 4; k++) S.low[half][e][k] = r.v[k];
  }
  factors(w);
  __syncthreads();
  qm31 b[8];
  b[0] = qm31_mul(ld_qm31(S.low[0][tid & 15]), ld_qm31(S.low[1][tid >> 4]));
#pragma unroll
  for (int k = 0; k < 3; k++)
#pragma unroll
    for (int i = 0; i < (1 << k); i++) b[(1 << k) + i] = qm31_mul(b[i], ld_factor(f, k < 2 ? k : 10));
  qm31 share = qm31_make(0, 0, 0, 0);
  uint32_t k_blk = 0;
  for (uint32_t block = w; block < n_blocks; block += R.wgs) {
#pragma unroll
    for (uint32_t j = 0; j < kDotCols; j++) {
      if (j >= n) break;
      uint64_t acc[4] = {0, 0, 0, 0};
#pragma unroll
      for (int i = 0; i < 8; i++) {
#pragma unroll
        for (int k = 0; k < 4; k++) acc[k] += (uint64_t)cv[j][i] * b[i].v[k];
        if (i == 3)
#pragma unroll
          for (int k = 0; k < 4; k++) acc[k] = m31_fold64(acc[k]);
      }
#pragma unroll
      for (int k = 0; k < 4; k++) S.red[4 * j + k][tid] = m31_reduce64(acc[k]);
    }
    if (block + R.wgs < n_blocks) load(block + R.wgs);
    __syncthreads();
    // Row r (column r / 4, limb r % 4): 8 lanes sum 32 entries each, then
    // combine across the 8 lanes (consecutive lanes of one wave).
    const uint32_t r = tid >> 3, seg = tid & 7;
    if (r < 4 * n) {
      uint64_t s = 0;
#pragma unroll
      for (int i = 0; i < 32; i++) s += S.red[r][seg * 32 + i];
      uint32_t v = m31_reduce64(s);
#pragma unroll
      for (int o = 1; o < 8; o <<= 1) v = m31_add(v, __shfl_xor(v, o, 8));
      if (seg == 0) S.sums[r] = v;
    }
    __syncthreads();
    if (tid < n) share = qm31_add(share, qm31_mul(ld_qm31(S.sums + 4 * tid), ld_qm31(S.fac[k_blk])));
    if (++k_blk == kEvalFactorBlocks) {
      k_blk = 0;
      __syncthreads();
      factors(block + R.wgs);  // seen after the next block's first barrier
    }
  }
  if (R.wgs == 1) {
    if (tid < n)
      for (int k = 0; k < 4; k++) out[4 * (size_t)(R.col0 + tid) + k] = share.v[k];
    return;
  }
  // The last workgroup of the run to count itself sums the shares (stored and
  // loaded at agent scope, complete before the count) and clears the counter.
  uint32_t *part = partials + R.part;
  if (tid < n)
    for (int k = 0; k < 4; k++) st_agent(part + ((size_t)w * n + tid) * 4 + k, share.v[k]);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    const uint32_t old =
        __hip_atomic_fetch_add(counters + ri, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t last = old + 1 == R.wgs;
    if (last) st_agent(counters + ri, 0);
    S.last = last;
  }
  __syncthreads();
  if (!S.last) return;
  const uint32_t j = tid >> 5, lane = tid & 31;  // 32 lanes a column
  if (j >= n) return;
  qm31 sum = qm31_make(0, 0, 0, 0);
  for (uint32_t i = lane; i < R.wgs; i += 32) {
    const uint32_t *p = part + ((size_t)i * n + j) * 4;
    sum = qm31_add(sum, qm31_make(ld_agent(p), ld_agent(p + 1), ld_agent(p + 2), ld_agent(p + 3)));
  }
#pragma unroll
  for (int o = 1; o < 32; o <<= 1)
#pragma unroll
    for (int k = 0; k < 4; k++) sum.v[k] = m31_add(sum.v[k], __shfl_xor(sum.v[k], o, 32));
  if (lane == 0)
    for (int k = 0; k < 4; k++) out[4 * (size_t)(R.col0 + j) + k] = sum.v[k];
}

// ---- fixed scratch for the entry point that allocates nothing -------------
//
// stwo_hip_eval_at_point_noalloc keeps its workgroups' shares and the
// per-column sums in this file-scope array (one copy per device, held until
// the process ends) instead of buffers it would allocate.  Layout in words:
// sums [0, 4 n_cols), shares after them.  The call's limit counts a share per
// column and block and 2^13 words besides, more than it now takes.  Host code never passes the array's name to a kernel or a copy (on
// the host it is only a stand-in for the symbol): it uses the per-device
// address that hipGetSymbolAddress returned at context creation.
constexpr size_t kNaScratchWords = 1u << 18;  // 1 MiB
constexpr size_t kNaReserved = (size_t)4 << kEvalBlockLog;
static __device__ __align__(256) uint32_t scratch[kNaScratchWords];

constexpr int kMaxDevices = 64;
static std::mutex g_na_mu;
static uint32_t *g_na_ptr[kMaxDevices];

}  // namespace stwo_hip

namespace stwo_hip {

// Resolves this device's address of `scratch` (the device is current).
// Called once per device, from context creation.
int eval_point_scratch_setup(stwo_hip_ctx *ctx) {
  const int dev = ctx->device;
  if (dev < 0 || dev >= kMaxDevices)
    return set_error(ctx, STWO_HIP_EDEVICE, "device %d beyond the %d the library supports", dev, kMaxDevices);
  std::lock_guard<std::mutex> lk(g_na_mu);
  if (g_na_ptr[dev]) return STWO_HIP_OK;
  void *ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr)
    return set_error(ctx, STWO_HIP_EDEVICE, "hipGetSymbolAddress(scratch) on device %d: %s", dev,
                     hipGetErrorString(e));
  g_na_ptr[dev] = (uint32_t *)ptr;
  return STWO_HIP_OK;
}

// `na_scratch`: NULL = buffers from the context's scratch pool (allocated on
// first use or growth); otherwise the fixed per-device array, with every
// size checked against it and no allocating call made.  `d_factors`: the
// point's factors already on the device (EvalFactors layout), `point` unused;
// `d_values`: the values stay on the device there (4 words per column),
// `values` unused.
static int eval_at_point_impl(stwo_hip_ctx *ctx, const uint32_t *const *coeffs, const uint32_t *log_sizes,
                              size_t n_cols, const stwo_hip_secure_point *point, uint32_t *values,
                              uint32_t *na_scratch, const uint32_t *d_factors = nullptr,
                              uint32_t *d_values = nullptr) {
  if (!ctx) return STWO_HIP_EINVAL;
  STWO_HIP_CHECK_ARG(ctx, (point || d_factors) && (values || d_values) && (coeffs || !n_cols) &&
                              (log_sizes || !n_cols),
                     "eval_at_point: NULL argument");
  if (n_cols == 0) return STWO_HIP_OK;
  STWO_HIP_CHECK_ARG(ctx, n_cols <= 65536, "eval_at_point: %zu columns in one call (at most 65536)", n_cols);
  uint64_t total = 0;
  uint32_t max_log = 0;
  for (size_t c = 0; c < n_cols; c++) {
    STWO_HIP_CHECK_ARG(ctx, coeffs[c] && log_sizes[c] <= 30, "eval_at_point: column %zu invalid", c);
    total += 1ull << (log_sizes[c] > kEvalBlockLog ? log_sizes[c] - kEvalBlockLog : 0);
    max_log = std::max(max_log, log_sizes[c]);
  }
  STWO_HIP_CHECK_ARG(ctx, total < (1ull << 31), "eval_at_point: too many blocks");
  // Factors g_0 = y, g_1 = x, g_k = pi^(k-1)(x) (CPUB/circle.rs:82-99).
  EvalFactors f{};
  if (!d_factors) {
    qm31 x = qm31_make(point->x[0], point->x[1], point->x[2], point->x[3]);
    memcpy(f.g[0], point->y, 16);
    for (uint32_t k = 1; k < 32 && k < max_log + 1; k++) {
      memcpy(f.g[k], x.v, 16);
      qm31 sq = qm31_mul(x, x);
      x = qm31_sub(qm31_add(sq, sq), qm31_make(1, 0, 0, 0));
    }
  }
  // Runs of up to kDotCols consecutive columns of one log size, each with
  // workgroups for an equal share of the blocks: about three a CU in all (as many
  // as their registers allow), one where the runs alone are more than the counters.
  std::vector<EvalRun> runs;
  uint64_t n_work = 0;  // blocks over all runs
  for (size_t c = 0; c < n_cols;) {
    size_t e = c + 1;
    while (e < n_cols && e - c < kDotCols && log_sizes[e] == log_sizes[c]) e++;
    runs.push_back({(uint32_t)c, (uint32_t)(e - c), log_sizes[c], 0, 0, 0});
    n_work += 1ull << (log_sizes[c] > kEvalBlockLog ? log_sizes[c] - kEvalBlockLog : 0);
    c = e;
  }
  const uint64_t per = (n_work + 767) / 768;
  uint32_t wgs = 0;
  size_t shares = 0;
  for (EvalRun &r : runs) {
    const uint64_t nblk = 1ull << (r.log_size > kEvalBlockLog ? r.log_size - kEvalBlockLog : 0);
    r.wg0 = wgs;
    r.wgs = runs.size() > kTreeCounters ? 1 : (uint32_t)((nblk + per - 1) / per);
    r.part = (uint32_t)shares;
    wgs += r.wgs;
    shares += (size_t)r.wgs * r.n * 4;
  }
  if (na_scratch) {
    // Everything must fit the fixed array, and the tables the ring arena
    // (larger ones would take an allocated buffer).
    STWO_HIP_CHECK_ARG(ctx, kNaReserved + 4 * ((uint64_t)n_cols + total) <= kNaScratchWords,
                       "eval_at_point_noalloc: %zu columns and %llu blocks of 2^11 coefficients need %llu words of "
                       "scratch, more than the %zu available",
                       n_cols, (unsigned long long)total,
                       (unsigned long long)(kNaReserved + 4 * ((uint64_t)n_cols + total)), kNaScratchWords);
    STWO_HIP_CHECK_ARG(ctx,
                       16 * (n_cols + n_work) + sizeof(EvalFactors) + 512 <= ctx->arena_cap / 2,
                       "eval_at_point_noalloc: %zu work items exceed the table arena", (size_t)n_work);
  }
  void *d_tab = nullptr, *d_runs = nullptr, *d_part = nullptr, *d_out = nullptr;
  const EvalFactors *d_f = (const EvalFactors *)d_factors;
  int rc;
  {
    const void *srcs[3] = {coeffs, runs.data(), &f};
    const size_t bytes[3] = {n_cols * sizeof(*coeffs), runs.size() * sizeof(EvalRun), sizeof f};
    void *d[3];
    // with the point on the device (the prove) the tables repeat from call to call
    rc = (d_factors && !na_scratch) ? upload_tables_cached(ctx, "eval_at_point", 2, srcs, bytes, d)
                                    : upload_tables(ctx, d_factors ? 2 : 3, srcs, bytes, d);
    if (rc) return rc;
    d_tab = d[0];
    d_runs = d[1];
    if (!d_factors) d_f = (const EvalFactors *)d[2];
  }
  if (na_scratch) {
    d_out = na_scratch;
    d_part = na_scratch + 4 * n_cols;
  } else {
    rc = get_scratch(ctx, "eval_point_partials", shares * 4, &d_part);
    if (rc) return rc;
    rc = get_scratch(ctx, "eval_point_out", n_cols * 16, &d_out);
    if (rc) return rc;
  }
  if (d_values) d_out = d_values;
  rc = launch(ctx, "eval_at_point", eval_point_kernel, dim3(wgs), dim3(256), 0, (const uint32_t *const *)d_tab,
              (const EvalRun *)d_runs, (uint32_t)runs.size(), d_f, (uint32_t *)d_part, ctx->d_counters,
              (uint32_t *)d_out);
  if (rc) return rc;
  if (d_values) return STWO_HIP_OK;
  return stwo_hip_download(ctx, values, (const uint32_t *)d_out, 4 * n_cols);
}

int eval_at_point_dev(stwo_hip_ctx *ctx, const uint32_t *const *coeffs, const uint32_t *log_sizes, size_t n_cols,
                      const uint32_t *d_factors, uint32_t *d_values) {
  if (!ctx) return STWO_HIP_EINVAL;
  STWO_HIP_CHECK_ARG(ctx, d_factors && d_values, "eval_at_point: NULL device factors or values");
  return eval_at_point_impl(ctx, coeffs, log_sizes, n_cols, nullptr, nullptr, nullptr, d_factors, d_values);
}

}  // namespace stwo_hip

using namespace stwo_hip;

extern "C" {

int stwo_hip_eval_at_point(stwo_hip_ctx *ctx, const uint32_t *const *coeffs, const uint32_t *log_sizes, size_t n_cols,
                           const stwo_hip_secure_point *point, uint32_t *values) {
  return eval_at_point_impl(ctx, coeffs, log_sizes, n_cols, point, values, nullptr);
}

int stwo_hip_eval_at_point_noalloc(stwo_hip_ctx *ctx, const uint32_t *const *coeffs, const uint32_t *log_sizes,
                                   size_t n_cols, const stwo_hip_secure_point *point, uint32_t *values) {
  if (!ctx) return STWO_HIP_EINVAL;
  uint32_t *ptr = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_na_mu);
    if (ctx->device >= 0 && ctx->device < kMaxDevices) ptr = g_na_ptr[ctx->device];
  }
  STWO_HIP_CHECK_ARG(ctx, ptr != nullptr, "eval_at_point_noalloc: scratch of device %d not set up", ctx->device);
  int rc = arena_quiesce(ctx);
  if (rc) return rc;
  return eval_at_point_impl(ctx, coeffs, log_sizes, n_cols, point, values, ptr);
}

}  // extern "C"
