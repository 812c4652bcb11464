// Transforms of few small columns, one workgroup per column (fft_column.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "common.hpp"
#include "internal.hpp"

namespace stwo_hip {

// A group of columns: interpolation (N = n), evaluation, or both.
struct ColumnFft {
  // {column, its evaluations}: interpolated in place, evaluated, or both
  const FftCol *cols;
  const uint32_t *itw_end, *tw_end;  // ends of the doubled trees
  uint32_t n, N;
  uint32_t scale, store;  // 1 / 2^n; store: keep the coefficients of an LDE
  uint32_t n_cols, wg_start;
};

// Coefficients in one launch at most.
constexpr size_t kColumnFftWords = (size_t)1 << 21;
// Whether a group is taken (alone, or at the side of others in one launch).
bool column_fft_takes(const stwo_hip_ctx *ctx, uint32_t n, uint32_t N, size_t n_cols, bool inv, bool fwd);
ColumnFft column_fft(const stwo_hip_twiddles *tw, const FftCol *d_cols, uint32_t n_cols, uint32_t n, uint32_t N,
                     bool store);
// One group, its columns given on the host.
int run_column_fft(stwo_hip_ctx *ctx, const stwo_hip_twiddles *tw, const std::vector<FftCol> &cols, uint32_t n,
                   uint32_t N, bool store, bool inv, bool fwd);
// n_groups groups from a table on the device; max_N: their largest N.
int launch_column_fft_multi(stwo_hip_ctx *ctx, const ColumnFft *d_groups, uint32_t n_groups, uint32_t wgs,
                            uint32_t max_N, bool inv, bool fwd);

}  // namespace stwo_hip
