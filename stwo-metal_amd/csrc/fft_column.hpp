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
bool column_fft_takes(const stwo_hip_ctx *ctx, uint32_t n, uint32_t N, size_t n_cols, bool inv, bool fwd,
                      bool batched);
ColumnFft column_fft(const stwo_hip_twiddles *tw, const FftCol *d_cols, uint32_t n_cols, uint32_t n, uint32_t N,
                     bool store);
// One group, its columns given on the host.
int run_column_fft(stwo_hip_ctx *ctx, const stwo_hip_twiddles *tw, const std::vector<FftCol> &cols, uint32_t n,
                   uint32_t N, bool store, bool inv, bool fwd);
// n_groups groups from a table on the device; max_n, max_N: their largest n and N.
int launch_column_fft_multi(stwo_hip_ctx *ctx, const ColumnFft *d_groups, uint32_t n_groups, uint32_t wgs,
                            uint32_t max_n, uint32_t max_N, bool inv, bool fwd);

// The 12-layer low pass (FftPass2::fixed == 1) in workgroups of 1,024 lanes, for
// launches of at most kChunkWgs: up to there it is 1 to 8% ahead of the register
// pass in whole calls (us, interpolation / evaluation at blowup 2: 2^16 x 16 27.1
// -> 26.8 / 33.6 -> 31.4, 2^18 x 8 35.9 -> 34.8 / 45.3 -> 43.1); at 2,048 and more
// the device is full either way and the interpolation gains nothing (59.3 -> 59.2).
constexpr uint32_t kChunkWgs = 1024;
constexpr int kFftChunk = 13;  // launch_fft_multi's kind for it
bool fft_chunk_takes(const FftPass2 &p, uint32_t total_wgs);
int launch_fft_chunk(stwo_hip_ctx *ctx, bool inverse, const FftPass2 &p, uint32_t wgs);
int launch_fft_chunk_multi(stwo_hip_ctx *ctx, bool inverse, const FftPass2 *d_groups, const uint32_t *d_wg_start,
                           uint32_t n_groups, uint32_t total_wgs);

}  // namespace stwo_hip
