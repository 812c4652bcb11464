// Descriptors and launchers of the matrix FFT passes (fft_matrix.hip).
#pragma once
#include <stdint.h>

#include "common.hpp"
#include "internal.hpp"

namespace stwo_hip {

constexpr uint32_t kMxMinLog = 12;     // smallest transform: one chunk of the low pass
constexpr uint32_t kMxMaxLog = 24;     // largest: top 8 layers, at most 4 in between, low 12
constexpr uint32_t kMxMaxBlowup = 2;   // blowups the matrix table covers (0.7 MB; twice that a log further)

// The top 4 or 8 layers of a group of columns of 2^n coefficients.  Inverse:
// icols' in (evaluations) -> coefficients, stored to icols' out when `store`;
// forward: the 2^b output blocks of fcols' out, from the inverse's registers
// or, forward only, from fcols' in.
struct MxTop {
  const FftCol *icols, *fcols;
  const uint32_t *mats;  // the twiddle tree's matrix table
  uint32_t n_cols, n, b, store;
  uint32_t wgs;       // workgroups of the group (8 layers: each takes every wgs-th tile)
  uint32_t wg_start;  // first workgroup of the group in a launch over several
};

// Layers [0, t0) of 4,096-word chunks of columns of 2^N words; reads index
// g mod 2^in_log.
struct MxLow {
  const FftCol *cols;
  const uint32_t *tw_end, *tw2_end;  // ends of the (inverse) tree and of its doubled copy
  uint32_t n_cols, N, t0, in_log, scale;
  uint32_t iters;  // a workgroup takes one chunk of 4 * iters columns
  uint32_t wg_start;
};

// The passes of one group: top (layers > 0), the vector passes between (n >
// 20, from the group's vector plan) and low.
struct MxPlan {
  uint32_t top_layers = 0;  // 0: n = 12, the low pass alone
  uint32_t t0 = 12;
  bool mid = false;
};

// Low-pass units (4 columns x 2^12 words) from which the matrix passes pay alone.
constexpr uint64_t kMxMinUnits = 256;

// Whether a group's transform (log coefficients n, log blowup b; b = 0 for an
// interpolation) takes the matrix passes, alone or in a batched launch, and
// their split.
bool mx_plan(const stwo_hip_ctx *ctx, const stwo_hip_twiddles *tw, uint32_t n, uint32_t b, bool inverse, size_t n_cols,
             bool aligned16, bool batched, MxPlan *plan);
// A group's tiles (8-layer top pass; 0 for the 4-layer one) and chunks of 4
// columns (low pass); the sums over a launch's groups set how many of them a
// workgroup takes.
uint64_t mx_top_units(uint32_t n_cols, uint32_t n, const MxPlan &plan);
uint64_t mx_low_units(uint32_t n_cols, uint32_t N);
MxTop mx_top(const stwo_hip_twiddles *tw, const FftCol *icols, const FftCol *fcols, uint32_t n_cols, uint32_t n,
             uint32_t b, bool store, const MxPlan &plan, uint64_t launch_units, bool batched, uint32_t *wgs);
MxLow mx_low(const stwo_hip_twiddles *tw, const FftCol *cols, uint32_t n_cols, uint32_t n, uint32_t N, bool inverse,
             const MxPlan &plan, uint64_t launch_units, bool batched, uint32_t *wgs);
// d_groups: on the device, or NULL to run `one` alone.
int launch_mx_top(stwo_hip_ctx *ctx, const MxTop *one, const MxTop *d_groups, uint32_t n_groups, uint32_t total_wgs,
                  uint32_t layers, bool inv, bool fwd);
int launch_mx_low(stwo_hip_ctx *ctx, const MxLow *one, const MxLow *d_groups, uint32_t n_groups, uint32_t total_wgs,
                  bool inverse);

// The matrix table kept with a twiddle tree of this root (0: none).
size_t mx_table_bytes(uint32_t root_log);
int mx_table_build(stwo_hip_ctx *ctx, const uint32_t *tw_end, const uint32_t *itw_end, uint32_t *table);

}  // namespace stwo_hip
