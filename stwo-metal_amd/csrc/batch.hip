// Batched LDE + Merkle commitment of columns of uneven sizes.
//
// The plain path dispatches per column (the reference's evaluate_polynomials
// submits one RFFT per column, MB/poly.rs:715-779, and its IFFT one per
// column, MB/poly.rs:364-391).  Here a plan covers a whole column set:
//   - columns are grouped by log size; each group's FFT is a list of passes
//     (radix-16, see fft.hip); passes of the same level from every group run
//     in ONE launch (fft_pass_multi_kernel), so the IFFT and the RFFT take
//     2-3 launches each whatever the number of sizes;
//   - the Merkle tree is built layer by layer: mixed degree injects the
//     evaluations of each size at their own layer (MerkleProver::commit,
//     STWO/prover/vcs/prover.rs:39-65), lifted hashes all columns into the
//     leaves (MerkleProverLifted::commit, STWO/prover/vcs_lifted/prover.rs:33-44);
//   - every table (column pointers, pass descriptors) is uploaded once at
//     plan time into plan-owned device memory, so the launch sequence has no
//     host-to-device copies and can be captured into a hipGraph and replayed.
#include <string.h>

#include <algorithm>
#include <functional>
#include <map>
#include <tuple>
#include <vector>

#include "common.hpp"
#include "fft_column.hpp"
#include "fft_matrix.hpp"
#include "field.hpp"
#include "internal.hpp"

struct stwo_hip_batch {
  int device = 0;
  void *d_mem = nullptr;
  bool mem_from_job = false;  // tables carved from a serving job's memory block
  std::function<int(stwo_hip_ctx *)> issue;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  size_t n_launches = 0;
};

namespace stwo_hip {

namespace {

// Bump allocator over one host staging vector mirrored by one device buffer.
struct Staging {
  std::vector<uint8_t> host;
  size_t put(const void *src, size_t bytes) {
    size_t off = (host.size() + 255) & ~(size_t)255;
    host.resize(off + bytes);
    memcpy(host.data() + off, src, bytes);
    return off;
  }
};

struct LevelLaunch {
  bool inverse;
  bool fused;  // the fused IFFT-last + RFFT-first pass (groups_off: IFFT descriptors, fwd_off: RFFT ones)
  int kind;  // launch_fft_multi's (or launch_lde_multi's) schedule kind for every group of the launch
  size_t groups_off, fwd_off, wgs_off;  // offsets into the device buffer
  uint32_t n_groups, total_wgs, wg_log;
  // matrix passes (groups_off: MxTop or MxLow descriptors): layers of a top
  // pass with its directions, or the low pass (mx_layers = 0)
  bool matrix = false, mx_inv = false, mx_fwd = false;
  uint32_t mx_layers = 0;
  // a workgroup per column (groups_off: ColumnFft descriptors), largest n and N
  uint32_t column_n = 0, column_N = 0;
};

// One tree's layer tables and shape.
struct TreeLaunches {
  struct LayerTab {
    uint32_t log_size;
    size_t off;
    uint32_t count;
  };
  std::vector<LayerTab> lt;
  uint32_t *layers;
  uint32_t max_log;
  int mode, kind;
  size_t counters_off;
};
// Steps of several trees in one launch, or one step alone (n = 1, by value).
struct TreeWave {
  MerkleStep step;
  size_t off;
  uint32_t n, wgs;
};

// One group of same-size columns: its tables' places in the staging.
struct GroupTabs {
  uint32_t n, b;
  int stage;
  size_t ifft_off, rfft_off, inplace_off;
  uint32_t count;
  bool aligned16;  // every column pointer of the group is 16-byte aligned
};

// A group of columns {in, out} (in place but for the evaluations).
GroupTabs put_group(Staging &st, uint32_t n, uint32_t b, int stage, const std::vector<FftCol> &cols) {
  std::vector<FftCol> a, c;
  GroupTabs t{};
  t.n = n;
  t.b = b;
  t.stage = stage;
  t.count = (uint32_t)cols.size();
  t.aligned16 = true;
  for (const FftCol &f : cols) {
    if (stage != BATCH_RFFT) a.push_back({f.in, (uint32_t *)f.in});
    c.push_back({f.out, f.out});
    if ((((uintptr_t)f.in) | ((uintptr_t)f.out)) & 15) t.aligned16 = false;
  }
  if (stage != BATCH_RFFT) t.ifft_off = st.put(a.data(), a.size() * sizeof(FftCol));
  if (stage != BATCH_IFFT) {
    t.rfft_off = st.put(cols.data(), cols.size() * sizeof(FftCol));
    t.inplace_off = st.put(c.data(), c.size() * sizeof(FftCol));
  } else {
    t.rfft_off = t.inplace_off = t.ifft_off;
  }
  return t;
}

// Upper bound on the descriptors that build_levels adds: one per group and pass
// (2 directions, at most 4 passes), plus the 256-byte alignment of two or three
// tables per launch (2 directions x 4 levels x 2 workgroup sizes x at most 14
// schedule kinds, and the fused launches).
size_t levels_bound(size_t n_groups) {
  return n_groups * (sizeof(MxTop) + 2 * sizeof(MxLow) + sizeof(ColumnFft)) + 14 * 256 + 2 * 4 * n_groups * (sizeof(FftPass2) + 8) +
         2 * 4 * 2 * 14 * 2 * 256 + 8192;
}

// Two workgroups of the vector passes a CU, half of what it holds (16 KB
// of LDS and 256 lanes each).
constexpr uint64_t kShareWgs = 512;

// The launches of the groups' transforms, over their tables and the descriptors
// put after them, all at dbase once uploaded.  drop: the fused passes need not
// store the coefficients.  matrix: groups that can take the matrix passes do.
int build_levels(stwo_hip_ctx *ctx, const stwo_hip_twiddles *tw, const std::vector<GroupTabs> &gt, uint8_t *dbase,
                 bool store_coeffs, bool matrix, Staging &st, std::vector<LevelLaunch> &levels) {
  // The radix-16 passes take the doubled trees.
  const uint32_t *itw_end = tw->d_itw2 + tw->len, *tw_end = tw->d_tw2 + tw->len;
  // Both transforms' passes of every group; where the IFFT's last pass and
  // the RFFT's first pass tile alike they become one fused pass.
  struct GroupPasses {
    std::vector<PassLaunch> inv, fwd;
    bool fused = false;
    bool matrix = false;  // first and last passes on the matrix cores
    bool column = false;  // a workgroup per column
    MxPlan mx;
  };
  std::vector<GroupPasses> gp(gt.size());
  // The smallest sizes take a workgroup per column, up to what one launch of
  // them may hold (the groups come largest first).
  size_t column_words = 0;
  for (size_t gi = gt.size(); gi-- > 0;) {
    const GroupTabs &t = gt[gi];
    const bool inv = t.stage != BATCH_RFFT, fwd = t.stage != BATCH_IFFT;
    const uint32_t N = t.n + (fwd ? t.b : 0);
    MxPlan mx;
    if (!column_fft_takes(ctx, t.n, N, t.count, inv, fwd, true) || column_words + ((size_t)t.count << t.n) > kColumnFftWords ||
        (matrix && (!inv || mx_plan(ctx, tw, t.n, 0, true, t.count, t.aligned16, true, &mx)) &&
         (!fwd || mx_plan(ctx, tw, t.n, t.b, false, t.count, t.aligned16, true, &mx))))
      continue;
    gp[gi].column = true;
    column_words += (size_t)t.count << t.n;
  }
  for (size_t gi = 0; gi < gt.size(); gi++) {
    const GroupTabs &t = gt[gi];
    if (gp[gi].column) continue;
    for (int dir = 0; dir < 2; dir++) {
      const bool inverse = dir == 0;
      if ((inverse && t.stage == BATCH_RFFT) || (!inverse && t.stage == BATCH_IFFT)) continue;
      const uint32_t n = t.n, N = t.n + (inverse ? 0 : t.b);
      const FftCol *first = (const FftCol *)(dbase + (inverse ? t.ifft_off : t.rfft_off));
      const FftCol *inpl = (const FftCol *)(dbase + t.inplace_off);
      int rc = make_group_passes(ctx, inverse ? N : n, N, inverse, first, inpl, t.count, inverse ? itw_end : tw_end,
                                 t.aligned16, inverse ? gp[gi].inv : gp[gi].fwd);
      if (rc) return rc;
    }
    GroupPasses &G = gp[gi];
    const bool has_inv = t.stage != BATCH_RFFT, has_fwd = t.stage != BATCH_IFFT;
    if (matrix &&
        (!has_inv || mx_plan(ctx, tw, t.n, 0, true, t.count, t.aligned16, true, &G.mx)) &&
        (!has_fwd || mx_plan(ctx, tw, t.n, t.b, false, t.count, t.aligned16, true, &G.mx))) {
      G.matrix = true;
      // what is left to the vector passes: the default plan's middle pass
      const FftTune def;
      for (int dir = 0; dir < 2; dir++) {
        std::vector<PassLaunch> &v = dir ? G.fwd : G.inv;
        if (v.empty()) continue;
        if (!G.mx.mid) {
          v.clear();
          continue;
        }
        const FftCol *in_place = (const FftCol *)(dbase + (dir ? t.inplace_off : t.ifft_off));
        int rc = make_group_passes(ctx, t.n, t.n + (dir ? t.b : 0), !dir, in_place, in_place, t.count,
                                   dir ? tw_end : itw_end, true, v, &def);
        if (!rc && v.size() != 3) rc = set_error(ctx, STWO_HIP_EINVAL, "internal: %zu passes of 2^%u", v.size(), t.n);
        if (rc) return rc;
        v = {v[1]};
      }
      continue;
    }
    gp[gi].fused = t.stage == BATCH_LDE && lde_fusable(gp[gi].inv.back(), gp[gi].fwd.front(), t.b);
  }
  auto add_level = [&](bool inverse, uint32_t wg_log, std::vector<PassLaunch> &v) -> int {
    // Groups whose pass matches a compile-time schedule get a launch per
    // schedule with that schedule's kernel; the rest share one.  Schedules that
    // together do not fill the device once (kShareWgs) share the run-time
    // schedule's launch instead: a launch costs more than the schedule gains
    // there (six schedules of 512 workgroups in all: 27 us in six launches, 12 us in
    // one).
    std::map<uint32_t, uint64_t> kinds;  // schedule -> workgroups
    for (auto &pl : v) kinds[pl.p.fixed] += pl.wgs;
    std::vector<std::pair<uint64_t, uint32_t>> by_wgs;
    for (auto &k : kinds) by_wgs.push_back({k.second, k.first});
    std::sort(by_wgs.begin(), by_wgs.end());
    uint64_t small = 0;
    std::vector<std::vector<uint32_t>> launches(1);
    for (auto &k : by_wgs)
      if ((small += k.first) <= kShareWgs)
        launches[0].push_back(k.second);
      else
        launches.push_back({k.second});
    for (const std::vector<uint32_t> &kds : launches) {
      const uint32_t kd = kds.size() == 1 ? kds[0] : 0;
      std::vector<FftPass2> descs;
      std::vector<uint32_t> starts;
      uint64_t acc = 0;
      bool uniform = true;
      for (auto &pl : v) {
        if (std::find(kds.begin(), kds.end(), pl.p.fixed) == kds.end()) continue;
        descs.push_back(pl.p);
        starts.push_back((uint32_t)acc);
        acc += pl.wgs;
        if (pl.p.T < 10) uniform = false;
      }
      if (descs.empty()) continue;
      if (acc >= (1ull << 31)) return set_error(ctx, STWO_HIP_EINVAL, "FFT groups too large for one launch");
      LevelLaunch ll{};
      ll.inverse = inverse;
      ll.fused = false;
      ll.kind = kd != 0 ? (int)kd : (uniform ? -1 : 0);
      if (kd == 1 && std::all_of(descs.begin(), descs.end(),
                                 [&](const FftPass2 &p) { return fft_chunk_takes(p, (uint32_t)acc); }))
        ll.kind = kFftChunk;
      ll.groups_off = st.put(descs.data(), descs.size() * sizeof(FftPass2));
      ll.wgs_off = st.put(starts.data(), starts.size() * sizeof(uint32_t));
      ll.n_groups = (uint32_t)descs.size();
      ll.total_wgs = (uint32_t)acc;
      ll.wg_log = wg_log;
      levels.push_back(ll);
    }
    return STWO_HIP_OK;
  };
  // The matrix passes of every group that takes them.  The low pass is the
  // first of the inverse levels and the last of the forward ones; the top pass
  // runs after the inverse levels, fused with the forward one where the set
  // has both.
  auto add_mx_low = [&](bool inverse) -> int {
    uint64_t units = 0, acc = 0;
    auto takes = [&](size_t gi) { return gp[gi].matrix && gt[gi].stage != (inverse ? BATCH_RFFT : BATCH_IFFT); };
    for (size_t gi = 0; gi < gt.size(); gi++)
      if (takes(gi)) units += mx_low_units(gt[gi].count, gt[gi].n + (inverse ? 0 : gt[gi].b));
    std::vector<MxLow> descs;
    for (size_t gi = 0; gi < gt.size(); gi++) {
      if (!takes(gi)) continue;
      const GroupTabs &t = gt[gi];
      const size_t tab = inverse ? t.ifft_off : gp[gi].mx.top_layers ? t.inplace_off : t.rfft_off;
      uint32_t wgs = 0;
      descs.push_back(mx_low(tw, (const FftCol *)(dbase + tab), t.count, t.n, t.n + (inverse ? 0 : t.b), inverse,
                             gp[gi].mx, units, true, &wgs));
      descs.back().wg_start = wgs;
    }
    if (descs.empty()) return STWO_HIP_OK;
    // the longest workgroups start first
    std::stable_sort(descs.begin(), descs.end(), [](const MxLow &a, const MxLow &c) { return a.iters > c.iters; });
    for (MxLow &d : descs) {
      const uint32_t wgs = d.wg_start;
      d.wg_start = (uint32_t)acc;
      acc += wgs;
    }
    if (acc >= (1ull << 31)) return set_error(ctx, STWO_HIP_EINVAL, "FFT groups too large for one launch");
    LevelLaunch ll{};
    ll.inverse = inverse;
    ll.matrix = true;
    ll.groups_off = st.put(descs.data(), descs.size() * sizeof(MxLow));
    ll.n_groups = (uint32_t)descs.size();
    ll.total_wgs = (uint32_t)acc;
    levels.push_back(ll);
    return STWO_HIP_OK;
  };
  auto add_mx_tops = [&](int stage) -> int {
    for (uint32_t layers : {8u, 4u}) {
      uint64_t units = 0, acc = 0;
      auto takes = [&](size_t gi) {
        return gp[gi].matrix && gt[gi].stage == stage && gp[gi].mx.top_layers == layers;
      };
      for (size_t gi = 0; gi < gt.size(); gi++)
        if (takes(gi)) units += mx_top_units(gt[gi].count, gt[gi].n, gp[gi].mx);
      std::vector<MxTop> descs;
      for (size_t gi = 0; gi < gt.size(); gi++) {
        if (!takes(gi)) continue;
        const GroupTabs &t = gt[gi];
        uint32_t wgs = 0;
        descs.push_back(mx_top(tw, (const FftCol *)(dbase + t.ifft_off), (const FftCol *)(dbase + t.rfft_off), t.count,
                               t.n, t.b, stage == BATCH_IFFT || store_coeffs, gp[gi].mx, units,
                               true, &wgs));
        descs.back().wg_start = (uint32_t)acc;
        acc += wgs;
      }
      if (descs.empty()) continue;
      if (acc >= (1ull << 31)) return set_error(ctx, STWO_HIP_EINVAL, "FFT groups too large for one launch");
      LevelLaunch ll{};
      ll.matrix = true;
      ll.mx_layers = layers;
      ll.mx_inv = stage != BATCH_RFFT;
      ll.mx_fwd = stage != BATCH_IFFT;
      ll.groups_off = st.put(descs.data(), descs.size() * sizeof(MxTop));
      ll.n_groups = (uint32_t)descs.size();
      ll.total_wgs = (uint32_t)acc;
      levels.push_back(ll);
    }
    return STWO_HIP_OK;
  };
  // Small and large columns apart, a launch's workgroups having the lanes and the
  // LDS of its largest; together where there is a CU for each (then the further
  // launch costs more, 5 us).
  auto add_columns = [&](int stage) {
    uint64_t cols = 0;
    for (size_t gi = 0; gi < gt.size(); gi++)
      if (gp[gi].column && gt[gi].stage == stage) cols += gt[gi].count;
    const bool apart = cols > 256;
    for (uint32_t large = 0; large <= (uint32_t)apart; large++) {
      std::vector<ColumnFft> descs;
      uint32_t acc = 0, max_n = 0, max_N = 0;
      for (size_t gi = 0; gi < gt.size(); gi++) {
        const GroupTabs &t = gt[gi];
        const uint32_t N = t.n + (stage == BATCH_IFFT ? 0 : t.b);
        if (!gp[gi].column || t.stage != stage || (apart && (N > 10) != large)) continue;
        descs.push_back(column_fft(tw, (const FftCol *)(dbase + t.rfft_off), t.count, t.n, N, store_coeffs));
        descs.back().wg_start = acc;
        acc += t.count;
        max_n = std::max(max_n, t.n);
        max_N = std::max(max_N, N);
      }
      if (descs.empty()) continue;
      LevelLaunch ll{};
      ll.column_n = max_n;
      ll.column_N = max_N;
      ll.mx_inv = stage != BATCH_RFFT;
      ll.mx_fwd = stage != BATCH_IFFT;
      ll.groups_off = st.put(descs.data(), descs.size() * sizeof(ColumnFft));
      ll.n_groups = (uint32_t)descs.size();
      ll.total_wgs = acc;
      levels.push_back(ll);
    }
  };
  for (int dir = 0; dir < 2; dir++) {
    const bool inverse = dir == 0;
    if (inverse) {
      add_columns(BATCH_IFFT);
      add_columns(BATCH_LDE);
    } else {
      add_columns(BATCH_RFFT);
    }
    int mrc = inverse ? add_mx_low(true) : add_mx_tops(BATCH_LDE);
    if (!mrc && !inverse) mrc = add_mx_tops(BATCH_RFFT);
    if (mrc) return mrc;
    // (level, workgroup size) -> passes of every group (the fused ones aside)
    std::map<std::pair<uint32_t, uint32_t>, std::vector<PassLaunch>> by_level;
    for (const GroupPasses &g : gp) {
      if (g.column) continue;
      const std::vector<PassLaunch> &passes = inverse ? g.inv : g.fwd;
      const size_t k0 = (!inverse && g.fused) ? 1 : 0, k1 = passes.size() - ((inverse && g.fused) ? 1 : 0);
      for (size_t k = k0; k < k1; k++) {
        uint32_t level = inverse ? (uint32_t)k : (uint32_t)(passes.size() - 1 - k);
        if (g.matrix) level = 1;  // the middle one of three
        by_level[{level, passes[k].wg_log}].push_back(passes[k]);
      }
    }
    if (!inverse) {
      // the fused passes run after every IFFT level and before every RFFT one
      std::map<std::pair<uint32_t, int>, std::vector<size_t>> fused;  // (wg_log, kind) -> groups
      for (size_t gi = 0; gi < gp.size(); gi++)
        if (gp[gi].fused)
          fused[{gp[gi].inv.back().wg_log, lde_kind(gp[gi].inv.back(), gp[gi].fwd.front())}].push_back(gi);
      for (auto &kv : fused) {
        std::vector<FftPass2> pis, pfs;
        std::vector<uint32_t> starts;
        uint64_t acc = 0;
        for (size_t gi : kv.second) {
          pis.push_back(gp[gi].inv.back().p);
          pfs.push_back(gp[gi].fwd.front().p);
          starts.push_back((uint32_t)acc);
          acc += gp[gi].inv.back().wgs;
        }
        if (acc >= (1ull << 31)) return set_error(ctx, STWO_HIP_EINVAL, "FFT groups too large for one launch");
        LevelLaunch ll{};
        ll.inverse = false;
        ll.fused = true;
        ll.kind = kv.first.second;
        ll.groups_off = st.put(pis.data(), pis.size() * sizeof(FftPass2));
        ll.fwd_off = st.put(pfs.data(), pfs.size() * sizeof(FftPass2));
        ll.wgs_off = st.put(starts.data(), starts.size() * sizeof(uint32_t));
        ll.n_groups = (uint32_t)pis.size();
        ll.total_wgs = (uint32_t)acc;
        ll.wg_log = kv.first.first;
        levels.push_back(ll);
      }
    }
    std::vector<std::pair<uint32_t, uint32_t>> order;
    for (auto &kv : by_level) order.push_back(kv.first);
    if (!inverse) std::reverse(order.begin(), order.end());  // forward: highest level first
    for (const auto &key : order) {
      int rc = add_level(inverse, key.second, by_level[key]);
      if (rc) return rc;
    }
    mrc = inverse ? add_mx_tops(BATCH_IFFT) : add_mx_low(false);
    if (mrc) return mrc;
  }
  return STWO_HIP_OK;
}

int issue_levels(stwo_hip_ctx *c, const std::vector<LevelLaunch> &levels, uint8_t *dbase, uint32_t keep_coeffs) {
  for (const LevelLaunch &ll : levels) {
    if (ll.column_N) {
      int rc = launch_column_fft_multi(c, (const ColumnFft *)(dbase + ll.groups_off), ll.n_groups, ll.total_wgs,
                                       ll.column_n, ll.column_N, ll.mx_inv, ll.mx_fwd);
      if (rc) return rc;
      continue;
    }
    if (ll.matrix) {
      int rc = ll.mx_layers
                   ? launch_mx_top(c, nullptr, (const MxTop *)(dbase + ll.groups_off), ll.n_groups, ll.total_wgs,
                                   ll.mx_layers, ll.mx_inv, ll.mx_fwd)
                   : launch_mx_low(c, nullptr, (const MxLow *)(dbase + ll.groups_off), ll.n_groups, ll.total_wgs,
                                   ll.inverse);
      if (rc) return rc;
      continue;
    }
    int rc = ll.fused ? launch_lde_multi(c, (const FftPass2 *)(dbase + ll.groups_off),
                                         (const FftPass2 *)(dbase + ll.fwd_off),
                                         (const uint32_t *)(dbase + ll.wgs_off), ll.n_groups, ll.total_wgs,
                                         ll.wg_log, ll.kind, keep_coeffs)
                      : launch_fft_multi(c, ll.inverse, (const FftPass2 *)(dbase + ll.groups_off),
                                         (const uint32_t *)(dbase + ll.wgs_off), ll.n_groups, ll.total_wgs,
                                         ll.wg_log, ll.kind);
    if (rc) return rc;
  }
  return STWO_HIP_OK;
}

}  // namespace

int batch_create_trees(stwo_hip_ctx *ctx, const BatchTree *trees, size_t n_trees, const stwo_hip_twiddles *tw,
                       int flags, stwo_hip_batch **out) {
  const int use_graph = flags & STWO_HIP_BATCH_GRAPH;
  if (!ctx || !out) return STWO_HIP_EINVAL;
  *out = nullptr;
  STWO_HIP_CHECK_ARG(ctx, n_trees > 0 && trees, "batch_create: no column sets");
  STWO_HIP_CHECK_ARG(ctx, tw && tw->device == ctx->device, "batch_create: twiddles missing or from another device");
  uint32_t all_max = 0;
  for (size_t t = 0; t < n_trees; t++) {
    const BatchTree &T = trees[t];
    STWO_HIP_CHECK_ARG(ctx, T.stage == BATCH_LDE || T.stage == BATCH_IFFT || T.stage == BATCH_RFFT,
                       "batch_create: unknown stage %d (set %zu)", T.stage, t);
    const bool has_outs = T.stage != BATCH_IFFT, has_tree = T.stage == BATCH_LDE || T.layers;
    STWO_HIP_CHECK_ARG(ctx, T.n_cols > 0 && T.cols && T.log_sizes && (T.outs || !has_outs) &&
                                (T.layers || T.stage != BATCH_LDE),
                       "batch_create: NULL or empty arguments (set %zu)", t);
    if (has_tree) {
      STWO_HIP_CHECK_ARG(ctx, T.tree_kind == STWO_HIP_TREE_MIXED || T.tree_kind == STWO_HIP_TREE_LIFTED,
                         "batch_create: unknown tree kind %d", T.tree_kind);
      STWO_HIP_CHECK_ARG(ctx, T.hash_mode == STWO_HIP_HASH_BLAKE2S || T.hash_mode == STWO_HIP_HASH_BLAKE2S_M31,
                         "batch_create: unknown hash mode %d", T.hash_mode);
    }
    const uint32_t b = T.stage == BATCH_IFFT ? 0 : T.log_blowup;
    for (size_t i = 0; i < T.n_cols; i++) {
      STWO_HIP_CHECK_ARG(ctx, T.cols[i] && (!has_outs || T.outs[i]), "batch_create: NULL column %zu", i);
      STWO_HIP_CHECK_ARG(ctx, T.log_sizes[i] >= 4 && T.log_sizes[i] <= 28 && b <= 24 && T.log_sizes[i] + b <= 28,
                         "batch_create: column %zu log size %u outside [4, 28 - blowup]", i, T.log_sizes[i]);
      all_max = std::max(all_max, T.log_sizes[i] + b);
    }
  }
  // Every CanonicCoset(k).circle_domain(), k <= max_log, must be a doubling of the root.
  uint32_t rl = tw->root.log_size;
  STWO_HIP_CHECK_ARG(ctx, all_max - 1 <= rl && tw->root.initial_index == half_odds_initial(rl),
                     "batch_create: twiddle root must be half_odds(r) with r >= %u", all_max - 1);

  // Groups by (log size, blowup, stage) over every set, largest first (their
  // workgroups start first): columns of different sets share launches.
  std::map<std::tuple<uint32_t, uint32_t, int>, std::vector<std::pair<size_t, size_t>>,
           std::greater<std::tuple<uint32_t, uint32_t, int>>> groups;
  for (size_t t = 0; t < n_trees; t++)
    for (size_t i = 0; i < trees[t].n_cols; i++)
      groups[{trees[t].log_sizes[i], trees[t].stage == BATCH_IFFT ? 0u : trees[t].log_blowup, trees[t].stage}]
          .push_back({t, i});

  Staging st;
  std::vector<GroupTabs> gt;
  for (auto &g : groups) {
    const int stage = std::get<2>(g.first);
    std::vector<FftCol> cols;
    for (auto &ti : g.second) {
      uint32_t *col = trees[ti.first].cols[ti.second];
      cols.push_back({col, stage == BATCH_IFFT ? col : trees[ti.first].outs[ti.second]});
    }
    gt.push_back(put_group(st, std::get<0>(g.first), std::get<1>(g.first), stage, cols));
  }
  // Merkle column tables, per set.
  std::vector<TreeLaunches> tl;
  for (size_t t = 0; t < n_trees; t++) {
    const BatchTree &T = trees[t];
    if (T.stage == BATCH_IFFT || !T.layers) continue;
    tl.emplace_back();
    TreeLaunches &L = tl.back();
    L.layers = T.layers;
    L.mode = T.hash_mode;
    L.kind = T.tree_kind;
    L.max_log = 0;
    for (size_t i = 0; i < T.n_cols; i++) L.max_log = std::max(L.max_log, T.log_sizes[i] + T.log_blowup);
    if (T.tree_kind == STWO_HIP_TREE_MIXED) {
      for (int l = (int)L.max_log; l >= 0; l--) {
        std::vector<ColRef> refs;
        for (size_t i = 0; i < T.n_cols; i++)
          if (T.log_sizes[i] + T.log_blowup == (uint32_t)l) refs.push_back({T.outs[i], 0, 0});
        if (!refs.empty())
          L.lt.push_back({(uint32_t)l, st.put(refs.data(), refs.size() * sizeof(ColRef)), (uint32_t)refs.size()});
      }
    } else {
      std::vector<size_t> order(T.n_cols);
      for (size_t i = 0; i < T.n_cols; i++) order[i] = i;
      std::stable_sort(order.begin(), order.end(),
                       [&](size_t a, size_t b) { return T.log_sizes[a] < T.log_sizes[b]; });
      std::vector<ColRef> refs;
      for (size_t i : order) refs.push_back({T.outs[i], L.max_log - (T.log_sizes[i] + T.log_blowup), 0});
      L.lt.push_back({L.max_log, st.put(refs.data(), refs.size() * sizeof(ColRef)), (uint32_t)refs.size()});
    }
  }
  // Reserve the pass descriptor area after the tables: the descriptors hold
  // device addresses of the tables, known once the buffer exists.
  // The trees' own counters: the plan may run on another context's stream than
  // the one that made it, and its trees share launches.
  for (TreeLaunches &L : tl) {
    const std::vector<uint32_t> zeros(tree_counters(L.max_log), 0);
    L.counters_off = st.put(zeros.data(), zeros.size() * sizeof(uint32_t));
  }
  size_t tables_bytes = (st.host.size() + 255) & ~(size_t)255;
  void *dmem = nullptr;
  bool from_job = false;
  // A tree's steps: its layers with columns and a run of nodes after each, at most
  // two launches of it; every launch's table starts aligned.
  size_t tree_steps_bound = 0;
  if (tl.size() > 1)
    for (const TreeLaunches &L : tl) tree_steps_bound += 3 * L.lt.size() * (sizeof(MerkleTree) + 256);
  const size_t desc_bytes = levels_bound(gt.size()) + tree_steps_bound;
  int arc = device_alloc(ctx, tables_bytes + desc_bytes, &dmem, &from_job);
  if (arc) return arc;
  auto release = [&]() { device_free(dmem, from_job); };
  uint8_t *dbase = (uint8_t *)dmem;
  std::vector<LevelLaunch> levels;
  int lrc = build_levels(ctx, tw, gt, dbase, !(flags & STWO_HIP_BATCH_DROP_COEFFS), true, st, levels);
  if (lrc) {
    release();
    return lrc;
  }
  // The trees, step by step (layers max_log .. 0 of a mixed tree with runs of
  // pure node layers in one; leaves and nodes of a lifted one): the steps of one
  // kind that the trees have at the same place share a launch.  Alone, most
  // trees leave the device idle: 12 trees of 2^13 and 2^17 leaves took 470 us
  // one after another, 205 us in shared launches.
  std::vector<TreeWave> waves;
  {
    std::vector<std::vector<MerkleStep>> steps(tl.size());
    size_t longest = 0;
    for (size_t k = 0; k < tl.size(); k++) {
      const TreeLaunches &L = tl[k];
      uint32_t *counters = (uint32_t *)(dbase + L.counters_off);
      const uint32_t n_counters = tree_counters(L.max_log);
      const bool lifted = L.kind == STWO_HIP_TREE_LIFTED;
      size_t ti = 0;
      for (int l = (int)L.max_log; l >= 0;) {
        const uint32_t *prev = l == (int)L.max_log ? nullptr : L.layers + tree_layer_off((uint32_t)l + 1);
        const auto *t = ti < L.lt.size() && L.lt[ti].log_size == (uint32_t)l ? &L.lt[ti++] : nullptr;
        const int next = ti < L.lt.size() ? (int)L.lt[ti].log_size : -1;  // the next layer with columns
        if (t) {
          steps[k].push_back(merkle_layer_step(prev, (const ColRef *)(dbase + t->off), t->count, (uint32_t)l,
                                               L.layers + tree_layer_off((uint32_t)l), L.mode, lifted));
          if (!merkle_tree_step(steps[k].back(), (uint32_t)(next + 1), counters, n_counters)) {
            l--;
            continue;
          }
          l = next;
        } else {
          steps[k].push_back(
              merkle_nodes_step(L.layers, (uint32_t)l + 1, (uint32_t)(next + 1), L.mode, counters, n_counters));
          l = (int)steps[k].back().nodes.stop_log - 1;
        }
      }
      longest = std::max(longest, steps[k].size());
    }
    for (size_t at = 0; at < longest; at++)
      for (uint32_t kind = 0; kind < kMerkleKinds; kind++) {
        std::vector<const MerkleStep *> same;
        for (const auto &v : steps)
          if (at < v.size() && v[at].kind == kind) same.push_back(&v[at]);
        if (same.empty()) continue;
        TreeWave w{*same[0], 0, (uint32_t)same.size(), same[0]->wgs};
        if (w.n > 1) {
          // the largest first: theirs are the longest workgroups (or chains of them)
          std::stable_sort(same.begin(), same.end(),
                           [](const MerkleStep *a, const MerkleStep *c) { return a->wgs > c->wgs; });
          std::vector<MerkleLayer> ls;
          std::vector<MerkleNodes> ns;
          std::vector<MerkleTree> ts;
          uint64_t acc = 0;
          for (const MerkleStep *s : same) {
            ls.push_back(s->layer);
            ls.back().wg_start = (uint32_t)acc;
            ns.push_back(s->nodes);
            ns.back().wg_start = (uint32_t)acc;
            ts.push_back(s->tree);
            ts.back().wg_start = (uint32_t)acc;
            acc += s->wgs;
          }
          if (acc >= (1ull << 31)) {
            release();
            return set_error(ctx, STWO_HIP_EINVAL, "batch_create: grid too large");
          }
          w.wgs = (uint32_t)acc;
          w.off = kind < kMerkleNodes64 ? st.put(ls.data(), ls.size() * sizeof(MerkleLayer))
                  : kind < kMerkleTree  ? st.put(ns.data(), ns.size() * sizeof(MerkleNodes))
                                        : st.put(ts.data(), ts.size() * sizeof(MerkleTree));
        }
        waves.push_back(w);
      }
  }
  if (st.host.size() > tables_bytes + desc_bytes) {
    release();
    return set_error(ctx, STWO_HIP_EINVAL, "internal: batch descriptor area overflow");
  }
  if (from_job) {
    // within a job: an ordered copy on the job's stream
    int rc = flush_uploads(ctx);
    if (rc) return rc;
    STWO_HIP_TRY(ctx, hipMemcpyAsync(dmem, st.host.data(), st.host.size(), hipMemcpyHostToDevice, ctx->stream));
    STWO_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
  } else if (hipMemcpy(dmem, st.host.data(), st.host.size(), hipMemcpyHostToDevice) != hipSuccess) {
    release();
    return set_error(ctx, STWO_HIP_EDEVICE, "batch_create: table upload failed");
  }

  stwo_hip_batch *b = new (std::nothrow) stwo_hip_batch();
  if (!b) {
    release();
    return set_error(ctx, STWO_HIP_ENOMEM, "host allocation failed");
  }
  b->device = ctx->device;
  b->d_mem = dmem;
  b->mem_from_job = from_job;
  const uint32_t keep_coeffs = (flags & STWO_HIP_BATCH_DROP_COEFFS) ? 0u : 1u;
  b->issue = [levels, waves, dbase, keep_coeffs](stwo_hip_ctx *c) -> int {
    int frc = issue_levels(c, levels, dbase, keep_coeffs);
    if (frc) return frc;
    for (const TreeWave &w : waves) {
      int rc = w.n > 1 ? launch_merkle_multi(c, w.step.kind, w.step.layer.lifted, dbase + w.off, w.n, w.wgs)
                       : launch_merkle(c, w.step);
      if (rc) return rc;
    }
    return STWO_HIP_OK;
  };
  b->n_launches = levels.size();
  if (use_graph) {
    // Tables of earlier calls still pending are copied outside the graph.
    int frc = flush_uploads(ctx);
    if (frc) {
      release();
      delete b;
      return frc;
    }
    bool prof = ctx->prof;
    ctx->prof = false;  // no event records inside the captured sequence
    hipError_t e = hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal);
    int rc = e == hipSuccess ? b->issue(ctx) : STWO_HIP_EDEVICE;
    hipGraph_t g = nullptr;
    hipError_t e2 = hipStreamEndCapture(ctx->stream, &g);
    ctx->prof = prof;
    if (rc == STWO_HIP_OK && e2 == hipSuccess && g) {
      if (hipGraphInstantiate(&b->exec, g, nullptr, nullptr, 0) != hipSuccess) rc = STWO_HIP_EDEVICE;
      b->graph = g;
    } else if (rc == STWO_HIP_OK) {
      rc = STWO_HIP_EDEVICE;
    }
    if (rc) {
      if (g) (void)hipGraphDestroy(g);
      release();
      delete b;
      (void)hipGetLastError();
      return set_error(ctx, rc, "batch_create: graph capture failed (%s)",
                       ctx->last_error.empty() ? "hip" : ctx->last_error.c_str());
    }
  }
  *out = b;
  return STWO_HIP_OK;
}

// The transforms of several groups in shared launches, straight away; *done =
// false (nothing launched) where their tables do not fit the upload ring or a
// group's output meets another group's columns, whose order then counts.
int run_fft_sets(stwo_hip_ctx *ctx, const std::vector<FftSet> &sets, const stwo_hip_twiddles *tw, bool store_coeffs,
                 bool *done) {
  *done = false;
  // [first, end) of every column, with its group and whether it is written
  struct Span {
    uintptr_t at, end;
    uint32_t group, out;
  };
  std::vector<Span> spans;
  for (uint32_t g = 0; g < sets.size(); g++)
    for (const FftCol &c : sets[g].cols) {
      const bool evaluates = sets[g].stage != BATCH_IFFT;
      spans.push_back({(uintptr_t)c.in, (uintptr_t)(c.in + ((size_t)1 << sets[g].n)), g, sets[g].stage != BATCH_RFFT});
      if (evaluates)  // also where it lies over the input
        spans.push_back({(uintptr_t)c.out, (uintptr_t)(c.out + ((size_t)1 << (sets[g].n + sets[g].b))), g, 1});
    }
  auto by_at = [](const Span &a, const Span &c) { return a.at < c.at; };
  if (!std::is_sorted(spans.begin(), spans.end(), by_at)) std::sort(spans.begin(), spans.end(), by_at);
  // The furthest end met so far, and the furthest of the other groups.
  struct Far {
    uintptr_t end = 0, end2 = 0;
    uint32_t group = 0;
    void add(uintptr_t e, uint32_t g) {
      if (g == group) {
        end = std::max(end, e);
      } else if (e > end) {
        end2 = end;
        end = e;
        group = g;
      } else {
        end2 = std::max(end2, e);
      }
    }
    uintptr_t other(uint32_t g) const { return g == group ? end2 : end; }
  } any, written;
  for (const Span &s : spans) {
    if (s.at < (s.out ? any : written).other(s.group)) return STWO_HIP_OK;
    any.add(s.end, s.group);
    if (s.out) written.add(s.end, s.group);
  }
  Staging st;
  std::vector<GroupTabs> gt;
  for (const FftSet &s : sets) gt.push_back(put_group(st, s.n, s.b, s.stage, s.cols));
  // The matrix passes where their units, over all groups, fill the device: they
  // are far fewer and longer than the vector passes' workgroups.
  uint64_t units = 0;
  for (const GroupTabs &t : gt) {
    MxPlan mx;
    if (mx_plan(ctx, tw, t.n, t.stage == BATCH_IFFT ? 0 : t.b, t.stage == BATCH_IFFT, t.count, t.aligned16, true, &mx))
      units += mx_low_units(t.count, t.n);
  }
  const size_t bound = ((st.host.size() + 255) & ~(size_t)255) + levels_bound(gt.size());
  uint8_t *h = nullptr, *d = nullptr;
  if (bound > ctx->arena_cap / 2) return STWO_HIP_OK;
  int rc = upload_begin(ctx, bound, &h, &d);
  if (rc) return rc;
  std::vector<LevelLaunch> levels;
  rc = build_levels(ctx, tw, gt, d, store_coeffs, units >= kMxMinUnits, st, levels);
  if (!rc && st.host.size() > bound) rc = set_error(ctx, STWO_HIP_EINVAL, "internal: FFT descriptor area overflow");
  if (rc) {
    upload_end(ctx, 0);
    return rc;
  }
  memcpy(h, st.host.data(), st.host.size());
  upload_end(ctx, st.host.size());
  *done = true;
  return issue_levels(ctx, levels, d, store_coeffs);
}

}  // namespace stwo_hip

using namespace stwo_hip;

extern "C" {

int stwo_hip_batch_create(stwo_hip_ctx *ctx, uint32_t *const *cols, const uint32_t *log_sizes, size_t n_cols,
                          uint32_t log_blowup, const stwo_hip_twiddles *tw, uint32_t *const *outs, uint32_t *layers,
                          int tree_kind, int hash_mode, int flags, stwo_hip_batch **out) {
  const BatchTree t = {cols, log_sizes, n_cols, log_blowup, outs, layers, tree_kind, hash_mode};
  return batch_create_trees(ctx, &t, 1, tw, flags, out);
}

int stwo_hip_batch_create_multi(stwo_hip_ctx *ctx, const stwo_hip_batch_set *sets, size_t n_sets,
                                const stwo_hip_twiddles *tw, int flags, stwo_hip_batch **out) {
  if (!ctx) return STWO_HIP_EINVAL;
  STWO_HIP_CHECK_ARG(ctx, sets && n_sets, "batch_create_multi: no column sets");
  std::vector<BatchTree> t(n_sets);
  for (size_t i = 0; i < n_sets; i++)
    t[i] = {sets[i].cols,   sets[i].log_sizes, sets[i].n_cols,    sets[i].log_blowup, sets[i].outs,
            sets[i].layers, sets[i].tree_kind, sets[i].hash_mode, sets[i].stage};
  return batch_create_trees(ctx, t.data(), n_sets, tw, flags, out);
}

int stwo_hip_lde_commit_per_column(stwo_hip_ctx *ctx, uint32_t *const *cols, const uint32_t *log_sizes,
                                   size_t n_cols, uint32_t log_blowup, const stwo_hip_twiddles *tw,
                                   uint32_t *const *outs, uint32_t *layers, int tree_kind, int hash_mode) {
  if (!ctx) return STWO_HIP_EINVAL;
  STWO_HIP_CHECK_ARG(ctx, n_cols > 0 && cols && log_sizes && outs && layers, "lde_commit_per_column: NULL arguments");
  STWO_HIP_CHECK_ARG(ctx, tree_kind == STWO_HIP_TREE_MIXED || tree_kind == STWO_HIP_TREE_LIFTED,
                     "lde_commit_per_column: unknown tree kind %d", tree_kind);
  uint32_t max_log = 0;
  std::vector<uint32_t> out_logs(n_cols);
  for (size_t i = 0; i < n_cols; i++) {
    STWO_HIP_CHECK_ARG(ctx, log_sizes[i] >= 1 && log_sizes[i] + log_blowup <= 28,
                       "lde_commit_per_column: column %zu log size %u", i, log_sizes[i]);
    const uint32_t n = log_sizes[i], N = n + log_blowup;
    // one interpolate and one evaluate call per column, as the reference's
    // plain path submits them
    int rc = stwo_hip_interpolate(ctx, cols[i], {half_odds_initial(n - 1), n - 1}, tw);
    if (rc) return rc;
    rc = stwo_hip_evaluate(ctx, cols[i], n, {half_odds_initial(N - 1), N - 1}, tw, outs[i]);
    if (rc) return rc;
    out_logs[i] = N;
    max_log = std::max(max_log, N);
  }
  std::vector<const uint32_t *> oc(outs, outs + n_cols);
  if (tree_kind == STWO_HIP_TREE_MIXED) return stwo_hip_merkle_commit(ctx, oc.data(), out_logs.data(), n_cols, layers,
                                                                      hash_mode);
  return stwo_hip_merkle_lifted_commit(ctx, oc.data(), out_logs.data(), n_cols, max_log, layers, hash_mode);
}

int stwo_hip_batch_run(stwo_hip_ctx *ctx, stwo_hip_batch *b) {
  if (!ctx || !b) return STWO_HIP_EINVAL;
  STWO_HIP_CHECK_ARG(ctx, b->device == ctx->device, "batch_run: plan belongs to another device");
  if (b->exec) {
    hipEvent_t start = nullptr;
    prof_begin(ctx, "batch_graph", &start);
    STWO_HIP_TRY(ctx, hipGraphLaunch(b->exec, ctx->stream));
    prof_end(ctx, "batch_graph", start);
    return STWO_HIP_OK;
  }
  return b->issue(ctx);
}

int stwo_hip_batch_destroy(stwo_hip_ctx *ctx, stwo_hip_batch *b) {
  if (!ctx || !b) return STWO_HIP_EINVAL;
  (void)hipStreamSynchronize(ctx->stream);
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  device_free(b->d_mem, b->mem_from_job);
  delete b;
  return STWO_HIP_OK;
}

}  // extern "C"
