// FRI folds (FriOps) and the FRI commitment driver (FriProver::commit).
//
// Fold factors come from the resident inverse twiddle tree, as SimdBackend
// does (SIMD/fri.rs:32-172): for a circle domain of log size N the factor of
// pair i is 1/p.y with p = domain.at(bitrev(2i, N)) -- the inverse circle
// twiddle of pair i -- and for a line domain of log size n the factor of
// pair i is 1/x with x = domain.at(bitrev(2i, n)) -- entry i of the inverse
// tree level of that domain, itw[len - 2^n + i].  QM31 columns are 4
// coordinate columns (SoA), so each lane's loads are coalesced.
//
// fold_line folds up to 4 steps per launch with the 2^step inputs of an
// output held in VGPRs (alpha, alpha^2, ... per step, SIMD/fri.rs:52-111).
#include <string.h>

#include <algorithm>

#include <vector>

#include "blake2s.hpp"
#include "channel.hpp"
#include "common.hpp"
#include "field.hpp"
#include "internal.hpp"
#include "merkle_dev.hpp"

namespace stwo_hip {

struct Qm31Cols {
  uint32_t *c[4];
};
struct Qm31ColsConst {
  const uint32_t *c[4];
};

__device__ __forceinline__ uint32_t circle_itwiddle(const uint32_t *itw_end, uint32_t N, uint32_t h) {
  const uint32_t *l0 = itw_end - ((int64_t)1 << (N - 1));
  uint32_t x = l0[2 * (h >> 2)], y = l0[2 * (h >> 2) + 1];
  uint32_t v = (h & 2) ? x : y;
  bool neg = ((h & 3) == 1) || ((h & 3) == 2);
  return neg ? m31_neg(v) : v;
}

__device__ __forceinline__ qm31 load_qm31(const uint32_t *p) { return qm31_make(p[0], p[1], p[2], p[3]); }

// Per-output folds (shared by the standalone fold kernels, the fused FRI
// layer kernel and the small-layer tail).  Circle: output i of the fold of a
// circle evaluation of log size N (f0 = f[2i] + f[2i+1], f1 = (f[2i] -
// f[2i+1]) / p.y, f0 + alpha f1).
__device__ __forceinline__ qm31 fold_circle_at(const Qm31ColsConst &src, const uint32_t *itw_end, uint32_t N,
                                               const qm31 &alpha, uint32_t i) {
  const uint32_t iy = circle_itwiddle(itw_end, N, i);
  qm31 f0, f1;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    uint2 v = reinterpret_cast<const uint2 *>(src.c[k])[i];
    f0.v[k] = m31_add(v.x, v.y);
    f1.v[k] = m31_mul(m31_sub(v.x, v.y), iy);
  }
  return qm31_add(f0, qm31_mul(alpha, f1));
}

// Line: output i of STEP successive folds of a line evaluation of log size n
// (the 2^STEP inputs of the output in VGPRs; alpha, alpha^2, ... per fold).
template <int STEP>
__device__ __forceinline__ qm31 fold_line_at(const Qm31ColsConst &src, const uint32_t *itw_end, uint32_t n,
                                             qm31 a, uint32_t i) {
  constexpr int W = 1 << STEP;
  qm31 v[W];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const uint32_t *s = src.c[k] + (size_t)i * W;
#pragma unroll
    for (int j = 0; j < W; j++) v[j].v[k] = s[j];
  }
#pragma unroll
  for (int layer = 0; layer < STEP; layer++) {
    const int half = W >> (layer + 1);
    const uint32_t *lvl = itw_end - ((int64_t)1 << (n - layer));
#pragma unroll
    for (int j = 0; j < half; j++) {
      uint32_t xi = lvl[(size_t)i * half + j];
      qm31 f0, f1;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        f0.v[k] = m31_add(v[2 * j].v[k], v[2 * j + 1].v[k]);
        f1.v[k] = m31_mul(m31_sub(v[2 * j].v[k], v[2 * j + 1].v[k]), xi);
      }
      v[j] = qm31_add(f0, qm31_mul(a, f1));
    }
    a = qm31_mul(a, a);
  }
  return v[0];
}

// `alpha_dev`, when not NULL, holds alpha in device memory (written by the
// device channel) and replaces the by-value alpha.
__global__ void __launch_bounds__(256) fold_circle_kernel(Qm31Cols dst, Qm31ColsConst src, const uint32_t *itw_end,
                                                          uint32_t N, qm31 alpha, qm31 alpha_sq, uint32_t accumulate,
                                                          const uint32_t *alpha_dev) {
  const uint32_t n_out = 1u << (N - 1);
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_out) return;
  if (alpha_dev) {
    alpha = load_qm31(alpha_dev);
    alpha_sq = qm31_mul(alpha, alpha);
  }
  qm31 r = fold_circle_at(src, itw_end, N, alpha, i);
  if (accumulate) {
    qm31 d = qm31_make(dst.c[0][i], dst.c[1][i], dst.c[2][i], dst.c[3][i]);
    r = qm31_add(qm31_mul(d, alpha_sq), r);
  }
#pragma unroll
  for (int k = 0; k < 4; k++) dst.c[k][i] = r.v[k];
}

template <int STEP>
__global__ void __launch_bounds__(256) fold_line_kernel(Qm31Cols dst, Qm31ColsConst src, const uint32_t *itw_end,
                                                        uint32_t n, qm31 alpha, const uint32_t *alpha_dev) {
  const uint32_t n_out = 1u << (n - STEP);
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_out) return;
  if (alpha_dev) alpha = load_qm31(alpha_dev);
  const qm31 r = fold_line_at<STEP>(src, itw_end, n, alpha, i);
#pragma unroll
  for (int k = 0; k < 4; k++) dst.c[k][i] = r.v[k];
}

// out = in^(2^k) (alpha for the folds after the first 4 of a longer fold step).
__global__ void alpha_pow2k_kernel(const uint32_t *in, uint32_t *out, uint32_t k) {
  if (threadIdx.x != 0) return;
  qm31 a = load_qm31(in);
  for (uint32_t i = 0; i < k; i++) a = qm31_mul(a, a);
  for (int j = 0; j < 4; j++) out[j] = a.v[j];
}

// One Fiat-Shamir step of the FRI layer loop on the device, for the
// Blake2sChannel (STWO/core/channel/blake2s.rs): digest = H(digest || root)
// (MerkleChannel::mix_root, STWO/core/vcs_lifted/blake2_merkle.rs:49-55),
// n_draws = 0, then alpha = draw_secure_felt(): draw H(digest || le32(n_draws)
// || 0x00) until all 8 words are < 2P (blake2s.rs:36-51,103-117) and reduce
// the first 4.  chan = [digest 8 words, n_draws, error flag].  The root is
// also copied to root_out.  The retry loop is bounded (each try fails with
// probability about 2^-28); running out sets the error flag.
// Run by the 4 lanes of one quad (lanes 0-3 of a wave, all active), each
// compression shared by the quad (b2_compress_quad).  In registers: m = the
// digest (8 words) || the root; digest gets the new digest, the lane's word of
// alpha is returned.
__device__ __forceinline__ uint32_t channel_core(uint32_t m[16], uint32_t digest[8], uint32_t &n_draws, bool &ok) {
  const b2_quad_iv iv = b2_quad_init();
  uint32_t lo = iv.lo, hi = iv.hi;
  b2_compress_quad(iv, lo, hi, m, b2_quad_d(iv, 64, true));
  b2_quad_gather(lo, hi, digest);
  const uint32_t d37 = b2_quad_d(iv, 37, true);
  n_draws = 0;
  ok = false;
#pragma unroll 1
  for (int tries = 0; tries < 64 && !ok; tries++) {
#pragma unroll
    for (int k = 0; k < 8; k++) m[k] = digest[k];
    m[8] = n_draws;
#pragma unroll
    for (int k = 9; k < 16; k++) m[k] = 0;  // the 0x00 separator byte and zero padding
    lo = iv.lo;
    hi = iv.hi;
    b2_compress_quad(iv, lo, hi, m, d37);
    n_draws++;
    const uint64_t bal = __ballot(lo < 2u * P && hi < 2u * P);
    ok = ((bal >> (__lane_id() & ~3u)) & 0xF) == 0xF;
  }
  return b2_reduce_word(lo);
}
__device__ void channel_step(uint32_t *chan, const uint32_t *root, uint32_t *root_out, uint32_t *alpha_out) {
  const uint32_t j = __lane_id() & 3;
  uint32_t m[16], digest[8], n_draws;
  bool ok;
  for (int k = 0; k < 8; k++) {
    m[k] = chan[k];
    m[8 + k] = root[k];
  }
  root_out[j] = root[j];
  root_out[4 + j] = root[4 + j];
  const uint32_t al = channel_core(m, digest, n_draws, ok);
  chan[j] = digest[j];
  chan[4 + j] = digest[4 + j];
  if (j == 0) {
    chan[8] = n_draws;
    if (!ok) chan[9] = 1;
  }
  alpha_out[j] = al;
}

// The device words of one FRI commit: the channel (digest, n_draws, error flag),
// the alpha drawn last, a slot for its powers, the root mixed before the first
// layer (commits of a group), the roots, then flags, the grind's
// best nonce (8-byte aligned) and prefix, and the last layer: its coefficients
// when the end runs on the device, its evaluation otherwise.
constexpr uint32_t kMaxRoots = 32;  // one per layer, at most log_size <= 28
constexpr uint32_t kDevLastMax = 6;  // largest log of a last layer held here
constexpr uint32_t kAlphaOff = 10, kAlphaTmpOff = 14, kMixedOff = 18, kRootsOff = 32, kFlagsOff = kRootsOff + 8 * kMaxRoots,
                   kBestOff = kFlagsOff + 2, kPrefixOff = kBestOff + 2, kPolyOff = kPrefixOff + 8,
                   kFriStateWords = kPolyOff + (4u << kDevLastMax);
static_assert(kBestOff % 2 == 0, "best nonce alignment");

// FRI commits that run side by side (fri_commit_jobs): blockIdx.y.
constexpr uint32_t kFriJobs = 16;

constexpr int kFoldCircle = 5;  // FOLD for the circle fold

// A layer's value i: FOLD = 0, src at i; FOLD = 1..4, line folds of that many
// steps from a layer of log lg + FOLD; kFoldCircle, the circle fold from log
// lg + 1.  A fold writes the layer to dst (coordinates 2^lg words apart).
template <int FOLD>
__device__ __forceinline__ qm31 fri_value(const Qm31ColsConst &src, uint32_t *dst, const uint32_t *itw_end,
                                          const qm31 &alpha, uint32_t lg, uint32_t i, bool store) {
  if constexpr (FOLD == 0) {
    return qm31_make(as_global(src.c[0])[i], as_global(src.c[1])[i], as_global(src.c[2])[i], as_global(src.c[3])[i]);
  } else {
    qm31 v;
    if constexpr (FOLD == kFoldCircle)
      v = fold_circle_at(src, itw_end, lg + 1, alpha, i);
    else
      v = fold_line_at<FOLD>(src, itw_end, lg + FOLD, alpha, i);
    if (store)
#pragma unroll
      for (int k = 0; k < 4; k++) as_global(dst + ((size_t)k << lg))[i] = v.v[k];
    return v;
  }
}

// ---- the small layers in one launch ---------------------------------------
//
// Below kTailLog a layer's work (a few hundred hashes) is far shorter than a
// launch, so one workgroup runs every remaining inner layer: the fold that
// produces the first of them, then per layer the lifted leaves of
// the 4 coordinate columns, the node layers, the channel step and the line
// fold into the next layer's evaluation.  The layer's values, all folds'
// twiddles (read once: a load between the layers would wait for the stores
// before it) and the channel stay in LDS from phase to phase; the trees, roots, channel state and folded evaluations
// written are the ones the per-layer launches write.  What bounds it is the
// chain of compressions: lg + 3 a layer.  Layers of 2^9 and 2^10 cost one
// workgroup as much as a launch over several costs (four compressions per
// lane for the leaves of 2^10 alone).  The commits of a group take a workgroup
// each.
constexpr uint32_t kTailLog = 8;
constexpr uint32_t kTailMax = 16;

struct FriTailLayer {
  uint32_t *tree;  // the layer's packed lifted tree
  uint32_t *dst;   // the fold's output (log lg - step, coordinates that far apart)
  uint32_t lg, step;
};
struct FriTail {
  Qm31ColsConst src;  // what `fold` folds into the first layer's evaluation first (fold = 0: that evaluation)
  uint32_t *first;
  FriTailLayer l[kTailMax];
  uint32_t n, fold, root;  // root: the first layer's slot
  const uint32_t *itw_end;
  uint32_t *state;
};

struct TailLds {
  TreeLds t;
  uint32_t v[4][1u << kTailLog], tw[1u << kTailLog], chan[8], alpha[4];
};

// Output i of STEP line folds of the layer in LDS (fold_line_at, from LDS).
template <int STEP>
__device__ __forceinline__ qm31 tail_fold(const TailLds &S, const uint32_t *tw, uint32_t n, uint32_t i) {
  constexpr int W = 1 << STEP;
  qm31 a = qm31_make(S.alpha[0], S.alpha[1], S.alpha[2], S.alpha[3]), v[W];
#pragma unroll
  for (int j = 0; j < W; j++)
#pragma unroll
    for (int k = 0; k < 4; k++) v[j].v[k] = S.v[k][i * W + j];
#pragma unroll
  for (int layer = 0; layer < STEP; layer++) {
    const int half = W >> (layer + 1);
    const uint32_t *lvl = tw + (n - (n >> layer));
#pragma unroll
    for (int j = 0; j < half; j++) {
      const uint32_t xi = lvl[i * half + j];
      qm31 f0, f1;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        f0.v[k] = m31_add(v[2 * j].v[k], v[2 * j + 1].v[k]);
        f1.v[k] = m31_mul(m31_sub(v[2 * j].v[k], v[2 * j + 1].v[k]), xi);
      }
      v[j] = qm31_add(f0, qm31_mul(a, f1));
    }
    if (layer + 1 < STEP) a = qm31_mul(a, a);
  }
  return v[0];
}

__device__ __forceinline__ void fri_tail(const FriTail &t) {
  __shared__ __align__(16) TailLds S;
  const uint32_t tid = threadIdx.x, q = tid >> 2, j = tid & 3;
  uint32_t *chan = t.state, *alpha = t.state + kAlphaOff;
  uint32_t n = 1u << t.l[0].lg;
  if (tid < n) {
    // the folds' twiddles: levels lg, lg - 1, ... end the tree
    S.tw[tid] = t.itw_end[(ptrdiff_t)tid - (ptrdiff_t)n];
    const uint32_t lg = t.l[0].lg;
    qm31 v, a = qm31_make(0, 0, 0, 0);
    if (t.fold) a = load_qm31(alpha);
    switch (t.fold) {
      case 0: v = fri_value<0>(t.src, t.first, t.itw_end, a, lg, tid, false); break;
      case 1: v = fri_value<1>(t.src, t.first, t.itw_end, a, lg, tid, true); break;
      case 2: v = fri_value<2>(t.src, t.first, t.itw_end, a, lg, tid, true); break;
      case 3: v = fri_value<3>(t.src, t.first, t.itw_end, a, lg, tid, true); break;
      case 4: v = fri_value<4>(t.src, t.first, t.itw_end, a, lg, tid, true); break;
      default: v = fri_value<kFoldCircle>(t.src, t.first, t.itw_end, a, lg, tid, true); break;
    }
#pragma unroll
    for (int k = 0; k < 4; k++) S.v[k][tid] = v.v[k];
  }
  if (tid < 8) S.chan[tid] = chan[tid];
  uint32_t n_draws = 0;
  bool ok = true;
#pragma unroll 1
  for (uint32_t li = 0; li < t.n; li++) {
    const FriTailLayer &L = t.l[li];
    n = 1u << L.lg;
    __syncthreads();
    const uint32_t n_out = n >> L.step;
    // lifted leaves: H(le32 of the 4 coordinates), one 16-byte block
    uint32_t *leaves = L.tree + tree_layer_off(L.lg);
    uint32_t m[16];
#pragma unroll
    for (int k = 4; k < 16; k++) m[k] = 0;
    if (n > 128) {
      if (tid < n) {
#pragma unroll
        for (int k = 0; k < 4; k++) m[k] = S.v[k][tid];
        b2_state s;
        b2_init(s);
        b2_compress(s, m, 16, true);
        store_hash(leaves + 8 * (size_t)tid, s, 0);
        tree_keep(S.t, 0, tid, s);
      }
    } else {
      for (uint32_t i = q; i < n; i += kTreeThreads / 4) {
#pragma unroll
        for (int k = 0; k < 4; k++) m[k] = S.v[k][i];
        uint32_t lo = b2_iv_lo(j), hi = b2_iv_hi(j);
        b2_compress_quad(lo, hi, m, 16, true);
        as_global(leaves)[8 * i + j] = lo;
        as_global(leaves)[8 * i + 4 + j] = hi;
        tree_row(S.t, 0, i)[j] = lo;
        tree_row(S.t, 0, i)[4 + j] = hi;
      }
    }
    const uint32_t buf = tree_levels(S.t, 0, n, 0, L.lg, L.lg, L.tree, 0, false);
    if (tid < 4) {
      const uint32_t *root = tree_row(S.t, buf, 0);
      uint32_t digest[8];
#pragma unroll
      for (int k = 0; k < 8; k++) {
        m[k] = S.chan[k];
        m[8 + k] = root[k];
      }
      uint32_t *ro = t.state + kRootsOff + 8 * (t.root + li);
      as_global(ro)[j] = root[j];
      as_global(ro)[4 + j] = root[4 + j];
      bool drawn;
      S.alpha[j] = channel_core(m, digest, n_draws, drawn);
      ok = ok && drawn;
      if (j == 0)
#pragma unroll
        for (int k = 0; k < 8; k++) S.chan[k] = digest[k];
    }
    __syncthreads();
    qm31 r;
    const uint32_t *tw = S.tw + ((1u << t.l[0].lg) - n);
    if (tid < n_out) {
      switch (L.step) {
        case 1: r = tail_fold<1>(S, tw, n, tid); break;
        case 2: r = tail_fold<2>(S, tw, n, tid); break;
        case 3: r = tail_fold<3>(S, tw, n, tid); break;
        default: r = tail_fold<4>(S, tw, n, tid); break;
      }
    }
    __syncthreads();
    if (tid < n_out)
#pragma unroll
      for (int k = 0; k < 4; k++) {
        as_global(L.dst + ((size_t)k << (L.lg - L.step)))[tid] = r.v[k];
        S.v[k][tid] = r.v[k];
      }
  }
  if (tid < 8) chan[tid] = S.chan[tid];
  if (tid < 4) alpha[tid] = S.alpha[tid];
  if (tid == 0) {
    chan[8] = n_draws;
    if (!ok) chan[9] = 1;
  }
}
__global__ void __launch_bounds__(kTreeThreads) fri_tail_kernel(FriTail t) { fri_tail(t); }
__global__ void __launch_bounds__(kTreeThreads) fri_tails_kernel(const FriTail *t) { fri_tail(t[blockIdx.x]); }

// ---- one FRI layer in one launch ------------------------------------------
//
// Above kTailLog a layer is committed by fri_layer_kernel: the fold that
// produces it (from the previous layer, with alpha from the device channel),
// its lifted leaves, the node levels (a subtree per workgroup, then the last
// of each group of workgroups to finish, merkle_dev.hpp) and, in the workgroup
// that hashes the root, the channel step.  The trees, roots, channel state and
// folded evaluations written are the ones the separate fold, leaf, node and
// channel launches write.
// A channel's starting state: digest, n_draws, 0.
struct ChanInit {
  uint32_t w[10];
};

struct FriLayerJob {
  const uint32_t *src[4];
  uint32_t *dst;  // a fold's output, coordinates 2^lg words apart
  uint32_t *tree, *state, *counters;
  uint32_t root;  // the layer's slot
};
struct FriLayerJobs {
  FriLayerJob j[kFriJobs];
  // the first layer of a lone commit starts from this channel, not from a state
  uint32_t digest[8], has_digest;
};

// LEAVES per workgroup (tree_leaves_log): 64 with a quad per leaf, 256, 1,024.
template <int FOLD, uint32_t LEAVES>
__global__ void __launch_bounds__(kTreeThreads) fri_layer_kernel(FriLayerJobs jobs, const uint32_t *itw_end,
                                                                 uint32_t lg) {
  __shared__ __align__(16) TreeLds S;
  const FriLayerJob &J = jobs.j[blockIdx.y];
  const Qm31ColsConst src = {{J.src[0], J.src[1], J.src[2], J.src[3]}};
  uint32_t *dst = J.dst, *tree = J.tree, *counters = J.counters;
  uint32_t *chan = J.state, *alpha_dev = J.state + kAlphaOff, *root_out = J.state + kRootsOff + 8 * J.root;
  const uint32_t n = 1u << lg, first = blockIdx.x * LEAVES, tid = threadIdx.x;
  const uint32_t q = tid >> 2, j = tid & 3;
  uint32_t *leaves = tree + tree_layer_off(lg);
  const qm31 alpha = FOLD ? load_qm31(alpha_dev) : qm31_make(0, 0, 0, 0);
  // the channel, for the workgroup that hashes the root
  uint32_t cm[16];
  if (tid < 4)
#pragma unroll
    for (int k = 0; k < 8; k++) cm[k] = FOLD == 0 && jobs.has_digest ? jobs.digest[k] : chan[k];
  uint32_t top = lg, cnt = min(LEAVES, n), row0 = first;  // the level held in S
  // lifted leaf: H(le32 of the 4 coordinates), one 16-byte block
  uint32_t m[16];
#pragma unroll
  for (int k = 4; k < 16; k++) m[k] = 0;
  auto leaf = [&](uint32_t i) {
    const qm31 v = fri_value<FOLD>(src, dst, itw_end, alpha, lg, i, true);
#pragma unroll
    for (int k = 0; k < 4; k++) m[k] = v.v[k];
    b2_state s;
    b2_init(s);
    b2_compress(s, m, 16, true);
    store_hash(leaves + 8 * (size_t)i, s, 0);
    return s;
  };
  auto node = [&](const b2_state &a, const b2_state &b, uint32_t l, size_t i) {
    uint32_t w[16];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      w[k] = a.h[k];
      w[8 + k] = b.h[k];
    }
    b2_state s;
    b2_init(s);
    b2_compress(s, w, 64, true);
    store_hash(tree + tree_layer_off(l) + 8 * i, s, 0);
    return s;
  };
  if constexpr (LEAVES == 64) {
    const uint32_t i = first + q;
    if (i < n) {  // the quad's lanes fold alike, the first stores
      const qm31 v = fri_value<FOLD>(src, dst, itw_end, alpha, lg, i, j == 0);
#pragma unroll
      for (int k = 0; k < 4; k++) m[k] = v.v[k];
      uint32_t lo = b2_iv_lo(j), hi = b2_iv_hi(j);
      b2_compress_quad(lo, hi, m, 16, true);
      as_global(leaves + 8 * (size_t)i)[j] = lo;
      as_global(leaves + 8 * (size_t)i)[4 + j] = hi;
      tree_row(S, 0, q)[j] = lo;
      tree_row(S, 0, q)[4 + j] = hi;
    }
  } else if constexpr (LEAVES == 256) {
    const uint32_t i = first + tid;
    if (i < n) tree_keep(S, 0, tid, leaf(i));
  } else {
    // four leaves per lane and, from registers, the two levels above them
    const uint32_t i = first + 4 * tid;
    b2_state keep;
#pragma unroll 1
    for (uint32_t p = 0; p < 2; p++) {
      const b2_state a = leaf(i + 2 * p), b = leaf(i + 2 * p + 1);
      const b2_state c = node(a, b, lg - 1, i / 2 + p);
      if (p == 0)
        keep = c;
      else
        tree_keep(S, 0, tid, node(keep, c, lg - 2, i / 4));
    }
    top -= 2;
    cnt >>= 2;
    row0 >>= 2;
  }
  const uint32_t lv = 31 - __clz(cnt), l = top - lv;
  uint32_t buf = tree_levels(S, 0, cnt, row0, top, lv, tree, 0, l > 0);
  const int done = tree_finish(S, buf, blockIdx.x, l, 0, tree, 0, counters);
  if (done < 0 || tid >= 4) return;
  const uint32_t *root = tree_row(S, (uint32_t)done, 0);
  uint32_t digest[8], n_draws;
  bool ok;
#pragma unroll
  for (int k = 0; k < 8; k++) cm[8 + k] = root[k];
  root_out[j] = root[j];
  root_out[4 + j] = root[4 + j];
  const uint32_t al = channel_core(cm, digest, n_draws, ok);
  alpha_dev[j] = al;
  if (j == 0) {
#pragma unroll
    for (int k = 0; k < 8; k++) chan[k] = digest[k];
    chan[8] = n_draws;
    if (FOLD == 0 && jobs.has_digest)
      chan[9] = !ok;
    else if (!ok)
      chan[9] = 1;
  }
}

template <int FOLD>
static int launch_fri_layer(stwo_hip_ctx *ctx, const FriLayerJobs &jobs, uint32_t n_jobs, const uint32_t *itw_end,
                            uint32_t lg) {
  const uint32_t per = fri_leaves_log(lg, n_jobs);
  const dim3 grid(1u << (lg > per ? lg - per : 0), n_jobs), block(kTreeThreads);
  return launch(ctx, "fri_layer",
                per == 6   ? fri_layer_kernel<FOLD, 64>
                : per == 8 ? fri_layer_kernel<FOLD, 256>
                           : fri_layer_kernel<FOLD, 1024>,
                grid, block, 0, jobs, itw_end, lg);
}

// The starting states of a group of commits (blockIdx.x): a fresh channel that
// has mixed the root at the head of `tree`, kept in the state (the commit's own
// layers overwrite that tree), and the counters cleared.
struct ChanInits {
  struct {
    uint32_t *state;
    const uint32_t *tree;
    uint32_t *counters, n_counters;
  } c[kFriJobs];
};
__global__ void __launch_bounds__(64) chan_inits_kernel(ChanInits init) {
  const auto &c = init.c[blockIdx.x];
  const uint32_t tid = threadIdx.x;
  for (uint32_t k = tid; k < c.n_counters; k += 64) c.counters[k] = 0;
  if (tid >= 4) return;
  const b2_quad_iv iv = b2_quad_init();
  uint32_t m[16], lo = iv.lo, hi = iv.hi;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    m[k] = 0;
    m[8 + k] = c.tree[k];
  }
  c.state[kMixedOff + tid] = c.tree[tid];
  c.state[kMixedOff + 4 + tid] = c.tree[4 + tid];
  b2_compress_quad(iv, lo, hi, m, b2_quad_d(iv, 64, true));
  c.state[tid] = lo;
  c.state[4 + tid] = hi;
  if (tid < 2) c.state[8 + tid] = 0;
}

// One Fiat-Shamir step of the prove on the device: chan (optionally first
// set to [init digest, 0, 0]) mixes `root` and draws a secure felt t into
// draw_out (channel_step).  When point_out is set, the draw is the OODS
// point's parameter (CirclePoint::get_random_point, STWO/core/circle.rs:169-181):
// p = ((1 - t^2) / (1 + t^2), 2t / (1 + t^2)); point_out receives the point's
// factors for eval_at_point, g_0 = p.y, g_1 = p.x, g_k = pi^(k-1)(p.x) for
// k <= point_log and 0 above (pi(x) = 2x^2 - 1; 128 words), then p.x, p.y and
// vn = pi^(point_log - 1)(p.x) (12 words) for the barycentric weights.
// One wave; the step runs on lanes 0-3.
__global__ void __launch_bounds__(64) prove_channel_kernel(uint32_t *chan, ChanInit init, uint32_t has_init,
                                                           const uint32_t *root, uint32_t *root_out,
                                                           uint32_t *draw_out, uint32_t *point_out,
                                                           uint32_t point_log) {
  const uint32_t tid = threadIdx.x;
  if (has_init) {
    if (tid < 10) chan[tid] = init.w[tid];
    __syncthreads();
  }
  if (tid < 4) channel_step(chan, root, root_out, draw_out);
  if (!point_out) return;
  __syncthreads();
  if (tid != 0) return;
  const qm31 t = load_qm31(draw_out);
  const qm31 one = qm31_make(1, 0, 0, 0);
  const qm31 t2 = qm31_mul(t, t);
  const qm31 inv = qm31_inv(qm31_add(t2, one));
  const qm31 px = qm31_mul(qm31_sub(one, t2), inv);
  const qm31 py = qm31_mul(qm31_add(t, t), inv);
  qm31 vn = px;
  for (int k = 0; k < 4; k++) point_out[k] = py.v[k];
  // g_1 .. g_point_log (the samples read g_k only for k below their log
  // size, which is at most point_log); zeros above
  qm31 x = px;
  for (uint32_t g = 1; g < 32; g++) {
    if (g == point_log) vn = x;
    for (int k = 0; k < 4; k++) point_out[4 * g + k] = g <= point_log ? x.v[k] : 0u;
    if (g < point_log) {
      const qm31 sq = qm31_mul(x, x);
      x = qm31_sub(qm31_add(sq, sq), one);
    }
  }
  for (int k = 0; k < 4; k++) {
    point_out[128 + k] = px.v[k];
    point_out[132 + k] = py.v[k];
    point_out[136 + k] = vn.v[k];
  }
}

int prove_channel_step(stwo_hip_ctx *ctx, uint32_t *chan, const uint8_t *init_digest, const uint32_t *root,
                       uint32_t *root_out, uint32_t *draw_out, uint32_t *point_out, uint32_t point_log) {
  STWO_HIP_CHECK_ARG(ctx, point_log >= 1 && point_log < 32, "internal: OODS point log %u", point_log);
  ChanInit init{};
  if (init_digest) memcpy(init.w, init_digest, 32);
  return launch(ctx, "prove_channel", prove_channel_kernel, dim3(1), dim3(64), 0, chan, init,
                (uint32_t)(init_digest != nullptr), root, root_out, draw_out, point_out, point_log);
}

// ---- the end of the FRI commit and the grind's prefix on the device ------
//
// For a last layer of at most 2^kDevLastMax values: LinePoly::interpolate of
// the last evaluation (fri.rs:274-291; line.rs:131-160: into natural order,
// the line IFFT with x^-1 twiddles of each doubling of the line domain,
// 1/n), into_ordered_coefficients (bit reverse), the degree check (every
// coefficient at or above 2^bound_log must be zero, else flags[0] = 1),
// from_ordered_coefficients (bit reverse of the kept ones) into poly, then
// mix_felts(poly) into the channel (blake2s.rs:58-68: H(digest || poly)),
// then the proof-of-work prefix H(le32(POW_PREFIX) || 0^12 || digest ||
// le32(pow_bits)) (blake2s.rs:122-139) into prefixed, and the grind's
// best-nonce word reset.  One workgroup; the hashing on lanes 0-3.
// The natural-order butterfly i of a line domain of log m uses the inverse x
// of point i, held at itw_end - 2^m + bitrev_{m-1}(i) (the tree keeps each
// doubling's x's of the first half in bit-reversed order).
struct LastLayerArgs {
  const uint32_t *src[4];
  const uint32_t *itw_end;
  uint32_t lg, bound_log, pow_bits, n_inv;
  uint32_t *chan, *poly, *prefixed, *flags;
  unsigned long long *best;
};
__global__ void __launch_bounds__(256) fri_last_layer_kernel(LastLayerArgs a) {
  __shared__ uint32_t v[4][1u << kDevLastMax];
  __shared__ uint32_t msg[8 + (4u << kDevLastMax) + 16];
  const uint32_t tid = threadIdx.x, n = 1u << a.lg;
  if (tid == 0) a.flags[0] = 0;
  for (uint32_t j = tid; j < n; j += blockDim.x)
    for (int c = 0; c < 4; c++) v[c][j] = a.src[c][bitrev32(j, a.lg)];
  __syncthreads();
  for (uint32_t m = a.lg; m >= 1; m--) {
    const uint32_t half = 1u << (m - 1);
    const uint32_t *lvl = a.itw_end - ((size_t)1 << m);
    for (uint32_t b = tid; b < n / 2; b += blockDim.x) {
      const uint32_t i = b & (half - 1), base = (b >> (m - 1)) << m;
      const uint32_t xinv = lvl[bitrev32(i, m - 1)];
      for (int c = 0; c < 4; c++) {
        const uint32_t x = v[c][base + i], y = v[c][base + i + half];
        v[c][base + i] = m31_add(x, y);
        v[c][base + i + half] = m31_mul(m31_sub(x, y), xinv);
      }
    }
    __syncthreads();
  }
  const uint32_t bound = 1u << a.bound_log;
  if (tid < 8) msg[tid] = a.chan[tid];
  for (uint32_t j = tid; j < n; j += blockDim.x) {
    // ordered coefficient j = natural-order IFFT output at bitrev(j), times 1/n
    uint32_t cf[4];
    bool nz = false;
    for (int c = 0; c < 4; c++) {
      cf[c] = m31_mul(v[c][bitrev32(j, a.lg)], a.n_inv);
      nz = nz || cf[c] != 0;
    }
    if (j >= bound) {
      if (nz) a.flags[0] = 1;
    } else {
      const uint32_t o = 4 * bitrev32(j, a.bound_log);
      for (int c = 0; c < 4; c++) {
        a.poly[o + c] = cf[c];
        msg[8 + o + c] = cf[c];
      }
    }
  }
  __syncthreads();
  if (tid >= 4) return;
  const uint32_t j = tid;
  // digest = H(digest || poly): 32 + 16 bound bytes, streamed as the blake2
  // crate buffers it (the last block, full or partial, is the finalized one)
  const uint32_t total = 32 + 16 * bound, n_blocks = (total + 63) / 64;
  uint32_t lo = b2_iv_lo(j), hi = b2_iv_hi(j);
  for (uint32_t k = 0; k < n_blocks; k++) {
    uint32_t m[16];
    for (uint32_t w = 0; w < 16; w++) {
      const uint32_t idx = 16 * k + w;
      m[w] = idx < total / 4 ? msg[idx] : 0u;
    }
    const bool last = k + 1 == n_blocks;
    b2_compress_quad(lo, hi, m, last ? total : 64 * (k + 1), last);
  }
  uint32_t d[8];
  b2_quad_gather(lo, hi, d);
  a.chan[j] = d[j];
  a.chan[4 + j] = d[4 + j];
  if (j == 0) a.chan[8] = 0;  // mixing resets the draw counter
  uint32_t m[16];
  m[0] = kPowPrefix;
  m[1] = m[2] = m[3] = 0;
  for (int w = 0; w < 8; w++) m[4 + w] = d[w];
  m[12] = a.pow_bits;
  m[13] = m[14] = m[15] = 0;
  lo = b2_iv_lo(j);
  hi = b2_iv_hi(j);
  b2_compress_quad(lo, hi, m, 52, true);
  a.prefixed[j] = lo;
  a.prefixed[4 + j] = hi;
  if (j == 0) *a.best = ~0ull;
}

static int check_line_domain(stwo_hip_ctx *ctx, stwo_hip_coset dom, const stwo_hip_twiddles *tw) {
  STWO_HIP_CHECK_ARG(ctx, tw != nullptr && tw->device == ctx->device, "twiddles missing or from another device");
  STWO_HIP_CHECK_ARG(ctx, dom.log_size <= tw->root.log_size, "domain log %u exceeds twiddle root log %u",
                     dom.log_size, tw->root.log_size);
  uint32_t k = tw->root.log_size - dom.log_size;
  uint32_t expect = (uint32_t)(((uint64_t)tw->root.initial_index << k) & IDX_MASK);
  STWO_HIP_CHECK_ARG(ctx, (dom.initial_index & IDX_MASK) == expect,
                     "domain (initial %u, log %u) is not a doubling of the twiddle root (initial %u, log %u)",
                     dom.initial_index, dom.log_size, tw->root.initial_index, tw->root.log_size);
  return STWO_HIP_OK;
}

static int fold_circle(stwo_hip_ctx *ctx, uint32_t *const dst[4], const uint32_t *const src[4], uint32_t N,
                       const qm31 &alpha, const stwo_hip_twiddles *tw, bool accumulate,
                       const uint32_t *alpha_dev = nullptr) {
  Qm31Cols d;
  Qm31ColsConst s;
  for (int k = 0; k < 4; k++) {
    d.c[k] = dst[k];
    s.c[k] = src[k];
  }
  uint32_t n_out = 1u << (N - 1);
  return launch(ctx, accumulate ? "fold_circle_into_line" : "fold_circle_first_layer", fold_circle_kernel,
                dim3((n_out + 255) / 256), dim3(256), 0, d, s, (const uint32_t *)(tw->d_itw + tw->len), N, alpha,
                qm31_mul(alpha, alpha), (uint32_t)accumulate, alpha_dev);
}

// fold_step folds of a line evaluation of log size n (domain checked by caller).
// With `alpha_dev` (alpha in device memory), `alpha_tmp` is a 4-word device
// slot that receives alpha^(2^4k) for fold steps beyond the first 4.
static int fold_line_steps(stwo_hip_ctx *ctx, const uint32_t *const src[4], uint32_t n, qm31 alpha, uint32_t fold_step,
                           const stwo_hip_twiddles *tw, uint32_t *const dst[4], const uint32_t *alpha_dev = nullptr,
                           uint32_t *alpha_tmp = nullptr) {
  const uint32_t *itw_end = tw->d_itw + tw->len;
  const uint32_t *cur[4] = {src[0], src[1], src[2], src[3]};
  uint32_t iter = 0;
  while (fold_step > 0) {
    uint32_t step = std::min<uint32_t>(fold_step, 4);
    uint32_t n_out_log = n - step;
    uint32_t *out[4];
    if (fold_step == step) {
      for (int k = 0; k < 4; k++) out[k] = dst[k];
    } else {
      // Intermediate results alternate between two scratch buffers.
      void *p = nullptr;
      int rc = get_scratch(ctx, (iter & 1) ? "fold_line_b" : "fold_line_a", ((size_t)4 << n_out_log) * 4, &p);
      if (rc) return rc;
      for (int k = 0; k < 4; k++) out[k] = (uint32_t *)p + ((size_t)k << n_out_log);
    }
    Qm31Cols d;
    Qm31ColsConst s;
    for (int k = 0; k < 4; k++) {
      d.c[k] = out[k];
      s.c[k] = cur[k];
    }
    uint32_t blocks = ((1u << n_out_log) + 255) / 256;
    int rc;
    switch (step) {
      case 1: rc = launch(ctx, "fold_line", fold_line_kernel<1>, dim3(blocks), dim3(256), 0, d, s, itw_end, n, alpha, alpha_dev); break;
      case 2: rc = launch(ctx, "fold_line", fold_line_kernel<2>, dim3(blocks), dim3(256), 0, d, s, itw_end, n, alpha, alpha_dev); break;
      case 3: rc = launch(ctx, "fold_line", fold_line_kernel<3>, dim3(blocks), dim3(256), 0, d, s, itw_end, n, alpha, alpha_dev); break;
      default: rc = launch(ctx, "fold_line", fold_line_kernel<4>, dim3(blocks), dim3(256), 0, d, s, itw_end, n, alpha, alpha_dev); break;
    }
    if (rc) return rc;
    for (uint32_t k = 0; k < step; k++) alpha = qm31_mul(alpha, alpha);
    if (alpha_dev && fold_step > step) {
      rc = launch(ctx, "alpha_pow2k", alpha_pow2k_kernel, dim3(1), dim3(64), 0, alpha_dev, alpha_tmp, step);
      if (rc) return rc;
      alpha_dev = alpha_tmp;
    }
    for (int k = 0; k < 4; k++) cur[k] = out[k];
    n = n_out_log;
    fold_step -= step;
    iter++;
  }
  return STWO_HIP_OK;
}

// LineEvaluation::interpolate on the host (STWO/prover/line.rs:54-99): the
// last FRI layer has at most 2^(10 + 16) values and usually 2^1..2^4.
static void host_line_interpolate(std::vector<qm31> &vals, uint32_t line_initial, uint32_t log_n) {
  size_t n = (size_t)1 << log_n;
  for (size_t i = 0; i < n; i++) {
    size_t j = bitrev32((uint32_t)i, log_n);
    if (j > i) std::swap(vals[i], vals[j]);
  }
  uint32_t init = line_initial, lg = log_n;
  while (lg >= 1) {
    size_t size = (size_t)1 << lg;
    cpoint c = host_index_to_point(init), st = host_index_to_point(coset_step(lg));
    for (size_t i = 0; i < size / 2; i++) {
      uint32_t xinv = m31_inv(c.x);
      for (size_t base = 0; base < n; base += size) {
        qm31 &a = vals[base + i], &b = vals[base + i + size / 2];
        qm31 s = qm31_add(a, b), d = qm31_mul_m31(qm31_sub(a, b), xinv);
        a = s;
        b = d;
      }
      c = cp_add(c, st);
    }
    init = (uint32_t)(((uint64_t)init * 2) & IDX_MASK);
    lg--;
  }
  uint32_t inv = m31_inv((uint32_t)(n % P));
  for (auto &v : vals) v = qm31_mul_m31(v, inv);
}

static inline size_t layer_off(uint32_t l) { return (((size_t)1 << l) - 1) * 8; }

}  // namespace stwo_hip

using namespace stwo_hip;

extern "C" {

int stwo_hip_fold_circle_into_line(stwo_hip_ctx *ctx, uint32_t *const dst[4], const uint32_t *const src[4],
                                   stwo_hip_coset src_domain, const uint32_t alpha[4], const stwo_hip_twiddles *tw) {
  if (!ctx) return STWO_HIP_EINVAL;
  STWO_HIP_CHECK_ARG(ctx, dst && src && alpha, "fold_circle_into_line: NULL argument");
  for (int k = 0; k < 4; k++) STWO_HIP_CHECK_ARG(ctx, dst[k] && src[k], "fold_circle_into_line: NULL coordinate");
  int rc = check_line_domain(ctx, src_domain, tw);
  if (rc) return rc;
  uint32_t N = src_domain.log_size + 1;
  STWO_HIP_CHECK_ARG(ctx, N >= 3, "fold_circle_into_line: domain of log size %u is below 3", N);
  return fold_circle(ctx, dst, src, N, qm31_make(alpha[0], alpha[1], alpha[2], alpha[3]), tw, true);
}

int stwo_hip_fold_line(stwo_hip_ctx *ctx, const uint32_t *const src[4], stwo_hip_coset line_domain,
                       const uint32_t alpha[4], uint32_t fold_step, const stwo_hip_twiddles *tw,
                       uint32_t *const dst[4]) {
  if (!ctx) return STWO_HIP_EINVAL;
  STWO_HIP_CHECK_ARG(ctx, dst && src && alpha, "fold_line: NULL argument");
  for (int k = 0; k < 4; k++) STWO_HIP_CHECK_ARG(ctx, dst[k] && src[k], "fold_line: NULL coordinate");
  STWO_HIP_CHECK_ARG(ctx, fold_step >= 1 && fold_step <= line_domain.log_size,
                     "fold_line: fold_step %u invalid for log size %u", fold_step, line_domain.log_size);
  int rc = check_line_domain(ctx, line_domain, tw);
  if (rc) return rc;
  return fold_line_steps(ctx, src, line_domain.log_size, qm31_make(alpha[0], alpha[1], alpha[2], alpha[3]), fold_step,
                         tw, dst);
}

}  // extern "C"

namespace stwo_hip {
// The layer schedule of FriProver::commit (fri.rs:188-262): the first
// (circle) layer of log N folds once into the line domain of log N - 1;
// inner layers fold line_fold_step at a time, the last one exactly down to
// the last layer of log (log_last_layer_degree_bound + log_blowup_factor).
std::vector<FriLayerShape> fri_schedule(const stwo_hip_fri_config &cfg, uint32_t log_size) {
  const uint32_t last_log = cfg.log_last_layer_degree_bound + cfg.log_blowup_factor;
  std::vector<FriLayerShape> out;
  out.push_back({log_size, 1});
  uint32_t lg = log_size - 1;
  if (lg != last_log) {
    for (;;) {
      bool last = !(lg > last_log + cfg.line_fold_step);
      uint32_t step = last ? lg - last_log : cfg.line_fold_step;
      out.push_back({lg, step});
      lg -= step;
      if (last) break;
    }
  }
  return out;
}

static int check_fri_args(stwo_hip_ctx *ctx, const stwo_hip_fri_config &cfg, uint32_t log_size,
                          const stwo_hip_twiddles *tw) {
  const uint32_t last_log = cfg.log_last_layer_degree_bound + cfg.log_blowup_factor;
  STWO_HIP_CHECK_ARG(ctx, cfg.line_fold_step >= 1, "Line fold step must be positive.");
  // A step above the largest line domain (log 27) can only overshoot; larger
  // values would also wrap the layer-size arithmetic of the schedule.
  STWO_HIP_CHECK_ARG(ctx, cfg.line_fold_step <= 28, "line_fold_step %u exceeds 28", cfg.line_fold_step);
  STWO_HIP_CHECK_ARG(ctx, cfg.log_last_layer_degree_bound <= 10, "log_last_layer_degree_bound must be <= 10");
  STWO_HIP_CHECK_ARG(ctx, cfg.log_blowup_factor >= 1 && cfg.log_blowup_factor <= 16, "log_blowup_factor not in 1..=16");
  STWO_HIP_CHECK_ARG(ctx, log_size >= 3 && log_size - 1 >= last_log && log_size <= 28,
                     "fri_commit: log size %u incompatible with last layer log %u", log_size, last_log);
  stwo_hip_coset dom = {half_odds_initial(log_size - 1), log_size - 1};
  return check_line_domain(ctx, dom, tw);
}

// grind: NULL, or (prove) the end of the commit and the proof of work's first
// search range run on the device when the last layer allows
// (fri_last_layer_kernel): grind->found then says whether that range held
// the nonce.
struct FriGrind {
  uint32_t pow_bits;
  bool found;
  uint64_t nonce;
};
// A commit on its way through the layers (FriProver::commit).  With `keep`,
// every committed layer's tree and every folded evaluation stays in
// `keep->mem` (laid out by the caller from fri_schedule); without, one scratch
// tree and two layer buffers are reused, and a last layer of at most
// 2^kDevLastMax values lies in the state, for one download of both.
struct FriChain {
  stwo_hip_fri_config cfg;
  uint32_t log_size;
  const uint32_t *column[4];
  uint32_t *tree, *lay[2], *state, *counters;
  stwo_hip_fri_prover *keep;

  // The layer to commit next (done: the last layer, not committed): its log,
  // its evaluation (from cur on, coordinates 2^lg words apart; the first
  // layer's is `column`) and the fold that writes it from src, if not launched
  // yet: the circle fold or `pending` line folds.
  uint32_t lg, last_log, nr, n_folds, line_init, pending;
  bool first, circle, done;
  uint32_t *cur;
  const uint32_t *src[4];

  void start() {
    last_log = cfg.log_last_layer_degree_bound + cfg.log_blowup_factor;
    lg = log_size;
    nr = n_folds = line_init = pending = 0;
    first = true;
    circle = done = false;
    cur = nullptr;
    for (int k = 0; k < 4; k++) src[k] = column[k];
  }
  bool last_in_state() const { return !keep && last_log <= kDevLastMax; }
  uint32_t *layer_tree() const { return keep ? keep->layers[nr].tree : tree; }
  // The layer at lg is committed: on to the next (fri.rs:188-262).
  void next() {
    const uint32_t step = first ? 1 : std::min(cfg.line_fold_step, lg - last_log);
    for (int k = 0; k < 4; k++) {
      src[k] = first ? column[k] : cur + ((size_t)k << lg);
      if (keep) keep->layers[nr].cols[k] = src[k];
    }
    lg -= step;
    line_init = first ? half_odds_initial(lg) : (uint32_t)(((uint64_t)line_init << step) & IDX_MASK);
    circle = first;
    pending = step;
    first = false;
    done = lg == last_log;
    cur = keep                      ? keep->evals[n_folds]
          : done && last_in_state() ? state + kPolyOff
                                    : lay[n_folds & 1];
    n_folds++;
    nr++;
  }
  // The remaining layers are the tail's.
  bool in_tail() const { return !first && lg <= kTailLog && cfg.line_fold_step <= 4; }
};

// Launches the pending fold on its own (a line fold of more than 4 steps, or
// the fold into the last layer when no tail runs).
static int fri_flush(stwo_hip_ctx *ctx, FriChain &c, const stwo_hip_twiddles *tw) {
  if (!c.pending) return STWO_HIP_OK;
  const qm31 unused = qm31_make(0, 0, 0, 0);
  uint32_t *dst[4];
  for (int k = 0; k < 4; k++) dst[k] = c.cur + ((size_t)k << c.lg);
  const uint32_t src_log = c.lg + c.pending, step = c.pending;
  uint32_t *alpha = c.state + kAlphaOff;
  int rc = c.circle ? fold_circle(ctx, dst, c.src, src_log, unused, tw, false, alpha)
                    : fold_line_steps(ctx, c.src, src_log, unused, step, tw, dst, alpha, c.state + kAlphaTmpOff);
  c.pending = 0;
  for (int k = 0; k < 4; k++) c.src[k] = dst[k];
  return rc;
}

// Runs the chains (each with its channel in its state; a lone one with it in
// `digest`) up to their last layers: on the stream, without host round trips.  After each
// layer's Merkle commit, the kernel that hashes its root (fri_layer_kernel
// or the tail) mixes the root into the device copy of the channel and
// draws the next alpha, which the folds read from device memory.
//
// A chain is a row of dependent launches that leave the device nearly idle, so
// chains that stand at the same layer size share theirs (the larger ones begin
// alone): 12 commits of 2^13 and 2^17 one after another took 2.6 ms of
// device time, side by side they take 0.5 ms.
static int fri_run(stwo_hip_ctx *ctx, FriChain *const *chains, size_t n, const stwo_hip_twiddles *tw,
                   const uint8_t *digest = nullptr) {
  const uint32_t *itw_end = tw->d_itw + tw->len;
  int rc;
  for (;;) {
    FriChain *lead = nullptr;
    for (size_t i = 0; i < n; i++) {
      FriChain *c = chains[i];
      if (!c->done && !c->in_tail() && (!lead || c->lg > lead->lg)) lead = c;
    }
    if (!lead) break;
    auto kind = [](const FriChain &c) { return c.circle && c.pending ? kFoldCircle : (int)c.pending; };
    if (lead->pending > 4) {
      rc = fri_flush(ctx, *lead, tw);
      if (rc) return rc;
    }
    const int fold = kind(*lead);
    const uint32_t lg = lead->lg;
    FriLayerJobs jobs{};
    if (digest && lead->first) {
      memcpy(jobs.digest, digest, 32);
      jobs.has_digest = 1;
    }
    uint32_t nj = 0;
    for (size_t i = 0; i < n && nj < kFriJobs; i++) {
      FriChain &c = *chains[i];
      if (c.done || c.in_tail() || c.lg != lg || kind(c) != fold) continue;
      if (c.nr >= kMaxRoots || (c.keep && c.nr >= c.keep->layers.size()))
        return set_error(ctx, STWO_HIP_EINVAL, "internal: FRI layer overflow");
      FriLayerJob &j = jobs.j[nj++];
      for (int k = 0; k < 4; k++) j.src[k] = c.src[k];
      j.dst = c.cur;
      j.tree = c.layer_tree();
      j.state = c.state;
      j.counters = c.counters;
      j.root = c.nr;
      c.next();
    }
    switch (fold) {
      case 0: rc = launch_fri_layer<0>(ctx, jobs, nj, itw_end, lg); break;
      case 1: rc = launch_fri_layer<1>(ctx, jobs, nj, itw_end, lg); break;
      case 2: rc = launch_fri_layer<2>(ctx, jobs, nj, itw_end, lg); break;
      case 3: rc = launch_fri_layer<3>(ctx, jobs, nj, itw_end, lg); break;
      case 4: rc = launch_fri_layer<4>(ctx, jobs, nj, itw_end, lg); break;
      default: rc = launch_fri_layer<kFoldCircle>(ctx, jobs, nj, itw_end, lg); break;
    }
    if (rc) return rc;
  }
  // Every remaining inner layer of a chain (at most kTailLog of them) in one workgroup.
  std::vector<FriTail> tails;
  for (size_t i = 0; i < n; i++) {
    FriChain &c = *chains[i];
    if (c.done) {
      rc = fri_flush(ctx, c, tw);
      if (rc) return rc;
      continue;
    }
    tails.emplace_back();
    FriTail &t = tails.back();
    memset(&t, 0, sizeof(t));
    for (int k = 0; k < 4; k++) t.src.c[k] = c.src[k];
    t.first = c.cur;
    t.fold = c.circle ? kFoldCircle : c.pending;
    t.root = c.nr;
    t.itw_end = itw_end;
    t.state = c.state;
    while (!c.done) {
      if (t.n >= kTailMax || c.nr >= kMaxRoots || (c.keep && c.nr >= c.keep->layers.size()))
        return set_error(ctx, STWO_HIP_EINVAL, "internal: FRI tail overflow");
      FriTailLayer &L = t.l[t.n++];
      L.lg = c.lg;
      L.tree = c.layer_tree();
      c.next();
      L.step = c.pending;
      L.dst = c.cur;
    }
    c.pending = 0;
  }
  if (tails.empty()) return STWO_HIP_OK;
  if (tails.size() == 1)
    return launch(ctx, "fri_tail", fri_tail_kernel, dim3(1), dim3(kTreeThreads), 0, tails[0]);
  void *d_tails = nullptr;
  rc = upload_table(ctx, tails.data(), tails.size() * sizeof(FriTail), &d_tails);
  if (rc) return rc;
  return launch(ctx, "fri_tail", fri_tails_kernel, dim3((uint32_t)tails.size()), dim3(kTreeThreads), 0,
                (const FriTail *)d_tails);
}

// The end of a commit on the host, from the downloaded state and the last
// layer's evaluation (4 coordinates of 2^lg words): fri.rs:274-291.
static int fri_finish(stwo_hip_ctx *ctx, const FriChain &c, const uint32_t *st, const uint32_t *h,
                      uint8_t channel_digest[32], uint32_t *channel_n_draws, uint32_t *roots, uint32_t *n_roots,
                      uint32_t *last_layer_poly) {
  if (st[9]) return set_error(ctx, STWO_HIP_EDEVICE, "fri_commit: channel draw did not terminate");
  memcpy(roots, st + kRootsOff, 32 * c.nr);
  HostChannel ch;
  memcpy(ch.digest, st, 32);
  ch.n_draws = st[8];
  const size_t n = (size_t)1 << c.lg;
  std::vector<qm31> vals(n);
  for (size_t i = 0; i < n; i++) vals[i] = qm31_make(h[i], h[n + i], h[2 * n + i], h[3 * n + i]);
  host_line_interpolate(vals, c.line_init, c.lg);
  // into_ordered_coefficients: bit reverse (line.rs:157-160)
  for (size_t i = 0; i < n; i++) {
    size_t j = bitrev32((uint32_t)i, c.lg);
    if (j > i) std::swap(vals[i], vals[j]);
  }
  size_t bound = (size_t)1 << c.cfg.log_last_layer_degree_bound;
  for (size_t i = bound; i < n; i++)
    for (int k = 0; k < 4; k++)
      if (vals[i].v[k]) return set_error(ctx, STWO_HIP_EDEGREE, "invalid degree");
  // from_ordered_coefficients bit-reverses the kept coefficients (line.rs:167-170)
  for (size_t i = 0; i < bound; i++) {
    size_t j = bitrev32((uint32_t)i, c.cfg.log_last_layer_degree_bound);
    for (int k = 0; k < 4; k++) last_layer_poly[4 * j + k] = vals[i].v[k];
  }
  ch.mix_felts(last_layer_poly, bound);
  memcpy(channel_digest, ch.digest, 32);
  *channel_n_draws = ch.n_draws;
  *n_roots = c.nr;
  return STWO_HIP_OK;
}

static int fri_commit_impl(stwo_hip_ctx *ctx, uint8_t channel_digest[32], uint32_t *channel_n_draws,
                           const stwo_hip_fri_config &cfg, const uint32_t *const column[4], uint32_t log_size,
                           const stwo_hip_twiddles *tw, uint32_t *roots, uint32_t *n_roots, uint32_t *last_layer_poly,
                           stwo_hip_fri_prover *keep, FriGrind *grind = nullptr) {
  int rc = check_fri_args(ctx, cfg, log_size, tw);
  if (rc) return rc;
  if (keep && keep->layers.size() != fri_schedule(cfg, log_size).size())
    return set_error(ctx, STWO_HIP_EINVAL, "internal: FRI prover storage does not match the schedule");
  FriChain c{};
  c.cfg = cfg;
  c.log_size = log_size;
  c.keep = keep;
  c.counters = ctx->d_counters;
  for (int k = 0; k < 4; k++) c.column[k] = column[k];
  void *p = nullptr;
  if (!keep) {
    rc = get_scratch(ctx, "fri_tree", layer_off(log_size + 1) * 4, &p);
    if (rc) return rc;
    c.tree = (uint32_t *)p;
    for (int k = 0; k < 2; k++) {
      rc = get_scratch(ctx, k ? "fri_layer_b" : "fri_layer_a", ((size_t)4 << (log_size - 1)) * 4, &p);
      if (rc) return rc;
      c.lay[k] = (uint32_t *)p;
    }
  }
  rc = get_scratch(ctx, "fri_state", kFriStateWords * 4, &p);
  if (rc) return rc;
  uint32_t *state = c.state = (uint32_t *)p;
  c.start();
  FriChain *chain = &c;
  rc = fri_run(ctx, &chain, 1, tw, channel_digest);
  if (rc) return rc;
  const uint32_t nr = c.nr, lg = c.lg;
  if (grind) grind->found = false;
  if (grind && lg <= kDevLastMax && grind->pow_bits + 6 < 20) {
    // The last layer, the channel mix and the grind's first range on the
    // device, then one synchronization.
    const uint32_t bound_log = cfg.log_last_layer_degree_bound;
    LastLayerArgs la{};
    for (int k = 0; k < 4; k++) la.src[k] = c.cur + ((size_t)k << lg);
    la.itw_end = tw->d_itw + tw->len;
    la.lg = lg;
    la.bound_log = bound_log;
    la.pow_bits = grind->pow_bits;
    la.n_inv = m31_inv((uint32_t)(((uint64_t)1 << lg) % P));
    la.chan = state;
    la.poly = state + kPolyOff;
    la.prefixed = state + kPrefixOff;
    la.flags = state + kFlagsOff;
    la.best = (unsigned long long *)(state + kBestOff);
    rc = launch(ctx, "fri_last_layer", fri_last_layer_kernel, dim3(1), dim3(256), 0, la);
    if (rc) return rc;
    rc = grind_first_range(ctx, state + kPrefixOff, grind->pow_bits, la.best);
    if (rc) return rc;
    const size_t bound = (size_t)1 << bound_log;
    std::vector<uint32_t> st(kPolyOff + 4 * bound);
    {
      const DownloadReq req = {st.data(), state, st.size()};
      rc = download_many(ctx, &req, 1);
      if (rc) return rc;
    }
    if (st[9]) return set_error(ctx, STWO_HIP_EDEVICE, "fri_commit: channel draw did not terminate");
    if (st[kFlagsOff]) return set_error(ctx, STWO_HIP_EDEGREE, "invalid degree");
    memcpy(roots, st.data() + kRootsOff, 32 * nr);
    if (keep)
      for (uint32_t k = 0; k < nr; k++) memcpy(keep->layers[k].root, roots + 8 * k, 32);
    memcpy(last_layer_poly, st.data() + kPolyOff, 16 * bound);
    memcpy(channel_digest, st.data(), 32);
    *channel_n_draws = st[8];
    uint64_t best;
    memcpy(&best, st.data() + kBestOff, 8);
    if (best != ~0ull) {
      grind->found = true;
      grind->nonce = best;
    }
    *n_roots = nr;
    if (keep) {
      keep->last_layer_poly.assign(last_layer_poly, last_layer_poly + 4 * bound);
      keep->last_log = lg;
      for (int k = 0; k < 4; k++) keep->last_layer_eval[k] = c.cur + ((size_t)k << lg);
    }
    return STWO_HIP_OK;
  }
  // One synchronization for the channel state, the roots and the last layer.
  std::vector<uint32_t> st(kPolyOff + ((size_t)4 << lg));
  {
    const bool one = c.last_in_state();
    const DownloadReq reqs[2] = {{st.data(), state, one ? st.size() : kRootsOff + 8 * nr},
                                 {st.data() + kPolyOff, c.cur, (size_t)4 << lg}};
    rc = download_many(ctx, reqs, one ? 1 : 2);
    if (rc) return rc;
  }
  rc = fri_finish(ctx, c, st.data(), st.data() + kPolyOff, channel_digest, channel_n_draws, roots, n_roots,
                  last_layer_poly);
  if (rc) return rc;
  if (keep) {
    for (uint32_t k = 0; k < nr; k++) memcpy(keep->layers[k].root, roots + 8 * k, 32);
    keep->last_layer_poly.assign(last_layer_poly, last_layer_poly + ((size_t)4 << cfg.log_last_layer_degree_bound));
    keep->last_log = lg;
    for (int k = 0; k < 4; k++) keep->last_layer_eval[k] = c.cur + ((size_t)k << lg);
  }
  return STWO_HIP_OK;
}

size_t fri_job_words(uint32_t log_size) { return kFriStateWords + tree_counters(log_size); }

int fri_commit_jobs(stwo_hip_ctx *ctx, FriJob *jobs, size_t n, const stwo_hip_twiddles *tw, uint32_t *mem) {
  int rc;
  std::vector<FriChain> chains(n);
  std::vector<FriChain *> order(n);
  // the states, then every job's counters
  uint32_t *counters = mem + n * kFriStateWords;
  ChanInits init{};
  uint32_t ni = 0;
  auto send = [&]() {
    const int r = launch(ctx, "fri_chan_init", chan_inits_kernel, dim3(ni), dim3(64), 0, init);
    ni = 0;
    return r;
  };
  for (size_t i = 0; i < n; i++) {
    FriJob &j = jobs[i];
    rc = check_fri_args(ctx, j.cfg, j.log_size, tw);
    if (rc) return rc;
    FriChain &c = chains[i];
    c = FriChain{};
    c.cfg = j.cfg;
    c.log_size = j.log_size;
    for (int k = 0; k < 4; k++) c.column[k] = j.column[k];
    c.tree = j.tree;
    c.lay[0] = j.layers;
    c.lay[1] = j.layers + ((size_t)4 << (j.log_size - 1));
    c.state = mem + i * kFriStateWords;
    c.counters = counters;
    init.c[ni++] = {c.state, j.tree, counters, tree_counters(j.log_size)};
    counters += tree_counters(j.log_size);
    c.start();
    order[i] = &c;
    if (ni == kFriJobs || i + 1 == n) {
      rc = send();
      if (rc) return rc;
    }
  }
  rc = fri_run(ctx, order.data(), n, tw);
  if (rc) return rc;
  // One download of the states, with the last layers of the usual sizes in them.
  std::vector<uint32_t> st(n * kFriStateWords);
  std::vector<std::vector<uint32_t>> big(n);
  std::vector<DownloadReq> reqs = {{st.data(), mem, st.size()}};
  for (size_t i = 0; i < n; i++) {
    const FriChain &c = chains[i];
    if (c.last_in_state()) continue;
    big[i].resize((size_t)4 << c.lg);
    reqs.push_back({big[i].data(), c.cur, big[i].size()});
  }
  rc = download_many(ctx, reqs.data(), reqs.size());
  if (rc) return rc;
  for (size_t i = 0; i < n; i++) {
    const uint32_t *s = st.data() + i * kFriStateWords;
    memcpy(jobs[i].mixed_root, s + kMixedOff, 32);
    uint32_t n_draws = 0;
    rc = fri_finish(ctx, chains[i], s, big[i].empty() ? s + kPolyOff : big[i].data(), jobs[i].digest, &n_draws,
                    jobs[i].roots, &jobs[i].n_roots, jobs[i].last_layer_poly);
    if (rc) return rc;
  }
  return STWO_HIP_OK;
}

}  // namespace stwo_hip

extern "C" {

int stwo_hip_fri_commit(stwo_hip_ctx *ctx, uint8_t channel_digest[32], uint32_t *channel_n_draws,
                        stwo_hip_fri_config cfg, const uint32_t *const column[4], uint32_t log_size,
                        const stwo_hip_twiddles *tw, uint32_t *roots, uint32_t *n_roots, uint32_t *last_layer_poly) {
  if (!ctx) return STWO_HIP_EINVAL;
  STWO_HIP_CHECK_ARG(ctx, channel_digest && channel_n_draws && column && roots && n_roots && last_layer_poly,
                     "fri_commit: NULL argument");
  return fri_commit_impl(ctx, channel_digest, channel_n_draws, cfg, column, log_size, tw, roots, n_roots,
                         last_layer_poly, nullptr);
}

int stwo_hip_fri_prover_commit(stwo_hip_ctx *ctx, uint8_t channel_digest[32], uint32_t *channel_n_draws,
                               stwo_hip_fri_config cfg, const uint32_t *const column[4], uint32_t log_size,
                               const stwo_hip_twiddles *tw, uint32_t *roots, uint32_t *n_roots,
                               uint32_t *last_layer_poly, stwo_hip_fri_prover **out) {
  return fri_prover_commit_mem(ctx, channel_digest, channel_n_draws, cfg, column, log_size, tw, roots, n_roots,
                               last_layer_poly, nullptr, out, -1, nullptr, nullptr);
}

}  // extern "C"

int stwo_hip::fri_prover_commit_mem(stwo_hip_ctx *ctx, uint8_t channel_digest[32], uint32_t *channel_n_draws,
                                    stwo_hip_fri_config cfg, const uint32_t *const column[4], uint32_t log_size,
                                    const stwo_hip_twiddles *tw, uint32_t *roots, uint32_t *n_roots,
                                    uint32_t *last_layer_poly, const char *scratch_key, stwo_hip_fri_prover **out,
                                    int pow_bits, uint64_t *nonce, bool *nonce_found) {
  if (!ctx) return STWO_HIP_EINVAL;
  STWO_HIP_CHECK_ARG(ctx, channel_digest && channel_n_draws && column && roots && n_roots && last_layer_poly && out,
                     "fri_prover_commit: NULL argument");
  *out = nullptr;
  for (int k = 0; k < 4; k++) STWO_HIP_CHECK_ARG(ctx, column[k] != nullptr, "fri_prover_commit: NULL column");
  int rc = check_fri_args(ctx, cfg, log_size, tw);
  if (rc) return rc;
  auto *pr = new stwo_hip_fri_prover();
  pr->device = ctx->device;
  pr->cfg = cfg;
  pr->log_size = log_size;
  const std::vector<FriLayerShape> sched = fri_schedule(cfg, log_size);
  // One allocation: a packed tree per committed layer, then the evaluation
  // written by each fold (the last one is the uncommitted last layer).
  size_t words = 0;
  std::vector<size_t> tree_off, eval_off;
  for (const FriLayerShape &l : sched) {
    tree_off.push_back(words);
    words += layer_off(l.log_size + 1);
  }
  uint32_t lg = log_size;
  for (size_t f = 0; f < sched.size(); f++) {
    lg -= sched[f].fold_step;
    eval_off.push_back(words);
    words += (size_t)4 << lg;
  }
  if (scratch_key) {
    void *m = nullptr;
    rc = get_scratch(ctx, scratch_key, words * 4, &m);
    pr->mem = (uint32_t *)m;
    pr->owns_mem = false;
  } else {
    rc = stwo_hip_alloc(ctx, words, &pr->mem);
  }
  if (rc) {
    delete pr;
    return rc;
  }
  pr->mem_words = words;
  pr->layers.resize(sched.size());
  for (size_t k = 0; k < sched.size(); k++) {
    pr->layers[k].shape = sched[k];
    pr->layers[k].tree = pr->mem + tree_off[k];
  }
  for (size_t f = 0; f < sched.size(); f++) pr->evals.push_back(pr->mem + eval_off[f]);
  FriGrind g{};
  if (pow_bits >= 0) g.pow_bits = (uint32_t)pow_bits;
  rc = fri_commit_impl(ctx, channel_digest, channel_n_draws, cfg, column, log_size, tw, roots, n_roots,
                       last_layer_poly, pr, pow_bits >= 0 ? &g : nullptr);
  if (!rc && nonce_found) {
    *nonce_found = g.found;
    if (g.found) *nonce = g.nonce;
  }
  if (rc) {
    if (pr->owns_mem) stwo_hip_free(ctx, pr->mem);
    delete pr;
    return rc;
  }
  *out = pr;
  return STWO_HIP_OK;
}

extern "C" {

// FriProver::decommit (fri.rs:294-347): draw the query positions from the
// channel (draw_queries, core/queries.rs:11-28; Queries::new sorts and
// deduplicates), then decommit every committed layer:
// compute_decommitment_positions_and_witness_evals (fri.rs:455-489) with the
// layer's fold step (1 for the circle layer), and the Merkle decommitment
// of the layer's tree on those positions; the queries fold by the layer's
// step between layers (Queries::fold, queries.rs:56-63).  Every value and
// hash read of all layers is one device gather.
int stwo_hip_fri_prover_decommit(stwo_hip_ctx *ctx, stwo_hip_fri_prover *pr, uint8_t channel_digest[32],
                                 uint32_t *channel_n_draws, uint32_t *query_positions, uint32_t *n_positions,
                                 uint32_t *unsorted_queries) {
  if (!ctx) return STWO_HIP_EINVAL;
  STWO_HIP_CHECK_ARG(ctx, query_positions && n_positions && unsorted_queries, "fri_prover_decommit: NULL argument");
  STWO_HIP_CHECK_ARG(ctx, channel_digest && channel_n_draws, "fri_prover_decommit: NULL argument");
  // The channel is written back only on success.
  uint8_t digest[32];
  memcpy(digest, channel_digest, 32);
  uint32_t n_draws = *channel_n_draws;
  Gatherer g;
  FriDecommitPlan plan;
  int rc = fri_decommit_plan(ctx, pr, digest, &n_draws, g, plan);
  if (rc) return rc;
  rc = g.run(ctx);
  if (rc) return rc;
  memcpy(channel_digest, digest, 32);
  *channel_n_draws = n_draws;
  memcpy(query_positions, plan.queries.data(), plan.queries.size() * 4);
  *n_positions = (uint32_t)plan.queries.size();
  memcpy(unsorted_queries, plan.raw.data(), plan.raw.size() * 4);
  fri_decommit_finish(pr, g, plan);
  return STWO_HIP_OK;
}

}  // extern "C"

extern "C" {

int stwo_hip_fri_prover_layer_proof(stwo_hip_ctx *ctx, const stwo_hip_fri_prover *pr, uint32_t layer,
                                    uint32_t commitment[8], uint32_t *fri_witness, size_t fri_cap, size_t *n_fri,
                                    uint32_t *hash_witness, size_t hash_cap, size_t *n_hash, uint32_t *positions,
                                    uint32_t *values, size_t pos_cap, size_t *n_pos) {
  if (!ctx) return STWO_HIP_EINVAL;
  STWO_HIP_CHECK_ARG(ctx, pr && commitment && n_fri && n_hash && n_pos, "fri_prover_layer_proof: NULL argument");
  STWO_HIP_CHECK_ARG(ctx, pr->decommitted, "fri_prover_layer_proof: not decommitted yet");
  STWO_HIP_CHECK_ARG(ctx, layer < pr->proofs.size(), "fri_prover_layer_proof: layer %u of %zu", layer,
                     pr->proofs.size());
  const FriLayerDecommit &d = pr->proofs[layer];
  memcpy(commitment, pr->layers[layer].root, 32);
  *n_fri = d.fri_witness.size() / 4;
  *n_hash = d.hash_witness.size() / 8;
  *n_pos = d.positions.size();
  if (!fri_witness && !hash_witness && !positions) return STWO_HIP_OK;  // size query
  STWO_HIP_CHECK_ARG(ctx, *n_fri <= fri_cap && *n_hash <= hash_cap && (!positions || *n_pos <= pos_cap),
                     "fri_prover_layer_proof: capacity too small (%zu, %zu, %zu needed)", *n_fri, *n_hash, *n_pos);
  STWO_HIP_CHECK_ARG(ctx, (fri_witness || !*n_fri) && (hash_witness || !*n_hash),
                     "fri_prover_layer_proof: NULL output");
  if (*n_fri) memcpy(fri_witness, d.fri_witness.data(), d.fri_witness.size() * 4);
  if (*n_hash) memcpy(hash_witness, d.hash_witness.data(), d.hash_witness.size() * 4);
  if (positions) {
    memcpy(positions, d.positions.data(), d.positions.size() * 4);
    if (values) memcpy(values, d.values.data(), d.values.size() * 4);
  }
  return STWO_HIP_OK;
}

int stwo_hip_fri_prover_destroy(stwo_hip_ctx *ctx, stwo_hip_fri_prover *prover) {
  if (!ctx) return STWO_HIP_EINVAL;
  if (!prover) return STWO_HIP_OK;
  int rc = stwo_hip_sync(ctx);
  int rc2 = prover->owns_mem ? stwo_hip_free(ctx, prover->mem) : STWO_HIP_OK;
  delete prover;
  return rc ? rc : rc2;
}

}  // extern "C"
