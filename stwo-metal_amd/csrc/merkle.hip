// Blake2s Merkle commitments: mixed-degree (MerkleOps::commit_on_layer,
// MerkleProver::commit) and lifted (MerkleOpsLifted).
//
// One hash per lane.  A node's message is streamed in 64-byte blocks exactly
// as the `blake2` crate buffers it (the last block, full or partial, is the
// finalized one, `t` counts the bytes so far):
//   mixed node i  = [prev[2i] || prev[2i+1]] || le32(c0[i]) || le32(c1[i]) || ...
//                   (STWO/core/vcs/blake2_merkle.rs:17-38, SIMD/blake2s.rs:60-144)
//   lifted leaf i = le32(c[lift(i, L - log c)]) for columns in ascending
//                   length order (CPUB/merkle_lifted.rs:44-78)
//   lifted node i = prev[2i] || prev[2i+1] (vcs_lifted/blake2_merkle.rs:18-27)
// Column words of one block are 16 columns at the same row: lane i reads
// column c at row i, so each load instruction is a coalesced run over the
// wave.  Column pointers come from a per-call device table (uniform across
// the wave -> scalar loads).
//
// A run of node layers without injected columns, to the next injected layer or
// the root, is one launch of `merkle_nodes_kernel` (two where its workgroups would
// meet on more counters than there are): each workgroup hashes a subtree through
// LDS, writing every layer to global memory, and the last of each group of
// workgroups to finish hashes on (merkle_dev.hpp).
#include <algorithm>
#include <type_traits>
#include <vector>

#include "blake2s.hpp"
#include "common.hpp"
#include "field.hpp"
#include "internal.hpp"
#include "merkle_dev.hpp"

namespace stwo_hip {


__device__ __forceinline__ void load_block64(uint32_t m[16], const uint32_t *src) {
  const uint4 *s = reinterpret_cast<const uint4 *>(src);
#pragma unroll
  for (int k = 0; k < 4; k++) {
    uint4 v = s[k];
    m[4 * k] = v.x;
    m[4 * k + 1] = v.y;
    m[4 * k + 2] = v.z;
    m[4 * k + 3] = v.w;
  }
}

__device__ __forceinline__ b2_state hash_block(const uint32_t m[16], uint32_t m31) {
  b2_state s;
  b2_init(s);
  b2_compress(s, m, 64, true);
  if (m31)
#pragma unroll
    for (int k = 0; k < 8; k++) s.h[k] = b2_reduce_word(s.h[k]);
  return s;
}
// Node i: H(prev[2i] || prev[2i+1]), stored to out.
__device__ __forceinline__ b2_state hash_node(const uint32_t *prev, uint32_t i, uint32_t *out, uint32_t m31) {
  uint32_t m[16];
  load_block64(m, prev + 16 * (size_t)i);
  const b2_state s = hash_block(m, m31);
  store_hash(out + 8 * (size_t)i, s, 0);
  return s;
}
__device__ __forceinline__ b2_state hash_pair(const b2_state &a, const b2_state &b, uint32_t m31) {
  uint32_t m[16];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    m[k] = a.h[k];
    m[8 + k] = b.h[k];
  }
  return hash_block(m, m31);
}

// Word at byte `off` of a column.  Layers are at most 2^30 rows, so the offset
// fits 32 bits: the load takes the column pointer as an SGPR base and a
// 32-bit lane offset (no per-column 64-bit address arithmetic).
__device__ __forceinline__ uint32_t ld_col_byte(const uint32_t *col, uint32_t off) {
  return *(gconst_u32 *)((gconst_u8 *)as_global(col) + off);
}
__device__ __forceinline__ uint32_t ld_col_word(const uint32_t *col, uint32_t idx) { return ld_col_byte(col, idx << 2); }

// Mixed-degree layer: optional previous layer, then the layer's columns.
// `lifted` selects the lifted leaf index for column words.
// AHEAD: each block's column words are loaded one compression ahead, so
// their latency overlaps the previous compression.  Used for layers of few
// nodes, where a node's chain of blocks is the launch's critical path; on
// large layers the other waves hide the latency and the extra registers and
// copies cost more than they save.
// TABLE: the columns' table is in device memory (not among the arguments,
// whose address must not be taken).
template <bool AHEAD, bool TABLE>
__device__ __forceinline__ b2_state layer_hash(const MerkleLayer &L, const ColRef *cols, uint32_t i) {
  const uint32_t *prev = L.prev;
  const uint32_t n_cols = L.n_cols, lifted = L.lifted;
  // The words of columns c0 .. c0 + 15 at this row (zeros past n_cols).  A full
  // block reads its 16 table entries together, and where the columns lie at the
  // layer's own size they share one offset: entry by entry, each with its wait
  // and its offset, a block cost 48 more instructions beside the compression's
  // 976.  256 columns of 2^20 committed at blowup 4: 6.07 -> 6.00 ms.
  auto load_cols = [&](uint32_t c0, uint32_t (&dst)[16]) {
    const uint32_t cnt = min(16u, n_cols - c0);
    if (cnt == 16) {
      uint64_t ref[32];  // a ColRef each two, by scalar loads of 64 bytes
      if (TABLE) {
        typedef const __attribute__((address_space(4))) uint64_t const_u64;
        const_u64 *src = (const_u64 *)readfirstlane_u64((uint64_t)(cols + c0));
#pragma unroll
        for (uint32_t k = 0; k < 32; k++) ref[k] = src[k];
      } else {
        __builtin_memcpy(ref, cols + c0, sizeof(ref));
      }
      uint32_t shifts = 0;
#pragma unroll
      for (uint32_t k = 0; k < 16; k++) shifts |= (uint32_t)ref[2 * k + 1];
      uint32_t row4 = i << 2, odd4 = (i & 1) << 2;
      asm("" : "+v"(row4), "+v"(odd4));  // stays a 32-bit offset beside the pointer in SGPRs
      if (lifted && shifts) {
#pragma unroll
        for (uint32_t k = 0; k < 16; k++)
          dst[k] = ld_col_byte((const uint32_t *)ref[2 * k], ((i >> ((uint32_t)ref[2 * k + 1] + 1)) << 3) + odd4);
      } else {
#pragma unroll
        for (uint32_t k = 0; k < 16; k++) dst[k] = ld_col_byte((const uint32_t *)ref[2 * k], row4);
      }
      return;
    }
#pragma unroll
    for (uint32_t k = 0; k < 16; k++) {
      uint32_t v = 0;
      if (k < cnt) {
        const ColRef cr = cols[c0 + k];
        uint32_t idx = lifted ? (((i >> (cr.shift + 1)) << 1) + (i & 1)) : i;
        v = ld_col_word(cr.p, idx);
      }
      dst[k] = v;
    }
  };
  b2_state s;
  b2_init(s);
  uint32_t m[16], nx[16];
  uint32_t t = 0;
  if (AHEAD && n_cols) load_cols(0, nx);
  if (prev) {
    load_block64(m, prev + 16 * (size_t)i);
    t = 64;
    b2_compress(s, m, t, n_cols == 0);
  } else if (n_cols == 0) {
#pragma unroll
    for (int k = 0; k < 16; k++) m[k] = 0;
    b2_compress(s, m, 0, true);
  }
  for (uint32_t c0 = 0; c0 < n_cols; c0 += 16) {
    const uint32_t cnt = min(16u, n_cols - c0);
    if (AHEAD) {
#pragma unroll
      for (int k = 0; k < 16; k++) m[k] = nx[k];
      if (c0 + 16 < n_cols) load_cols(c0 + 16, nx);
    } else {
      load_cols(c0, m);
    }
    t += 4 * cnt;
    b2_compress(s, m, t, c0 + 16 >= n_cols);
  }
  if (L.m31)
#pragma unroll
    for (int k = 0; k < 8; k++) s.h[k] = b2_reduce_word(s.h[k]);
  return s;
}

// Layers of few nodes, where a node's hash is the launch's critical path: one
// node per quad (b2_compress_quad, about 380 instructions per lane instead of 960
// on one lane).  Same hash as layer_hash, of at most 16 columns, words j and 4 + j
// of it in lane j.
__device__ __forceinline__ void layer_hash_quad(const MerkleLayer &L, const ColRef *cols, uint32_t i, uint32_t &lo,
                                                uint32_t &hi) {
  const uint32_t j = threadIdx.x & 3;
  const uint32_t n_cols = L.n_cols;
  uint32_t w[16], m[16];
#pragma unroll
  for (uint32_t k = 0; k < 16; k++) {
    w[k] = 0;
    if (k < n_cols) {
      const ColRef cr = cols[k];
      w[k] = ld_col_word(cr.p, L.lifted ? (((i >> (cr.shift + 1)) << 1) + (i & 1)) : i);
    }
  }
  lo = b2_iv_lo(j);
  hi = b2_iv_hi(j);
  uint32_t t = 0;
  if (L.prev) {
    load_block64(m, L.prev + 16 * (size_t)i);
    t = 64;
    b2_compress_quad(lo, hi, m, t, n_cols == 0);
  }
  if (n_cols || !L.prev) b2_compress_quad(lo, hi, w, t + 4 * n_cols, true);
  if (L.m31) {
    lo = b2_reduce_word(lo);
    hi = b2_reduce_word(hi);
  }
}

// Small layers with many columns (up to 2^14 nodes): the chain
// of blocks per node is the critical path and, with one block loaded ahead,
// each block waits on a table load followed by a column load.  Here a
// workgroup owns 64 consecutive nodes (a quad each) and stages its columns
// through LDS in chunks of MQ_CHUNK columns: the chunk's column pointers
// first, then every column's 64 words (one coalesced 256-byte run per wave
// and load, 32 loads in flight per lane), so a chunk costs about two memory
// round trips and its blocks then read their words from LDS.  Same hash
// as layer_hash.  Lifted trees of 2^13 leaves over 12 to 98 columns, six in a
// launch: 47 us, with the loads a block ahead 65 us.
constexpr uint32_t MQ_CHUNK = 240;  // 15 blocks; 61,440 B of words + 2,880 B of pointers and shifts
struct QuadTile {
  const uint32_t *ptrs[MQ_CHUNK];
  uint32_t shift[MQ_CHUNK];
  uint32_t tile[MQ_CHUNK * 64];
};
__device__ __forceinline__ void layer_hash_quad_lds(const MerkleLayer &L, uint32_t i0, QuadTile &S, uint32_t &lo,
                                                    uint32_t &hi) {
  const uint32_t *prev = L.prev;
  const ColRef *cols = L.cols;
  const uint32_t n_cols = L.n_cols, n = 1u << L.log_size;
  const uint32_t tid = threadIdx.x, node = tid >> 2, j = tid & 3, i = i0 + node;
  const bool active = i < n;  // every lane stays for the barriers
  lo = b2_iv_lo(j);
  hi = b2_iv_hi(j);
  uint32_t m[16];
  uint32_t t = 0;
  if (prev) {
    if (active) {
      load_block64(m, prev + 16 * (size_t)i);
      b2_compress_quad(lo, hi, m, 64, n_cols == 0);
    }
    t = 64;
  } else if (n_cols == 0) {
#pragma unroll
    for (int k = 0; k < 16; k++) m[k] = 0;
    if (active) b2_compress_quad(lo, hi, m, 0, true);
  }
  const uint32_t w = tid & 63, row = i0 + w;
  for (uint32_t cb = 0; cb < n_cols; cb += MQ_CHUNK) {
    const uint32_t cnt = min(MQ_CHUNK, n_cols - cb), words = cnt * 64;
    __syncthreads();  // the previous chunk's words are consumed
    for (uint32_t c = tid; c < cnt; c += 256) {
      const ColRef cr = cols[cb + c];
      S.ptrs[c] = cr.p;
      S.shift[c] = cr.shift;
    }
    __syncthreads();
    auto stage = [&](auto lifted) {
      for (uint32_t e0 = 0; e0 < words; e0 += 256 * 32) {
        uint32_t v[32];
#pragma unroll
        for (uint32_t k = 0; k < 32; k++) {
          const uint32_t e = e0 + tid + 256 * k;  // column e >> 6 is uniform over the wave
          v[k] = 0;
          if (e < words && row < n)
            v[k] = ld_col_word(S.ptrs[e >> 6],
                               lifted ? ((row >> (S.shift[e >> 6] + 1)) << 1) + (row & 1) : row);
        }
#pragma unroll
        for (uint32_t k = 0; k < 32; k++) {
          const uint32_t e = e0 + tid + 256 * k;
          if (e < words) S.tile[e] = v[k];
        }
      }
    };
    if (L.lifted)
      stage(std::true_type{});
    else
      stage(std::false_type{});
    __syncthreads();
    for (uint32_t b = 0; b < cnt; b += 16) {
      const uint32_t bc = min(16u, cnt - b);
#pragma unroll
      for (uint32_t k = 0; k < 16; k++) m[k] = k < bc ? S.tile[(b + k) * 64 + node] : 0u;
      t += 4 * bc;
      if (active) b2_compress_quad(lo, hi, m, t, cb + b + 16 >= n_cols);
    }
  }
  if (L.m31) {
    lo = b2_reduce_word(lo);
    hi = b2_reduce_word(hi);
  }
}

// One layer: its nodes alone.
template <bool AHEAD, bool TABLE>
__device__ __forceinline__ void merkle_layer(const MerkleLayer &L, const ColRef *cols, uint32_t wg) {
  const uint32_t i = wg * 256 + threadIdx.x;
  if (i >= 1u << L.log_size) return;
  store_hash(L.out + 8 * (size_t)i, layer_hash<AHEAD, TABLE>(L, cols, i), 0);
}
__device__ __forceinline__ void store_quad(uint32_t *out, uint32_t i, uint32_t lo, uint32_t hi) {
  g_u32 *o = as_global(out + 8 * (size_t)i);
  o[threadIdx.x & 3] = lo;
  o[4 + (threadIdx.x & 3)] = hi;
}
__device__ __forceinline__ void merkle_layer_quad_lds(const MerkleLayer &L, uint32_t wg) {
  __shared__ QuadTile S;
  const uint32_t i = wg * 64 + (threadIdx.x >> 2);
  uint32_t lo, hi;
  layer_hash_quad_lds(L, wg * 64, S, lo, hi);
  if (i < 1u << L.log_size) store_quad(L.out, i, lo, hi);
}

// A layer of at most 2^14 nodes and the run of node layers below it, down to
// stop_log, in one launch (out lies in the packed tree): a workgroup hashes 64
// nodes of the layer, a quad each (LDS: with the columns staged through it), and
// goes on as merkle_nodes does.  The layer's digests are not read back, and the
// second launch and its first loads go: a tree over 16 columns of 2^11 takes
// 17.4 us, in two launches 5.6 + 14.6.
template <bool LDS>
__device__ __forceinline__ void merkle_tree(const MerkleTree &T, const ColRef *cols, uint32_t wg) {
  // the column words are consumed when the digests come
  constexpr size_t kBytes = LDS && sizeof(QuadTile) > sizeof(TreeLds) ? sizeof(QuadTile) : sizeof(TreeLds);
  __shared__ __align__(16) uint8_t mem[kBytes];
  TreeLds &S = *reinterpret_cast<TreeLds *>(mem);
  const MerkleLayer &L = T.layer;
  const uint32_t n = 1u << L.log_size, first = wg * 64, q = threadIdx.x >> 2, j = threadIdx.x & 3, i = first + q;
  uint32_t lo, hi;
  if constexpr (LDS) {
    layer_hash_quad_lds(L, first, *reinterpret_cast<QuadTile *>(mem), lo, hi);
    __syncthreads();
  } else if (i < n) {
    layer_hash_quad(L, cols, i, lo, hi);
  }
  if (i < n) {
    store_quad(L.out, i, lo, hi);
    tree_row(S, 0, q)[j] = lo;
    tree_row(S, 0, q)[4 + j] = hi;
  }
  const uint32_t cnt = min(64u, n), lv = min(31 - __clz(cnt), L.log_size - T.stop_log), l = L.log_size - lv;
  uint32_t *packed = L.out - tree_layer_off(L.log_size);
  const uint32_t buf = tree_levels(S, 0, cnt, first, L.log_size, lv, packed, L.m31, l > T.stop_log);
  tree_finish(S, buf, wg, l, T.stop_log, packed, L.m31, T.counters);
}

// Node layers out_log .. stop_log below `prev` (of log size out_log + 1), each
// written at its place in the packed layout.  A workgroup takes NODES nodes of
// layer out_log: 1,024 (four per lane, with the two levels above them from
// registers) where there are enough of them, which leaves little of a subtree to
// its narrow levels; 64 (a quad each) in small trees, where latency counts; 256
// between.
template <uint32_t NODES>
__device__ __forceinline__ void merkle_nodes(const MerkleNodes &L, uint32_t wg) {
  __shared__ __align__(16) TreeLds S;
  uint32_t *packed = L.packed;
  const uint32_t out_log = L.out_log, stop_log = L.stop_log, m31 = L.m31;
  const uint32_t *prev = packed + tree_layer_off(out_log + 1);
  const uint32_t n = 1u << out_log, first = wg * NODES, tid = threadIdx.x;
  uint32_t *out = packed + tree_layer_off(out_log);
  uint32_t lg = out_log, cnt = min(NODES, n), row0 = first;  // the level held in S
  if constexpr (NODES == 64) {
    const uint32_t q = tid >> 2, j = tid & 3, i = first + q;
    if (i < n) {
      uint32_t m[16];
      load_block64(m, prev + 16 * (size_t)i);
      uint32_t lo = b2_iv_lo(j), hi = b2_iv_hi(j);
      b2_compress_quad(lo, hi, m, 64, true);
      if (m31) {
        lo = b2_reduce_word(lo);
        hi = b2_reduce_word(hi);
      }
      as_global(out + 8 * (size_t)i)[j] = lo;
      as_global(out + 8 * (size_t)i)[4 + j] = hi;
      tree_row(S, 0, q)[j] = lo;
      tree_row(S, 0, q)[4 + j] = hi;
    }
  } else if constexpr (NODES == 256) {
    const uint32_t i = first + tid;
    if (i < n) tree_keep(S, 0, tid, hash_node(prev, i, out, m31));
  } else {
    // four nodes per lane and, from registers, the two levels above them
    const uint32_t i = first + 4 * tid;
    b2_state keep;
#pragma unroll 1
    for (uint32_t p = 0; p < 2; p++) {
      const b2_state a = hash_node(prev, i + 2 * p, out, m31), b = hash_node(prev, i + 2 * p + 1, out, m31);
      const b2_state c = hash_pair(a, b, m31);
      store_hash(packed + tree_layer_off(out_log - 1) + 8 * (size_t)(i / 2 + p), c, 0);
      if (p == 0) {
        keep = c;
      } else {
        const b2_state t = hash_pair(keep, c, m31);
        store_hash(packed + tree_layer_off(out_log - 2) + 8 * (size_t)(i / 4), t, 0);
        tree_keep(S, 0, tid, t);
      }
    }
    lg -= 2;
    cnt >>= 2;
    row0 >>= 2;
  }
  const uint32_t lv = min(31 - __clz(cnt), lg - stop_log), l = lg - lv;
  const uint32_t buf = tree_levels(S, 0, cnt, row0, lg, lv, packed, m31, l > stop_log);
  tree_finish(S, buf, wg, l, stop_log, packed, m31, L.counters);
}

// The launches: one layer or run of node layers by value, or several from a
// table, each owning the workgroups from its wg_start on (0, then increasing).
template <typename T>
__device__ __forceinline__ const T &step_of(const T *t, uint32_t n) {
  uint32_t g = 0, hi = n;
  while (hi - g > 1) {
    const uint32_t mid = (g + hi) / 2;
    if (t[mid].wg_start <= blockIdx.x) g = mid; else hi = mid;
  }
  return t[g];
}
template <bool AHEAD>
__global__ void __launch_bounds__(256) merkle_layer_kernel(MerkleLayer L) {
  merkle_layer<AHEAD, true>(L, L.cols, blockIdx.x);
}
template <bool AHEAD>
__global__ void __launch_bounds__(256) merkle_layer_multi_kernel(const MerkleLayer *t, uint32_t n) {
  const MerkleLayer L = step_of(t, n);
  merkle_layer<AHEAD, true>(L, L.cols, blockIdx.x - L.wg_start);
}
__global__ void __launch_bounds__(256) merkle_layer_quad_lds_kernel(MerkleLayer L) {
  merkle_layer_quad_lds(L, blockIdx.x);
}
__global__ void __launch_bounds__(256) merkle_layer_quad_lds_multi_kernel(const MerkleLayer *t, uint32_t n) {
  const MerkleLayer L = step_of(t, n);
  merkle_layer_quad_lds(L, blockIdx.x - L.wg_start);
}
template <bool LDS>
__global__ void __launch_bounds__(kTreeThreads) merkle_tree_kernel(MerkleTree T) {
  merkle_tree<LDS>(T, T.layer.cols, blockIdx.x);
}
template <bool LDS>
__global__ void __launch_bounds__(kTreeThreads) merkle_tree_multi_kernel(const MerkleTree *t, uint32_t n) {
  const MerkleTree T = step_of(t, n);
  merkle_tree<LDS>(T, T.layer.cols, blockIdx.x - T.wg_start);
}
// The columns among the arguments: their upload costs a small commit as much as
// its leaves (2.3 us and a launch's gap; leaves of 16 columns of 2^17 take 9.7).
struct InlineCols {
  ColRef c[kInlineCols];
};
template <bool AHEAD>
__global__ void __launch_bounds__(256) merkle_layer_inline_kernel(MerkleLayer L, InlineCols cols) {
  merkle_layer<AHEAD, false>(L, cols.c, blockIdx.x);
}
__global__ void __launch_bounds__(kTreeThreads) merkle_tree_inline_kernel(MerkleTree T, InlineCols cols) {
  merkle_tree<false>(T, cols.c, blockIdx.x);
}
template <uint32_t NODES>
__global__ void __launch_bounds__(kTreeThreads) merkle_nodes_kernel(MerkleNodes L) {
  merkle_nodes<NODES>(L, blockIdx.x);
}
template <uint32_t NODES>
__global__ void __launch_bounds__(kTreeThreads) merkle_nodes_multi_kernel(const MerkleNodes *t, uint32_t n) {
  const MerkleNodes L = step_of(t, n);
  merkle_nodes<NODES>(L, blockIdx.x - L.wg_start);
}

static inline size_t layer_off(uint32_t l) { return tree_layer_off(l); }

// Up to 2^14 nodes with more than one block per node, the layer is
// latency-bound even at four lanes per node: a quad per node, with the columns
// staged through LDS.  Below 2^16 nodes, a lane per node with the loads one block
// ahead.
MerkleStep merkle_layer_step(const uint32_t *prev, const ColRef *d_cols, uint32_t n_cols, uint32_t log_size,
                             uint32_t *out, int mode, bool lifted) {
  MerkleStep s{};
  s.layer = {prev, d_cols, out, n_cols, log_size, (uint32_t)(mode == STWO_HIP_HASH_BLAKE2S_M31), (uint32_t)lifted, 0};
  const uint32_t n = 1u << log_size;
  const bool quad = log_size <= 14 && n_cols > 16;
  s.kind = quad ? kMerkleQuadLds : log_size < 16 && n_cols > 16 ? kMerkleAhead : kMerkleLayer;
  s.wgs = quad ? (n + 63) / 64 : (n + 255) / 256;
  return s;
}

// Node layers top_log-1 .. stop_log (< top_log) of a packed tree whose layer
// top_log is filled.  counters: n_counters zeros, left zero, used by no launch
// that may overlap this one.  A run that needs more ends at its workgroups' own
// level (then no workgroup meets another) and leaves the rest to a further
// launch, which costs 4 us where the levels before it take milliseconds.
MerkleStep merkle_nodes_step(uint32_t *layers, uint32_t top_log, uint32_t stop_log, int mode, uint32_t *counters,
                             uint32_t n_counters) {
  MerkleStep s{};
  const uint32_t out_log = top_log - 1;
  // (four nodes per lane take the two levels above along)
  const uint32_t per = std::min<uint32_t>(tree_leaves_log(out_log), out_log >= stop_log + 2 ? 10 : 8);
  const uint32_t own = out_log > per ? out_log - per : 0;  // the workgroups' level
  if (own > stop_log && tree_counters_needed(own, stop_log) > n_counters) stop_log = own;
  s.nodes = {layers, counters, out_log, stop_log, (uint32_t)(mode == STWO_HIP_HASH_BLAKE2S_M31), 0};
  s.kind = per == 6 ? kMerkleNodes64 : per == 8 ? kMerkleNodes256 : kMerkleNodes1024;
  s.wgs = 1u << own;
  return s;
}

// Up to 2^14 nodes, where the node layers alone also take a quad for each of 64.
// With a lane for each of 256 above that there is nothing to gain: 2^17 leaves of
// 16 columns 37.6 us, in two launches 9.2 + 27.5.
bool merkle_tree_step(MerkleStep &s, uint32_t stop_log, uint32_t *counters, uint32_t n_counters) {
  const uint32_t lg = s.layer.log_size, own = lg > 6 ? lg - 6 : 0;
  if (lg > 14 || stop_log >= lg || tree_counters_needed(own, stop_log) > n_counters) return false;
  s.tree = {s.layer, counters, stop_log, 0};
  s.kind = s.layer.n_cols > 16 ? kMerkleTreeLds : kMerkleTree;
  s.wgs = 1u << own;
  return true;
}

static const char *step_name(uint32_t kind, bool lifted) {
  return kind >= kMerkleTree ? "merkle_tree" : kind >= kMerkleNodes64 ? "merkle_nodes" : lifted ? "merkle_lifted_leaves" : "merkle_commit_on_layer";
}

int launch_merkle(stwo_hip_ctx *ctx, const MerkleStep &s) {
  const char *name = step_name(s.kind, s.layer.lifted);
  const dim3 grid(s.wgs), block(256);
  switch (s.kind) {
    case kMerkleLayer: return launch(ctx, name, merkle_layer_kernel<false>, grid, block, 0, s.layer);
    case kMerkleAhead: return launch(ctx, name, merkle_layer_kernel<true>, grid, block, 0, s.layer);
    case kMerkleQuadLds: return launch(ctx, name, merkle_layer_quad_lds_kernel, grid, block, 0, s.layer);
    case kMerkleNodes64: return launch(ctx, name, merkle_nodes_kernel<64>, grid, block, 0, s.nodes);
    case kMerkleNodes256: return launch(ctx, name, merkle_nodes_kernel<256>, grid, block, 0, s.nodes);
    case kMerkleNodes1024: return launch(ctx, name, merkle_nodes_kernel<1024>, grid, block, 0, s.nodes);
    case kMerkleTree: return launch(ctx, name, merkle_tree_kernel<false>, grid, block, 0, s.tree);
    default: return launch(ctx, name, merkle_tree_kernel<true>, grid, block, 0, s.tree);
  }
}

int launch_merkle_multi(stwo_hip_ctx *ctx, uint32_t kind, bool lifted, const void *d_steps, uint32_t n, uint32_t wgs) {
  const char *name = step_name(kind, lifted);
  const dim3 grid(wgs), block(256);
  const MerkleLayer *l = (const MerkleLayer *)d_steps;
  const MerkleNodes *t = (const MerkleNodes *)d_steps;
  const MerkleTree *r = (const MerkleTree *)d_steps;
  switch (kind) {
    case kMerkleLayer: return launch(ctx, name, merkle_layer_multi_kernel<false>, grid, block, 0, l, n);
    case kMerkleAhead: return launch(ctx, name, merkle_layer_multi_kernel<true>, grid, block, 0, l, n);
    case kMerkleQuadLds: return launch(ctx, name, merkle_layer_quad_lds_multi_kernel, grid, block, 0, l, n);
    case kMerkleNodes64: return launch(ctx, name, merkle_nodes_multi_kernel<64>, grid, block, 0, t, n);
    case kMerkleNodes256: return launch(ctx, name, merkle_nodes_multi_kernel<256>, grid, block, 0, t, n);
    case kMerkleNodes1024: return launch(ctx, name, merkle_nodes_multi_kernel<1024>, grid, block, 0, t, n);
    case kMerkleTree: return launch(ctx, name, merkle_tree_multi_kernel<false>, grid, block, 0, r, n);
    default: return launch(ctx, name, merkle_tree_multi_kernel<true>, grid, block, 0, r, n);
  }
}

static int check_mode(stwo_hip_ctx *ctx, int mode) {
  STWO_HIP_CHECK_ARG(ctx, mode == STWO_HIP_HASH_BLAKE2S || mode == STWO_HIP_HASH_BLAKE2S_M31,
                     "merkle: unknown hash mode %d", mode);
  return STWO_HIP_OK;
}

// A layer with columns, and the node layers below it down to stop_log, where they
// share a launch; *done: whether they did.
static int launch_layer(stwo_hip_ctx *ctx, const uint32_t *prev, const std::vector<ColRef> &cols, uint32_t log_size,
                        uint32_t *out, int mode, bool lifted, uint32_t stop_log, bool *done) {
  int rc = check_mode(ctx, mode);
  if (rc) return rc;
  MerkleStep s = merkle_layer_step(prev, nullptr, (uint32_t)cols.size(), log_size, out, mode, lifted);
  *done = merkle_tree_step(s, stop_log, ctx->d_counters, kTreeCounters);
  const bool in_args = s.kind == kMerkleTree || s.kind == kMerkleLayer || s.kind == kMerkleAhead;
  if (in_args && cols.size() <= kInlineCols) {
    InlineCols in{};
    std::copy(cols.begin(), cols.end(), in.c);
    const dim3 grid(s.wgs), block(256);
    const char *name = step_name(s.kind, lifted);
    if (s.kind == kMerkleTree) return launch(ctx, name, merkle_tree_inline_kernel, grid, block, 0, s.tree, in);
    return launch(ctx, name, s.kind == kMerkleAhead ? merkle_layer_inline_kernel<true> : merkle_layer_inline_kernel<false>,
                  grid, block, 0, s.layer, in);
  }
  if (!cols.empty()) {
    void *dtab = nullptr;
    rc = upload_table(ctx, cols.data(), cols.size() * sizeof(ColRef), &dtab);
    if (rc) return rc;
    s.layer.cols = s.tree.layer.cols = (const ColRef *)dtab;
  }
  return launch_merkle(ctx, s);
}
static int launch_layer(stwo_hip_ctx *ctx, const uint32_t *prev, const std::vector<ColRef> &cols, uint32_t log_size,
                        uint32_t *out, int mode, bool lifted) {
  bool done;
  return launch_layer(ctx, prev, cols, log_size, out, mode, lifted, log_size, &done);
}

static int hash_node_layers(stwo_hip_ctx *ctx, uint32_t *layers, uint32_t top_log, uint32_t stop_log, int mode) {
  int rc = check_mode(ctx, mode);
  while (!rc && top_log > stop_log) {
    const MerkleStep s = merkle_nodes_step(layers, top_log, stop_log, mode, ctx->d_counters, kTreeCounters);
    rc = launch_merkle(ctx, s);
    top_log = s.nodes.stop_log;
  }
  return rc;
}

}  // namespace stwo_hip

using namespace stwo_hip;

extern "C" {

int stwo_hip_merkle_commit_on_layer(stwo_hip_ctx *ctx, uint32_t log_size, const uint32_t *prev,
                                    const uint32_t *const *cols, size_t n_cols, uint32_t *out, int hash_mode) {
  if (!ctx) return STWO_HIP_EINVAL;
  STWO_HIP_CHECK_ARG(ctx, out != nullptr && log_size <= 30, "commit_on_layer: bad output");
  STWO_HIP_CHECK_ARG(ctx, n_cols == 0 || cols != nullptr, "commit_on_layer: NULL column array");
  std::vector<ColRef> refs(n_cols);
  for (size_t c = 0; c < n_cols; c++) {
    STWO_HIP_CHECK_ARG(ctx, cols[c] != nullptr, "commit_on_layer: NULL column %zu", c);
    refs[c] = {cols[c], 0, 0};
  }
  return launch_layer(ctx, prev, refs, log_size, out, hash_mode, false);
}

int stwo_hip_merkle_commit(stwo_hip_ctx *ctx, const uint32_t *const *cols, const uint32_t *log_sizes, size_t n_cols,
                           uint32_t *layers, int hash_mode) {
  if (!ctx) return STWO_HIP_EINVAL;
  STWO_HIP_CHECK_ARG(ctx, layers != nullptr, "merkle_commit: NULL output");
  if (n_cols == 0) return launch_layer(ctx, nullptr, {}, 0, layers, hash_mode, false);
  STWO_HIP_CHECK_ARG(ctx, cols && log_sizes, "merkle_commit: NULL arrays");
  uint32_t max_log = 0;
  for (size_t c = 0; c < n_cols; c++) {
    STWO_HIP_CHECK_ARG(ctx, cols[c] && log_sizes[c] <= 30, "merkle_commit: bad column %zu", c);
    max_log = std::max(max_log, log_sizes[c]);
  }
  for (int l = (int)max_log; l >= 0;) {
    std::vector<ColRef> refs;
    for (size_t c = 0; c < n_cols; c++)  // input order == stable order among equal lengths
      if (log_sizes[c] == (uint32_t)l) refs.push_back({cols[c], 0, 0});
    const uint32_t *prev = (l == (int)max_log) ? nullptr : layers + layer_off(l + 1);
    // below it, a run of pure node layers down to the next injected layer (or the root)
    int next = -1;
    for (size_t c = 0; c < n_cols; c++)
      if ((int)log_sizes[c] < l) next = std::max(next, (int)log_sizes[c]);
    const uint32_t stop = (uint32_t)(next + 1);
    bool done = false;
    int rc = launch_layer(ctx, prev, refs, (uint32_t)l, layers + layer_off((uint32_t)l), hash_mode, false, stop, &done);
    if (!rc && !done) rc = hash_node_layers(ctx, layers, (uint32_t)l, stop, hash_mode);
    if (rc) return rc;
    l = next;
  }
  return STWO_HIP_OK;
}

// The leaves of a lifted tree, and its node layers where they share the launch.
static int lifted_leaves(stwo_hip_ctx *ctx, const uint32_t *const *cols, const uint32_t *log_sizes, size_t n_cols,
                         uint32_t lifting_log_size, uint32_t *out, int hash_mode, uint32_t stop_log, bool *done) {
  STWO_HIP_CHECK_ARG(ctx, cols && log_sizes && lifting_log_size <= 30, "lifted_build_leaves: bad arguments");
  std::vector<size_t> order(n_cols);
  for (size_t c = 0; c < n_cols; c++) {
    order[c] = c;
    STWO_HIP_CHECK_ARG(ctx, cols[c] != nullptr, "lifted_build_leaves: NULL column %zu", c);
    STWO_HIP_CHECK_ARG(ctx, log_sizes[c] >= 1, "A column must be of length >= 2.");
    STWO_HIP_CHECK_ARG(ctx, log_sizes[c] <= lifting_log_size, "column %zu longer than the lifting size", c);
  }
  std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) { return log_sizes[a] < log_sizes[b]; });
  std::vector<ColRef> refs;
  for (size_t c : order) refs.push_back({cols[c], lifting_log_size - log_sizes[c], 0});
  return launch_layer(ctx, nullptr, refs, lifting_log_size, out, hash_mode, true, stop_log, done);
}

int stwo_hip_merkle_lifted_build_leaves(stwo_hip_ctx *ctx, const uint32_t *const *cols, const uint32_t *log_sizes,
                                        size_t n_cols, uint32_t lifting_log_size, uint32_t *out, int hash_mode) {
  if (!ctx) return STWO_HIP_EINVAL;
  STWO_HIP_CHECK_ARG(ctx, out != nullptr, "lifted_build_leaves: NULL output");
  if (n_cols == 0) return launch_layer(ctx, nullptr, {}, 0, out, hash_mode, true);
  bool done;
  return lifted_leaves(ctx, cols, log_sizes, n_cols, lifting_log_size, out, hash_mode, lifting_log_size, &done);
}

int stwo_hip_merkle_lifted_build_next_layer(stwo_hip_ctx *ctx, const uint32_t *prev, uint32_t out_log_size,
                                            uint32_t *out, int hash_mode) {
  if (!ctx) return STWO_HIP_EINVAL;
  STWO_HIP_CHECK_ARG(ctx, prev && out && out_log_size < 30, "lifted_build_next_layer: bad arguments");
  return launch_layer(ctx, prev, {}, out_log_size, out, hash_mode, false);
}

int stwo_hip_merkle_lifted_commit(stwo_hip_ctx *ctx, const uint32_t *const *cols, const uint32_t *log_sizes,
                                  size_t n_cols, uint32_t lifting_log_size, uint32_t *layers, int hash_mode) {
  if (!ctx) return STWO_HIP_EINVAL;
  STWO_HIP_CHECK_ARG(ctx, layers != nullptr, "lifted_commit: NULL output");
  if (n_cols == 0) return stwo_hip_merkle_lifted_build_leaves(ctx, cols, log_sizes, 0, 0, layers, hash_mode);
  STWO_HIP_CHECK_ARG(ctx, lifting_log_size <= 30, "lifted_build_leaves: bad arguments");
  bool done = false;
  int rc = lifted_leaves(ctx, cols, log_sizes, n_cols, lifting_log_size, layers + layer_off(lifting_log_size),
                         hash_mode, 0, &done);
  if (rc || done) return rc;
  return hash_node_layers(ctx, layers, lifting_log_size, 0, hash_mode);
}

int stwo_hip_debug_tree_plan(int what, uint32_t top_log, uint32_t stop_log, uint32_t n, uint32_t plan_log,
                             uint32_t *out, uint32_t max_steps, uint32_t *n_steps) {
  if (!out || !n_steps || what < 0 || what > 2 || top_log > 30 || stop_log > top_log || plan_log > 30 ||
      (what == 2 && (n < 1 || n > 16 || stop_log)))
    return STWO_HIP_EINVAL;
  const uint32_t there = plan_log ? tree_counters(plan_log) : kTreeCounters;
  uint32_t k = 0;
  auto put = [&](uint32_t first, uint32_t own, uint32_t stop, uint32_t wgs) {
    own = std::max(own, stop);  // a workgroup ends at the run's end
    if (k < max_steps) {
      uint32_t *o = out + 6 * k;
      o[0] = first;
      o[1] = own;
      o[2] = stop;
      o[3] = wgs;
      o[4] = (uint32_t)tree_counters_needed(own, stop);
      o[5] = there;
    }
    k++;
  };
  auto log2 = [](uint32_t v) { return 31u - (uint32_t)__builtin_clz(v); };
  uint32_t top = top_log;
  if (what == 2) {
    const uint32_t per = fri_leaves_log(top, n), own = top > per ? top - per : 0;
    put(top, own, 0, 1u << own);
    top = 0;
  } else if (what == 1) {
    MerkleStep s = merkle_layer_step(nullptr, nullptr, n, top, nullptr, STWO_HIP_HASH_BLAKE2S, false);
    if (merkle_tree_step(s, stop_log, nullptr, there)) {
      put(top, log2(s.wgs), s.tree.stop_log, s.wgs);
      top = s.tree.stop_log;
    } else {
      put(top, top, top, s.wgs);
    }
  }
  while (top > stop_log) {
    const MerkleStep s = merkle_nodes_step(nullptr, top, stop_log, STWO_HIP_HASH_BLAKE2S, nullptr, there);
    put(s.nodes.out_log, log2(s.wgs), s.nodes.stop_log, s.wgs);
    top = s.nodes.stop_log;
  }
  *n_steps = k;
  return k <= max_steps ? STWO_HIP_OK : STWO_HIP_EINVAL;
}

}  // extern "C"
