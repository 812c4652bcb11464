// Device pieces shared by the Merkle node kernels and the fused FRI layer
// kernel: digest stores, the subtree over a workgroup's digests and the levels
// above it.
#pragma once
#include <stdint.h>

#include "blake2s.hpp"
#include "common.hpp"
#include "internal.hpp"

namespace stwo_hip {

__device__ __forceinline__ void store_hash(uint32_t *dst, const b2_state &s, uint32_t m31) {
  uint4 a, b;
  if (m31) {
    a = make_uint4(b2_reduce_word(s.h[0]), b2_reduce_word(s.h[1]), b2_reduce_word(s.h[2]), b2_reduce_word(s.h[3]));
    b = make_uint4(b2_reduce_word(s.h[4]), b2_reduce_word(s.h[5]), b2_reduce_word(s.h[6]), b2_reduce_word(s.h[7]));
  } else {
    a = make_uint4(s.h[0], s.h[1], s.h[2], s.h[3]);
    b = make_uint4(s.h[4], s.h[5], s.h[6], s.h[7]);
  }
  reinterpret_cast<uint4 *>(dst)[0] = a;
  reinterpret_cast<uint4 *>(dst)[1] = b;
}

// ---- a tree in one launch -----------------------------------------------------
//
// A workgroup hashes the subtree over its first digests down to one (or to
// level `stop`), then the workgroups meet: 2^s neighbours count themselves on
// a counter, and the last to arrive hashes their 2^s digests on, s levels at a
// time, until level `stop`.  No workgroup waits for another.  The digests that
// change hands are stored and loaded at agent scope (each XCD has its own L2),
// complete before the count; the last arriver sets the counter back to zero.
//
// A meeting costs about 1.5 us (stores out, count, loads); a further launch for
// the levels above costs 3 to 4.5 us before its first hash.  A level takes 0.8 us,
// the 380 instructions of one compression one after the other plus the way
// through LDS.

constexpr uint32_t kTreeThreads = 256;

__device__ __forceinline__ void st_agent(uint32_t *p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t ld_agent(const uint32_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Digests of a level held by a workgroup of kTreeThreads lanes: pairs of
// siblings, 16 consecutive words (a parent's message, four 16-byte reads) every
// 20 (quads reading different pairs meet different banks), in two buffers that
// the levels alternate between, so a level takes one barrier.
constexpr uint32_t kTreeRows = 256;
struct TreeLds {
  uint32_t d[2][kTreeRows / 2][20];
  uint32_t last;
};
__device__ __forceinline__ uint32_t *tree_row(TreeLds &S, uint32_t buf, uint32_t row) {
  return &S.d[buf][row >> 1][(row & 1) << 3];
}
__device__ __forceinline__ void tree_pair(const TreeLds &S, uint32_t buf, uint32_t i, uint32_t m[16]) {
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const uint4 v = *reinterpret_cast<const uint4 *>(&S.d[buf][i][4 * k]);
    m[4 * k] = v.x;
    m[4 * k + 1] = v.y;
    m[4 * k + 2] = v.z;
    m[4 * k + 3] = v.w;
  }
}
__device__ __forceinline__ void tree_keep(TreeLds &S, uint32_t buf, uint32_t row, const b2_state &s) {
  uint4 *o = reinterpret_cast<uint4 *>(tree_row(S, buf, row));
  o[0] = make_uint4(s.h[0], s.h[1], s.h[2], s.h[3]);
  o[1] = make_uint4(s.h[4], s.h[5], s.h[6], s.h[7]);
}

// Hashes n_levels levels over the cnt digests (a power of two, at most
// kTreeRows) in buffer `buf`, nodes first .. first + cnt - 1 of level lg:
// H(left || right) each, written to the packed tree and kept in the buffers.
// A quad per hash (their latency is the critical path), two after each other
// on a level of 128.  `handoff`: the last level is read by another workgroup.
// Starts and ends with a barrier; returns the buffer of the last level.
//
// Levels of 16 hashes and fewer are one wave's: in place, since a wave's LDS
// accesses are in order, and with every lane hashing (those past the level a
// stale row), so the loop has fixed addresses and no branch but its own. A
// level is 380 instructions of one compression, 1,500 cycles, and about 300 for
// the way through LDS; with the loop of the wide levels it was 2,200 in all
// (a tree over 16 columns of 2^11 17.4 -> 15.0 us).
__device__ __forceinline__ uint32_t tree_levels(TreeLds &S, uint32_t buf, uint32_t cnt, size_t first, uint32_t lg,
                                                uint32_t n_levels, uint32_t *packed, uint32_t m31, bool handoff) {
  const uint32_t q = threadIdx.x >> 2, j = threadIdx.x & 3;
  const b2_quad_iv iv = b2_quad_init();
  const uint32_t d0 = b2_quad_d(iv, 64, true);
  __syncthreads();
  uint32_t k = 0;
  for (; k < n_levels && cnt > 32; k++) {
    cnt >>= 1;
    first >>= 1;
    lg--;
    g_u32 *out = as_global(packed + tree_layer_off(lg) + 8 * first);
    const bool agent = handoff && k + 1 == n_levels;
    for (uint32_t i = q; i < cnt; i += kTreeThreads / 4) {
      uint32_t m[16];
      tree_pair(S, buf, i, m);
      uint32_t lo = iv.lo, hi = iv.hi;
      b2_compress_quad(iv, lo, hi, m, d0);
      if (m31) {
        lo = b2_reduce_word(lo);
        hi = b2_reduce_word(hi);
      }
      uint32_t *keep = tree_row(S, buf ^ 1, i);
      keep[j] = lo;
      keep[4 + j] = hi;
      if (agent) {
        st_agent((uint32_t *)(out + 8 * i + j), lo);
        st_agent((uint32_t *)(out + 8 * i + 4 + j), hi);
      } else {
        out[8 * i + j] = lo;
        out[8 * i + 4 + j] = hi;
      }
    }
    buf ^= 1;
    __syncthreads();
  }
  if (threadIdx.x < 64) {
    uint32_t *keep = tree_row(S, buf, q) + j;
    for (; k < n_levels; k++) {
      cnt >>= 1;
      first >>= 1;
      lg--;
      g_u32 *out = as_global(packed + tree_layer_off(lg) + 8 * first);
      uint32_t m[16];
      tree_pair(S, buf, q, m);
      uint32_t lo = iv.lo, hi = iv.hi;
      b2_compress_quad(iv, lo, hi, m, d0);
      if (m31) {
        lo = b2_reduce_word(lo);
        hi = b2_reduce_word(hi);
      }
      __builtin_amdgcn_wave_barrier();
      keep[0] = lo;
      keep[4] = hi;
      __builtin_amdgcn_wave_barrier();
      if (q < cnt) {
        if (handoff && k + 1 == n_levels) {
          st_agent((uint32_t *)(out + 8 * q + j), lo);
          st_agent((uint32_t *)(out + 8 * q + 4 + j), hi);
        } else {
          out[8 * q + j] = lo;
          out[8 * q + 4 + j] = hi;
        }
      }
    }
  }
  __syncthreads();
  return buf;
}

// The rest of the tree above the workgroup's subtree, whose one digest is node
// b of level l (stored by tree_levels with handoff, in buffer buf), down to
// level `stop`, in stages of tree_stage levels.  counters: tree_counters_needed(l, stop)
// zeros, left zero.
// Returns the buffer whose row 0 is then this workgroup's last digest (the root
// when stop = 0), or -1 in the workgroups that another one goes on for.
__device__ __forceinline__ int tree_finish(TreeLds &S, uint32_t buf, uint32_t b, uint32_t l, uint32_t stop,
                                           uint32_t *packed, uint32_t m31, uint32_t *counters) {
  const uint32_t tid = threadIdx.x;
  while (l > stop) {
    const uint32_t s = tree_stage(l, stop), group = b >> s;
    // every lane's handed-over words have left before the count
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
      const uint32_t old =
          __hip_atomic_fetch_add(counters + group, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const uint32_t last = old + 1 == (1u << s);
      if (last) st_agent(counters + group, 0);
      S.last = last;
    }
    __syncthreads();
    if (!S.last) return -1;
    counters += (size_t)1 << (l - s);
    const uint32_t *in = packed + tree_layer_off(l) + ((size_t)8 << s) * group;
    for (uint32_t e = tid; e < (8u << s); e += kTreeThreads) tree_row(S, 0, e >> 3)[e & 7] = ld_agent(in + e);
    l -= s;
    buf = tree_levels(S, 0, 1u << s, (size_t)group << s, l + s, s, packed, m31, l > stop);
    b = group;
  }
  return (int)buf;
}

}  // namespace stwo_hip
