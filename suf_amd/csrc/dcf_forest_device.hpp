// Broadcast DCF keys over a tile of points: the levels that the tile's points
// share are walked once per workgroup instead of once per point.
//
// A broadcast key's walk state after d levels depends only on the top d bits
// of the point.  The points of a gate are masked fixed-point values x + r,
// one r for the batch, so a tile spans a short interval of the 64-bit ring
// and its points agree on their first L bits (x of 30 bits: L is about 33).
// A workgroup finds L, walks the common prefix on 8 lanes (quad_walk),
// expands D more levels breadth-first into LDS (8 lanes per child) and starts
// every point at its node of depth L + D.  The points are public, and any
// set of them gives the same shares: with no common prefix L is 0.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "dcf_device.hpp"
#include "dcf_quad_device.hpp"

namespace sufhip {
namespace {

constexpr int kForestBlock = 1024;
// Nodes of all trees at the deepest expanded level: two passes of the
// workgroup's 128 groups of 8 lanes.
constexpr int kForestNodes = 256;

struct ForestLds {
  uint4 s[2][kForestNodes];
  uint64_t v[2][kForestNodes];
  uint32_t t[2][kForestNodes];
  uint32_t diff[2];
};

// One key of a forest; the trees of a forest share in_bits and the points.
struct ForestTree {
  const uint8_t* chunk;
  uint32_t party;
};

// Bits in which some of `count` points differs from the first, for the
// lanes' own share of them (xor_points), then over the workgroup
// (shared_levels: the leading levels of an in_bits walk that all points
// share).  lds.diff must be zero and the workgroup synchronised in between.
__device__ __forceinline__ uint64_t xor_points(const uint64_t* x, size_t count, uint64_t x0) {
  uint64_t d = 0;
  for (size_t i = threadIdx.x; i < count; i += kForestBlock) d |= x[i] ^ x0;
#pragma unroll
  for (int k = 32; k > 0; k >>= 1)
    d |= uint64_t(__shfl_xor(static_cast<unsigned long long>(d), k));
  return d;
}

__device__ __forceinline__ int shared_levels(ForestLds& lds, uint64_t d, int in_bits) {
  if ((threadIdx.x & 63u) == 0) {
    if (uint32_t(d)) atomicOr(&lds.diff[0], uint32_t(d));
    if (uint32_t(d >> 32)) atomicOr(&lds.diff[1], uint32_t(d >> 32));
  }
  __syncthreads();
  uint64_t m = uint64_t(lds.diff[0]) | uint64_t(lds.diff[1]) << 32;
  if (in_bits < 64) m &= (uint64_t(1) << in_bits) - 1;
  const int L = m == 0 ? in_bits : in_bits - (64 - __builtin_clzll(m));
  return __builtin_amdgcn_readfirstlane(L);
}

// Index of x's node at depth L + D, `left` levels above the leaves.
__device__ __forceinline__ int forest_node(uint64_t x, int left, int D) {
  return int(uint32_t(x >> (left & 63)) & ((1u << D) - 1u));
}

template <int kVal>
__device__ __forceinline__ void forest_put(ForestLds& lds, int buf, int node,
                                           const QuadState& st) {
  const uint32_t l = threadIdx.x & 7u;
  if (l < 4) reinterpret_cast<uint32_t*>(&lds.s[buf][node])[l] = st.s;
  if (l == 4) {
    lds.v[buf][node] = kVal == kQuadBit ? st.v.lo & 1u : st.v.lo;
    lds.t[buf][node] = st.t;
  }
}

__device__ __forceinline__ QuadState forest_get(const ForestLds& lds, int buf, int node) {
  return QuadState{reinterpret_cast<const uint32_t*>(&lds.s[buf][node])[threadIdx.x & 3u],
                   lds.t[buf][node], U128{lds.v[buf][node], 0}};
}

// The nodes at depth L + D of the kTrees trees (kTrees << D <= kForestNodes),
// node idx * kTrees + tree, in lds.s/v/t[D & 1].  x0: any of the points.
// Called by the whole workgroup; ends synchronised.
template <int kVal, int kTrees>
__device__ __forceinline__ void forest_build(const AesLds4& aes, const QuadKeys& K,
                                             const ForestTree (&tree)[kTrees], int in_bits,
                                             uint64_t x0, int L, int D, ForestLds& lds) {
  const int group = int(threadIdx.x >> 3);
  ForestTree tr = tree[0];
  if constexpr (kTrees == 2)
    if (group & 1) tr = tree[1];
  if (group < kTrees) {
    QuadState st = quad_root(tr.chunk, tr.party);
    quad_walk<kVal, SUFHIP_GROUP_ADD>(aes, K, tr.chunk, in_bits, 0, L, x0, tr.party, st);
    forest_put<kVal>(lds, 0, group, st);
  }
  // Each level's record is read a level ahead (a group keeps its tree).
  const uint32_t q = threadIdx.x & 3u;
  const uint8_t* cw = tr.chunk + 16 + 33 * L;
  QuadCw<kVal> c{};
  if (D > 0) c = load_quad_cw<kVal>(cw, q);
  __syncthreads();
  for (int l = 0; l < D; ++l) {
    if (l + 1 < D) cw += 33;
    const QuadCw<kVal> next = load_quad_cw<kVal>(cw, q);
    const int kids = kTrees << (l + 1);
    for (int k = group; k < kids; k += kForestBlock / 8) {
      const int idx = k / kTrees;
      QuadState st = forest_get(lds, l & 1, (idx >> 1) * kTrees + k % kTrees);
      quad_level<kVal, SUFHIP_GROUP_ADD>(aes, K, c, uint32_t(idx) & 1u, tr.party, st);
      forest_put<kVal>(lds, (l + 1) & 1, k, st);
    }
    c = next;
    __syncthreads();
  }
}

// Expansion depth for a tile of `points` points: none while their walks take
// one pass of the workgroup on 8 lanes each (a level of the expansion then
// costs what it saves), else about one node per point.
inline int forest_depth(size_t points, int trees) {
  if (points * size_t(trees) <= 128) return 0;
  int d = 0;
  while ((size_t(2) << d) <= points && (trees << (d + 1)) <= kForestNodes) ++d;
  return d;
}

}  // namespace
}  // namespace sufhip
