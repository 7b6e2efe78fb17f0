// Row-local task blocks for two parties on one GPU, each in one launch.
//
// With both parties in one process every open is a local sum, so a task
// chain whose rounds only combine values of one row needs no grid-wide
// synchronisation: one workgroup runs all rounds of its row, holding the row
// in registers, with workgroup sums for the row reductions and one lane for
// the per-row scalar gates.  Element indices, triples and keys are those of
// the launch-per-step evaluation, so the shares are bit-identical to it.
//
//   layernorm2_kernel  LayerNormTask (include/runtime/phase_tasks.hpp:
//                      2186-2668) with RsqrtTask (:1383-1700)
//   softmax2_team_kernel    SoftmaxBlockTask (include/nn/softmax_block_task.hpp:
//                      97-450) with RowMaxDiffTask, nExp, row sum, Recip
#include <hip/hip_runtime.h>

#include <type_traits>

#include "chain_device.hpp"
#include "digit_planes.hpp"
#include "reduce_device.hpp"
#include "relu_tree_device.hpp"
#include "walk_device.hpp"

namespace sufhip {
namespace {

// Rows of up to 1024 elements: 512 threads, up to two elements each (half
// the per-thread element work of 256 threads; the first LayerNorm of the
// layer 22.6 -> 21.4 us).  Longer rows (up to 2048): 256 threads, up to eight
// elements each (at 512 threads eight elements spill).
constexpr int kLnBlock = 512;
constexpr int kLnWideBlock = 256;
constexpr int kLnMaxPer = 2;      // elements per thread at kLnBlock: cols <= 1024
constexpr int kLnPairPer = 4;     // at kLnWideBlock, two rows per CU: cols <= 1024
constexpr int kLnWidePer = 8;     // at kLnWideBlock: cols <= 2048
constexpr int kLnCopies = 4;  // the T table serves one lane per workgroup
using LnAes = AesLds<kLnCopies>;  // one lane's chain: the small table fills fastest
// Key-only walks of later gates' tables, run by the workgroups past the rows'
// (hosted_walk_role): up to kLnWalkJobs jobs.
constexpr int kLnWalkJobs = 24;

struct LnArgs {
  const uint64_t* x[2];
  int rows, cols;
  uint64_t inv_len, eps;
  TruncEpi tr[5];  // mean, var0, var1, norm, and the input's (with in_slices)
  uint64_t mask[5];
  sufhip_triple2 sq, norm;
  ChainArgs rs;
  uint64_t* out[2];
  sufhip_x_planes xp;
  const uint64_t* in_slices;  // optional: [slices][2][rows cols] partial products
  int in_count;
  int row_groups;              // workgroups [0, row_groups) run the rows
  WalkJobs<kLnWalkJobs> w;     // the others walk these jobs' tables
};
static_assert(sizeof(LnArgs) <= 4096, "kernel argument blocks must fit in 4 KB");

enum { kTrMean = 0, kTrVar0 = 1, kTrVar1 = 2, kTrNorm = 3, kTrIn = 4 };
constexpr int kLnMaxSlices = 8;
constexpr int kLnMaxInPer = kLnMaxPer;  // in_slices rows of up to 1024 elements

// Every load that does not depend on an open is issued when the row starts:
// x, both triples' shares, and (lane 0) the rsqrt chain's triples; the key
// headers of all truncation gates sit in LDS.  What remains serial per row
// is one table read per truncation gate and the rsqrt LUT's AES.
// kWalk: the workgroups past the rows' walk A.w's jobs (a separate
// instantiation, so that launches without walks keep the rows' own register
// allocation and LDS).
template <int kPer, bool kIn, int kBlock, bool kWalk>
__global__ void __launch_bounds__(kBlock, kBlock == kLnWideBlock && kPer <= kLnPairPer ? 2 : 1)
    layernorm2_kernel(LnArgs A) {
  constexpr int kLnWaves = kBlock / 64;
  if constexpr (kWalk) {
    if (int(blockIdx.x) >= A.row_groups) {
      hosted_walk_role<kLnWalkJobs, true>(A.w,
                                          (blockIdx.x - A.row_groups) * kBlock + threadIdx.x);
      return;
    }
  }
  __shared__ __align__(16) uint32_t tab[256 * kLnCopies];
  __shared__ ChainLds L;
  constexpr int kRsProds = chain_products<SUFHIP_CHAIN_RSQRT>();
  __shared__ TruncHdr th[5][2];
  __shared__ TruncHdr rth[kRsProds][2];  // the rsqrt chain's truncation key headers
  __shared__ uint64_t red[2][kLnWaves];
  __shared__ uint64_t bc[2];
  __shared__ ChainPre pre;
  fill_ttable<kLnCopies>(tab, kTDev.v);
  chain_stage(A.rs, 2, L);
  if (threadIdx.x < (kIn ? 10 : 8))
    th[threadIdx.x >> 1][threadIdx.x & 1] =
        read_trunc_hdr(A.tr[threadIdx.x >> 1].key[threadIdx.x & 1]);
  {
    TruncHdrStager<kRsProds> hs;
    hs.load(A.rs, 64);
    hs.store(rth);
  }
  __syncthreads();
  chain_compare(A.rs, L);
  __syncthreads();
  const LnAes aes{tab, threadIdx.x % kLnCopies};
  const ChainKeyInfo K = chain_key_info(A.rs, L);
  auto gate = [&](int j, uint64_t v) {
    return Two{{trunc_table_eval_h(th[j][0], A.tr[j].table[0], A.tr[j].f, v),
                trunc_table_eval_h(th[j][1], A.tr[j].table[1], A.tr[j].f, v)}};
  };
  const int cols = A.cols;
  for (int r = blockIdx.x; r < A.rows; r += A.row_groups) {
    const size_t base = size_t(r) * size_t(cols);
    // The row's rsqrt triples, one word per lane (visible to lane 0 after
    // the row sum's barriers).
    if (threadIdx.x < 24) pre.word(threadIdx.x) = chain_triple_word(A.rs, threadIdx.x, size_t(r));
    // Loads in the order of use (x, the square's triple, the norm triple):
    // each step then waits only for its own words, and the norm triple's
    // arrive while lane 0 runs the rsqrt chain.
    uint64_t d[kPer][2], sa[kPer][2], sb[kPer][2], sc[kPer][2], na[kPer][2], nc[kPer][2];
    if (kIn) {
      // x = tr_in(the open of the product's slice sums) + addend, written
      // out as the product's output.  All slice and addend loads first.
      const size_t mn = size_t(A.rows) * size_t(cols);
      const TruncEpi& ti = A.tr[kTrIn];
      uint64_t ad[kPer][2];
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const int c = threadIdx.x + k * kBlock;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          d[k][p] = 0;
          ad[k][p] = c < cols && ti.add[0] ? ti.add[p][base + c] : 0;
        }
      }
      // Slices in groups of four, then one by one: every load of a group is
      // unconditional (a lane past the row end reads the row's first
      // element and drops the sum), so a group is one round trip.  A load
      // whose value a select or branch might drop would be sunk into the
      // branch and wait for the loads before it.
      const int ns = A.in_count;
      auto add_slices = [&](int z0, auto nz) {
        constexpr int kN = decltype(nz)::value;
        uint64_t t[kPer][2][kN];
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
          const int c = threadIdx.x + k * kBlock;
          const size_t e = c < cols ? base + c : base;
#pragma unroll
          for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int dz = 0; dz < kN; ++dz)
              t[k][p][dz] = A.in_slices[(size_t(z0 + dz) * 2 + p) * mn + e];
        }
        // Every load of the group before any add (the scheduler otherwise
        // waits for each element's loads before issuing the next one's).
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < kPer; ++k)
#pragma unroll
          for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int dz = 0; dz < kN; ++dz) d[k][p] += t[k][p][dz];
      };
      int z0 = 0;
      for (; z0 + 4 <= ns; z0 += 4) add_slices(z0, std::integral_constant<int, 4>{});
      for (; z0 < ns; ++z0) add_slices(z0, std::integral_constant<int, 1>{});
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        if (threadIdx.x + k * kBlock >= cols) d[k][0] = d[k][1] = 0;
      }
      uint64_t zh[kPer], w[kPer][2];
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        zh[k] = d[k][0] + d[k][1] + A.mask[kTrIn];
        w[k][0] = trunc_table_word(th[kTrIn][0], ti.table[0], ti.f, zh[k]);
        w[k][1] = trunc_table_word(th[kTrIn][1], ti.table[1], ti.f, zh[k]);
      }
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const int c = threadIdx.x + k * kBlock;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          d[k][p] = c < cols ? trunc_table_out(th[kTrIn][p], ti.f, zh[k], w[k][p]) + ad[k][p] : 0;
          if (c < cols) ti.y[p][base + c] = d[k][p];
        }
      }
    } else {
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const int c = threadIdx.x + k * kBlock;
#pragma unroll
        for (int p = 0; p < 2; ++p) d[k][p] = c < cols ? A.x[p][base + c] : 0;
      }
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int c = threadIdx.x + k * kBlock;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        sa[k][p] = c < cols ? A.sq.a[p][base + c] : 0;
        sb[k][p] = c < cols ? A.sq.b[p][base + c] : 0;
        sc[k][p] = c < cols ? A.sq.c[p][base + c] : 0;
      }
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int c = threadIdx.x + k * kBlock;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        na[k][p] = c < cols ? A.norm.a[p][base + c] : 0;
        nc[k][p] = c < cols ? A.norm.c[p][base + c] : 0;
      }
    }
    const uint64_t nb0 = A.norm.b[0][r], nb1 = A.norm.b[1][r];
    uint64_t s0 = 0, s1 = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      s0 += d[k][0];
      s1 += d[k][1];
    }
    // mu = tr_mean(inv_len * row sum).
    block_sum2_u64<kLnWaves>(s0, s1, red);
    const Two mu = gate(kTrMean, s0 * A.inv_len + s1 * A.inv_len + A.mask[kTrMean]);
    // d = x - mu; q = d * d (Beaver), summed over the row.
    uint64_t q0 = 0, q1 = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int c = threadIdx.x + k * kBlock;
      if (c < cols) {
        d[k][0] -= mu.v[0];
        d[k][1] -= mu.v[1];
        const uint64_t dd = (d[k][0] - sa[k][0]) + (d[k][1] - sa[k][1]);
        const uint64_t ee = (d[k][0] - sb[k][0]) + (d[k][1] - sb[k][1]);
        q0 += sc[k][0] + dd * sb[k][0] + ee * sa[k][0] + dd * ee;
        q1 += sc[k][1] + dd * sb[k][1] + ee * sa[k][1];
      }
    }
    block_sum2_u64<kLnWaves>(q0, q1, red);
    const Two va = gate(kTrVar0, q0 * A.inv_len + q1 * A.inv_len + A.mask[kTrVar0]);
    const Two var = gate(kTrVar1, va.v[0] + va.v[1] + A.mask[kTrVar1]);
    // rsqrt of the row's variance on the first wave (its keystream blocks
    // column-parallel on eight lanes, the rest of the chain on every lane).
    if (threadIdx.x < 64) {
      const Two v{{var.v[0] + A.eps, var.v[1]}};
      const Two rs =
          chain_eval_quad<SUFHIP_CHAIN_RSQRT, LnAes>(A.rs, L, K, aes, size_t(r), v, pre, rth);
      if (threadIdx.x == 0) {
        bc[0] = rs.v[0];
        bc[1] = rs.v[1];
      }
    }
    __syncthreads();
    // out = tr_norm(d * rs[row]) (row-broadcast Beaver).
    const uint64_t ee = (bc[0] - nb0) + (bc[1] - nb1);
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int c = threadIdx.x + k * kBlock;
      if (c < cols) {
        const size_t i = base + c;
        const uint64_t dd = (d[k][0] - na[k][0]) + (d[k][1] - na[k][1]);
        const uint64_t z0 = nc[k][0] + dd * nb0 + ee * na[k][0] + dd * ee;
        const uint64_t z1 = nc[k][1] + dd * nb1 + ee * na[k][1];
        const Two o = gate(kTrNorm, z0 + z1 + A.mask[kTrNorm]);
        if (A.out[0]) {
          A.out[0][i] = o.v[0];
          A.out[1][i] = o.v[1];
        }
        if (A.xp.planes) {
          put_x_digits(A.xp, size_t(A.rows), i, 0, o.v[0]);
          put_x_digits(A.xp, size_t(A.rows), i, 1, o.v[1]);
        }
      }
    }
    __syncthreads();  // bc is rewritten for the next row
  }
}

// Softmax rows: up to kSmSlots rows per workgroup of 768 lanes, every phase
// flat over the workgroup: a max-tree level's pairs, the scores' nExp chains
// and the normalisation are dealt to the lanes whatever row they belong to.
// What bounds a row is its chain of dependent steps (7 to 9 tree levels, two
// LUT chains), so a workgroup's rows go through it together: with rows of
// very different lengths (causal attention) a wave or two per row leaves most
// lanes idle, and a long row's levels run in turn on its own wave.
//   12 x 128 causal rows: 53 us (60 with two waves per row);
//   4 x 300 causal rows: 75 us (166 with one wave per row).
constexpr int kSmRounds = 10;
constexpr int kSmMaxRow = 512;
constexpr int kSmSlots = 8;
constexpr int kSmThreads = 768;
constexpr int kSmPer = 4;  // scores per lane: 6 rows of 512 or 8 of 384
using SmAes = AesLds2<32>;
constexpr size_t kSmLdsCap = 160 * 1024;

struct SmArgs {
  sufhip_operand2 x;
  int pre;
  TruncEpi pre_tr[2];
  uint64_t pre_mask[2];
  const int32_t* offs;
  const int32_t* round_off;
  TreeKeys<kSmRounds> keys;
  int rows, max_row, slots, groups;
  ChainArgs nexp, recip;
  sufhip_triple2 norm;
  TruncEpi tr_norm;
  uint64_t norm_mask;
  uint64_t* out[2];
  uint64_t* dense;
  const uint64_t* dense_a[2];
  int dense_cols;
  sufhip_kb_planes dkb;  // the dense open also as digit planes
};

struct SmStatic {
  uint32_t tab[SmAes::kSpanWords];
  TreeLds<kSmRounds> t;
  ChainLds nexp, recip;
  TruncHdr thn[3][2], thr[3][2];  // the chains' truncation key headers
  ChainPreN<3> rpre[kSmSlots];  // each row's reciprocal triples
  uint32_t j0[kSmSlots][kSmRounds];  // each row's tree slot offsets
  // The group's rows: global row (-1: none), first score, length, levels of
  // the max tree, and where the row's scores (even levels) and odd levels
  // start in the level buffers.
  int row[kSmSlots], first[kSmSlots], len[kSmSlots], levels[kSmSlots];
  int even0[kSmSlots + 1], odd0[kSmSlots];
  int pairs0[kSmRounds][kSmSlots + 1];  // first pair of each row in a level
  uint64_t sum[kSmSlots][2];   // row sums of e
  uint64_t inv[kSmSlots][2];   // their reciprocals
};

// Everything the block keeps in LDS for the whole launch -- the AES span,
// every tree round's keys, both chains' keys -- in one staging pass: a
// thread issues all of its global loads (about a dozen table words, up to
// two tree items and a few chain items, spread over the workgroup by a flat
// item index) before its first LDS store, so staging costs about one memory
// round trip.  load() and store() split the pass so that the first rows'
// loads go in between; the caller syncs after store().
template <int kThreads>
struct SmStagerT {
  static constexpr int kChainPer = 2;
  typename SmAes::template Filler<kThreads> tf;
  TreeStager<kSmRounds, 2> ts;
  TruncHdrStager<3> hn, hr;
  uint4 cv[kChainPer];
  int c0, nn, nc;
  __device__ __forceinline__ void load(const SmArgs& a) {
    static_assert(kSmRounds * kTreeItems <= 2 * kThreads, "SmStager: tree items in one pass");
    tf.load(kTDev.v);
    ts.load(kernarg_tree_keys<kSmRounds>(offsetof(SmArgs, keys)), int(threadIdx.x));
    hn.load(a.nexp, 0);
    hr.load(a.recip, 64);
    // Chain items continue the tree's flat item space.
    nn = chain_items(a.nexp, 4);
    nc = nn + chain_items(a.recip, 2);
    const int shift = (a.keys.rounds * kTreeItems) % kThreads;
    c0 = (int(threadIdx.x) + kThreads - shift) % kThreads;
#pragma unroll
    for (int u = 0; u < kChainPer; ++u) {
      // Unconditional loads on a clamped item (see TreeStager::load).
      const int c = c0 + u * kThreads < nc ? c0 + u * kThreads : 0;
      bool rn, rr;
      const uint64_t* an = chain_item_addr(a.nexp, 4, c < nn ? c : 0, &rn);
      const uint64_t* ar = chain_item_addr(a.recip, 2, c < nn ? 0 : c - nn, &rr);
      cv[u] = chain_item_fetch(c < nn ? an : ar, c < nn ? rn : rr);
    }
  }
  __device__ __forceinline__ void store(const SmArgs& a, SmStatic& st) const {
#pragma unroll
    for (int u = 0; u < kChainPer; ++u) {
      const int c = c0 + u * kThreads;
      if (c < nn)
        chain_item_store(a.nexp, 4, st.nexp, c, cv[u]);
      else if (c < nc)
        chain_item_store(a.recip, 2, st.recip, c - nn, cv[u]);
    }
    // Chains with more items than one pass covers (wide LUTs): the rest
    // item by item.
    for (int c = c0 + kChainPer * kThreads; c < nc; c += kThreads) {
      if (c < nn)
        chain_item_store(a.nexp, 4, st.nexp, c, chain_item_load(a.nexp, 4, c));
      else
        chain_item_store(a.recip, 2, st.recip, c - nn, chain_item_load(a.recip, 2, c - nn));
    }
    ts.store(st.t);
    tf.store(st.tab);
    hn.store(st.thn);
    hr.store(st.thr);
    if (threadIdx.x == 0) {
      st.t.diff = a.keys.own_ks;
      st.nexp.diff = a.nexp.own_ks;
      st.recip.diff = a.recip.own_ks;
    }
  }
};
// The kernel's argument read afresh from the kernarg segment: an opaque copy
// of its address per phase, so that a phase's pointers are scalar loads where
// they are used.  The block's ~100 uniform pointers exceed the scalar
// registers, and held over the whole kernel they are moved to vector lanes
// and back.
__device__ __forceinline__ const SmArgs& sm_args() {
  typedef const __attribute__((address_space(4))) SmArgs* Ptr;
  Ptr p = (Ptr)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const SmArgs*)p;
}

// kN values of a lane in registers, indexed by a (uniform) loop variable.
// (One or two are named members: the compiler puts a short indexed vector or
// array in private memory.)
template <int kN>
struct LaneVals {
  typedef uint64_t Vec __attribute__((ext_vector_type(kN)));
  Vec v = 0;
  __device__ __forceinline__ uint64_t get(int k) const { return v[k]; }
  __device__ __forceinline__ void set(int k, uint64_t x) { v[k] = x; }
};
template <>
struct LaneVals<1> {
  uint64_t a = 0;
  __device__ __forceinline__ uint64_t get(int) const { return a; }
  __device__ __forceinline__ void set(int, uint64_t x) { a = x; }
};
template <>
struct LaneVals<2> {
  uint64_t a = 0, b = 0;
  __device__ __forceinline__ uint64_t get(int k) const { return k ? b : a; }
  __device__ __forceinline__ void set(int k, uint64_t x) {
    a = k ? a : x;
    b = k ? x : b;
  }
};

// The slot whose range [start[s], start[s + 1]) holds x (the last one whose
// start is at most x; empty slots share their start with the next).
__device__ __forceinline__ int sm_slot(const int* start, int x) {
  int s = 0;
#pragma unroll
  for (int k = 1; k < kSmSlots; ++k) s += x >= start[k] ? 1 : 0;
  return s;
}

// Pairs p0 + Q + 192 u (Q the lane's quad, u < U) of level k over the
// workgroup's rows: tree_chunk's step with each pair's row looked up.  The
// AES block of a pair is spread over its quad; lane q then finishes the
// quad's pair u = q.
template <int U>
__device__ __forceinline__ void tree_flat(const SmArgs& a, const SmStatic& st, const SmAes& aes,
                                          int k, const uint64_t* src, int sw, const int* src0,
                                          uint64_t* dst, int dw, const int* dst0, int p0,
                                          int pairs, bool one_ks) {
  constexpr int kQuads = kSmThreads / 4;
  const TreeLds<kSmRounds>& L = st.t;
  const int Q = int(threadIdx.x >> 2), q = int(threadIdx.x & 3);
  uint64_t xh[U], xb[U][2];
  int iv[U][2], at[U];
  uint32_t blk[2][U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int p = p0 + Q + kQuads * u < pairs ? p0 + Q + kQuads * u : pairs - 1;
    const int r = sm_slot(st.pairs0[k], p);
    const int t = p - st.pairs0[k][r];
    const uint64_t* s = src + src0[r] + 2 * t;
    at[u] = dst0[r] + t;
    const uint64_t xa0 = s[0], xb0 = s[1], xa1 = s[sw], xb1 = s[sw + 1];
    xh[u] = (xa0 - xb0) + (xa1 - xb1) + a.keys.mask[k];
    xb[u][0] = xb0;
    xb[u][1] = xb1;
    const uint32_t j = st.j0[r][k] + uint32_t(t);
#pragma unroll
    for (int p2 = 0; p2 < 2; ++p2) {
      iv[u][p2] = (p2 == 1 && one_ks) ? iv[u][0] : tree_interval(a.keys, L, k, p2, xh[u]);
      const uint64_t ctr = L.nonce[k][p2] ^ (uint64_t(j) << 32) ^ (uint64_t(iv[u][p2]) * 2);
      blk[p2][u] = q == 0 ? uint32_t(ctr) : (q == 1 ? uint32_t(ctr >> 32) : 0u);
    }
  }
  tree_keystream<U>(aes, L, k, q, one_ks, blk);
  // Lane q takes block q: column c of it is lane c's word of blk[.][q].
  uint32_t w[2][4];
  uint64_t x = 0, b[2] = {0, 0};
  int ivq[2] = {0, 0}, o0 = 0;
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int c = 0; c < 4; ++c) w[p][c] = 0;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    uint32_t c[2][4];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const uint32_t v = blk[p][u];
      c[p][0] = quad_bcast<0>(v);
      c[p][1] = quad_bcast<1>(v);
      c[p][2] = quad_bcast<2>(v);
      c[p][3] = quad_bcast<3>(v);
    }
    if (q == u) {
#pragma unroll
      for (int p = 0; p < 2; ++p) {
#pragma unroll
        for (int j = 0; j < 4; ++j) w[p][j] = c[p][j];
        b[p] = xb[u][p];
        ivq[p] = iv[u][p];
      }
      x = xh[u];
      o0 = at[u];
    }
  }
  if (q < U && p0 + Q + kQuads * q < pairs) {
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const uint64_t k0 = uint64_t(w[p][0]) | uint64_t(w[p][1]) << 32;
      const uint64_t k1 = uint64_t(w[p][2]) | uint64_t(w[p][3]) << 32;
      const bool zero = L.party[k][p] == 0;
      const uint64_t q0 = zero ? k0 : L.pay[k][p][2 * ivq[p]] - k0;
      const uint64_t q1 = zero ? k1 : L.pay[k][p][2 * ivq[p] + 1] - k1;
      dst[(p ? dw : 0) + o0] = b[p] + q0 + q1 * x;
    }
  }
}

template <int kPer>
__global__ void __launch_bounds__(kSmThreads) softmax2_team_kernel(SmArgs) {
  const SmArgs& a = sm_args();
  __shared__ __align__(16) SmStatic st;
  extern __shared__ uint64_t rowbuf[];
  const int mr = a.max_row, half = (mr + 1) / 2;
  const int we = a.slots * mr, wo = a.slots * half;  // party strides of the level buffers
  uint64_t* even = rowbuf;
  uint64_t* odd = rowbuf + 2 * we;
  const int tid = int(threadIdx.x), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // This lane's scores, one in every 768 of the group's; the loops over them
  // stay loops (unrolled, the chains' code outgrows the instruction cache).
  LaneVals<kPer> s0, s1;
  // Group g's rows: slot k takes row k G + g or, for odd k, (k + 1) G - 1 - g,
  // which evens out the lengths of causal rows.  The offsets are uniform
  // (scalar) loads; every lane then loads its scores -- through the optional
  // truncations of their open -- into registers and level 0 of the tree, its
  // first score's normalisation triple, and (one wave per row) the
  // reciprocal's triples and the row's tree slots.  Before the first barrier
  // nothing staged is read, so the first group's loads overlap the staging.
  // Length of slot k's row r and its first score f (0: none).
  auto row_len = [&](const SmArgs& a, int k, int r, int& f) {
    if (k >= a.slots || r >= a.rows) return 0;
    f = a.offs[r];
    const int n = a.offs[r + 1] - f;
    return n < 1 || n > mr ? 0 : n;  // refused on the host
  };
  auto load_rows = [&](int g) {
    const SmArgs& a = sm_args();
    const auto row_of = [&](int k) {
      return (k & 1) ? (k + 1) * a.groups - 1 - g : k * a.groups + g;
    };
    int total = 0, ototal = 0;
    int e0[kSmSlots], f0[kSmSlots], ln[kSmSlots];
#pragma unroll
    for (int k = 0; k < kSmSlots; ++k) {
      const int r = row_of(k);
      int f = 0;
      const int n = row_len(a, k, r, f);
      e0[k] = total;
      f0[k] = f;
      ln[k] = n;
      if (tid == k) {
        st.row[k] = n > 0 ? r : -1;
        st.first[k] = f;
        st.len[k] = n;
        st.levels[k] = n > 1 ? 32 - __builtin_clz(uint32_t(n - 1)) : 0;
        st.even0[k] = total;
        st.odd0[k] = ototal;
        st.sum[k][0] = st.sum[k][1] = 0;
      }
      total += n;
      ototal += (n + 1) >> 1;
    }
    if (tid == 0) st.even0[kSmSlots] = total;
    if (wave < kSmSlots) {
      const int r = row_of(wave);
      int f = 0;
      const int n = row_len(a, wave, r, f);
      if (n > 0 && lane < 18)
        st.rpre[wave].word(lane) = chain_triple_word(a.recip, lane, size_t(r));
      tree_row_offsets(a.keys, a.round_off, a.rows, r, n, st.j0[wave]);
    }
    // Lane k of the wave after the rows': level k's pairs.
    if (wave == kSmSlots && lane < kSmRounds) {
      int p = 0;
#pragma unroll
      for (int k = 0; k < kSmSlots; ++k) {
        st.pairs0[lane][k] = p;
        const int n = ln[k] > 0 ? ((ln[k] - 1) >> lane) + 1 : 0;  // the level's length
        p += n >> 1;
      }
      st.pairs0[lane][kSmSlots] = p;
    }
#pragma unroll 1
    for (int k = 0; k < kPer && kSmThreads * k < total; ++k) {
      const int e = tid + kSmThreads * k;
      if (e >= total) continue;
      int base = 0, f = f0[0];
#pragma unroll
      for (int j = 1; j < kSmSlots; ++j)
        if (e >= e0[j]) {
          base = e0[j];
          f = f0[j];
        }
      const size_t i = size_t(f) + size_t(e - base);
      uint64_t v0 = operand_at(a.x, 0, i), v1 = operand_at(a.x, 1, i);
      // Compile-time gate indices: a runtime index into the argument block
      // would copy it to private scratch memory.
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if (t >= a.pre) break;
        const uint64_t o = v0 + v1 + a.pre_mask[t];
        v0 = trunc_table_eval(a.pre_tr[t].key[0], a.pre_tr[t].table[0], a.pre_tr[t].f, o);
        v1 = trunc_table_eval(a.pre_tr[t].key[1], a.pre_tr[t].table[1], a.pre_tr[t].f, o);
      }
      s0.set(k, v0);
      s1.set(k, v1);
      even[e] = v0;
      even[we + e] = v1;
    }
  };
  {
    SmStagerT<kSmThreads> stager;
    stager.load(a);
    load_rows(blockIdx.x);
    stager.store(a, st);
  }
  __syncthreads();
  tree_compare(a.keys, st.t);
  chain_compare(a.nexp, st.nexp);
  chain_compare(a.recip, st.recip);
  __syncthreads();
  const SmAes aes = SmAes::make(st.tab);
  const ChainKeyInfo Kn = chain_key_info(a.nexp, st.nexp);
  const ChainKeyInfo Kr = chain_key_info(a.recip, st.recip);
  const uint32_t shared = ~st.t.diff;
  for (int g = blockIdx.x; g < a.groups; g += gridDim.x) {
    if (g != int(blockIdx.x)) {
      load_rows(g);
      __syncthreads();
    }
    // The max tree, level by level over all rows.
    for (int k = 0; k < a.keys.rounds; ++k) {
      const SmArgs& a = sm_args();
      const int pairs = __builtin_amdgcn_readfirstlane(st.pairs0[k][kSmSlots]);
      if (pairs == 0) break;  // every row is down to one element
      const uint64_t* src = (k & 1) ? odd : even;
      uint64_t* dst = (k & 1) ? even : odd;
      const int sw = (k & 1) ? wo : we, dw = (k & 1) ? we : wo;
      const int* src0 = (k & 1) ? st.odd0 : st.even0;
      const int* dst0 = (k & 1) ? st.even0 : st.odd0;
      const bool one_ks = (shared >> k) & 1u;
      for (int p0 = 0; p0 < pairs; p0 += kSmThreads / 2) {
        const int left = pairs - p0;
        if (left <= 16 * wave) break;  // no pair for this wave's quads
        if (left > kSmThreads / 4)
          tree_flat<2>(a, st, aes, k, src, sw, src0, dst, dw, dst0, p0, pairs, one_ks);
        else
          tree_flat<1>(a, st, aes, k, src, sw, src0, dst, dw, dst0, p0, pairs, one_ks);
      }
      // An odd level's last element passes through.
      if (tid < kSmSlots && k < st.levels[tid]) {
        const int n = ((st.len[tid] - 1) >> k) + 1;
        if (n & 1) {
          dst[dst0[tid] + (n >> 1)] = src[src0[tid] + n - 1];
          dst[dw + dst0[tid] + (n >> 1)] = src[sw + src0[tid] + n - 1];
        }
      }
      __syncthreads();
    }
    // e = nExp(max - s) for the lane's scores, both parties' keystream blocks
    // in one lockstep group, and the row sums: a wave adds its lanes of a row,
    // then the waves meet in LDS.
    const int total = __builtin_amdgcn_readfirstlane(st.even0[kSmSlots]);
    LaneVals<kPer> ex0, ex1;
#pragma unroll 1
    for (int k = 0; k < kPer; ++k) {
      const SmArgs& a = sm_args();
      const int w0 = kSmThreads * k + 64 * wave;  // the wave's first score
      if (w0 >= total) break;
      const bool ok = w0 + lane < total;
      const int x = ok ? w0 + lane : total - 1;  // past the end: dropped
      const int q = sm_slot(st.even0, x);
      const uint64_t* fin = (st.levels[q] & 1) ? odd + st.odd0[q] : even + st.even0[q];
      const int fw = (st.levels[q] & 1) ? wo : we;
      const size_t i = size_t(st.first[q]) + size_t(x - st.even0[q]);
      const Two d{{fin[0] - s0.get(k), fin[fw] - s1.get(k)}};
      const Two ev = chain_eval<SUFHIP_CHAIN_CUBIC, SmAes, plain_loader<SUFHIP_CHAIN_CUBIC>,
                                kPer <= 2>(
          a.nexp, st.nexp, Kn, aes, i, d, plain_loader<SUFHIP_CHAIN_CUBIC>{&a.nexp, i}, st.thn);
      const uint64_t v0 = ok ? ev.v[0] : 0, v1 = ok ? ev.v[1] : 0;
      ex0.set(k, v0);
      ex1.set(k, v1);
      const int lo = __builtin_amdgcn_readfirstlane(q), hi = __builtin_amdgcn_readlane(q, 63);
      for (int r = lo; r <= hi; ++r) {
        const uint64_t p0 = wave_sum_u64(q == r ? v0 : 0);
        const uint64_t p1 = wave_sum_u64(q == r ? v1 : 0);
        if (lane < 2)
          atomicAdd(reinterpret_cast<unsigned long long*>(&st.sum[r][lane]),
                    static_cast<unsigned long long>(lane ? p1 : p0));
      }
    }
    // The normalisation triple of score x of the group (its row q): the first
    // pass's loads are issued here, to land under the reciprocal.
    uint64_t na[2], nb[2], nc[2];
    auto load_norm = [&](const SmArgs& a, int x, int q) {
      const size_t i = size_t(st.first[q]) + size_t(x - st.even0[q]);
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        na[p] = a.norm.a[p][i];
        nb[p] = a.norm.b[p][st.row[q]];
        nc[p] = a.norm.c[p][i];
      }
    };
    if (tid < total) load_norm(sm_args(), tid, sm_slot(st.even0, tid));
    __syncthreads();
    // inv = Recip(row sum), one wave per row (its keystream blocks
    // column-parallel on eight lanes).
    if (wave < kSmSlots && st.row[wave] >= 0) {
      const SmArgs& a = sm_args();
      const Two iv = chain_eval_quad<SUFHIP_CHAIN_RECIP, SmAes, ChainPreN<3>>(
          a.recip, st.recip, Kr, aes, size_t(st.row[wave]),
          Two{{st.sum[wave][0], st.sum[wave][1]}}, st.rpre[wave], st.thr);
      if (lane == 0) {
        st.inv[wave][0] = iv.v[0];
        st.inv[wave][1] = iv.v[1];
      }
    }
    __syncthreads();
    // prob = tr_norm(e * inv[row]) (row-broadcast Beaver), and the next
    // product's open over the dense row.
#pragma unroll 1
    for (int k = 0; k < kPer; ++k) {
      const SmArgs& a = sm_args();
      const int x = tid + kSmThreads * k;
      if (x >= total) break;
      const int q = sm_slot(st.even0, x), r = st.row[q], j = x - st.even0[q];
      const size_t i = size_t(st.first[q]) + size_t(j);
      if (k > 0) load_norm(a, x, q);
      const uint64_t ee = (st.inv[q][0] - nb[0]) + (st.inv[q][1] - nb[1]);
      const uint64_t dd = (ex0.get(k) - na[0]) + (ex1.get(k) - na[1]);
      const uint64_t z0 = nc[0] + dd * nb[0] + ee * na[0] + dd * ee;
      const uint64_t z1 = nc[1] + dd * nb[1] + ee * na[1];
      const uint64_t o = z0 + z1 + a.norm_mask;
      const uint64_t p0 = trunc_table_eval(a.tr_norm.key[0], a.tr_norm.table[0], a.tr_norm.f, o);
      const uint64_t p1 = trunc_table_eval(a.tr_norm.key[1], a.tr_norm.table[1], a.tr_norm.f, o);
      if (a.out[0]) {
        a.out[0][i] = p0;
        a.out[1][i] = p1;
      }
      if (a.dense) {
        const size_t di = size_t(r) * size_t(a.dense_cols) + size_t(j);
        const uint64_t dv = (p0 - a.dense_a[0][di]) + (p1 - a.dense_a[1][di]);
        a.dense[di] = dv;
        if (a.dkb.planes) put_kb_digits(a.dkb, di, dv);
      }
    }
    if (a.dense) {
      // Past the rows' ends the probability is 0.
      for (int x = tid; x < a.slots * a.dense_cols; x += kSmThreads) {
        const int q = x / a.dense_cols, j = x - q * a.dense_cols;
        if (st.row[q] < 0 || j < st.len[q]) continue;
        const size_t di = size_t(st.row[q]) * size_t(a.dense_cols) + size_t(j);
        const uint64_t dv = (uint64_t(0) - a.dense_a[0][di]) + (uint64_t(0) - a.dense_a[1][di]);
        a.dense[di] = dv;
        if (a.dkb.planes) put_kb_digits(a.dkb, di, dv);
      }
    }
    __syncthreads();  // the row buffers are rewritten by the next group
  }
}

// The dynamic LDS of a softmax launch goes past 64 KB; allowed once per
// kernel.
template <int kPer>
bool sm_lds_allowed() {
  static const bool ok =
      hipFuncSetAttribute(reinterpret_cast<const void*>(&softmax2_team_kernel<kPer>),
                          hipFuncAttributeMaxDynamicSharedMemorySize,
                          int(kSmLdsCap - sizeof(SmStatic))) == hipSuccess;
  return ok;
}

int triple_ok(const sufhip_triple2& t) {
  return t.a[0] && t.a[1] && t.b[0] && t.b[1] && t.c[0] && t.c[1];
}

int table_epi(const sufhip_trunc_epilogue& t, size_t n, const char* what, TruncEpi* e) {
  sufhip_trunc_epilogue c = t;
  if (c.add[0] || c.add[1]) {
    set_error(std::string(what) + ": the block's truncations take no addend");
    return SUFHIP_ERR_INVALID;
  }
  uint64_t dummy = 0;
  c.y[0] = c.y[1] = &dummy;  // the block writes its own outputs
  return make_epi(&c, n, what, e);
}

}  // namespace
}  // namespace sufhip

using namespace sufhip;

extern "C" {

int sufhip_layernorm2(const sufhip_layernorm2_args* args, void* stream) {
  SUFHIP_REQUIRE(args != nullptr, "sufhip_layernorm2: null args");
  const sufhip_layernorm2_args& g = *args;
  SUFHIP_REQUIRE(g.rows >= 0 && g.cols >= 1 && g.cols <= kLnWideBlock * kLnWidePer,
                 "sufhip_layernorm2: cols in [1, 2048]");
  SUFHIP_REQUIRE(g.walk_count >= 0 && (g.walk_count == 0 || (g.walk_jobs && g.walk_prg_state)),
                 "sufhip_layernorm2: walk_count >= 0, walk jobs and PRG state given");
  if (g.rows == 0)
    return g.walk_count > 0
               ? sufhip_trunc_prepare_batch(g.walk_prg_state, g.walk_jobs, g.walk_count, stream)
               : SUFHIP_OK;
  SUFHIP_REQUIRE((g.in_slices || (g.x[0] && g.x[1])) &&
                     (g.out[0] == nullptr) == (g.out[1] == nullptr) &&
                     (g.out[0] || g.out_planes.planes),
                 "sufhip_layernorm2: null input or output");
  SUFHIP_REQUIRE(!g.in_slices || (g.in_slice_count >= 2 && g.in_slice_count <= kLnMaxSlices),
                 "sufhip_layernorm2: in_slice_count in [2, 8]");
  SUFHIP_REQUIRE(!g.in_slices || g.cols <= kLnBlock * kLnMaxInPer,
                 "sufhip_layernorm2: in_slices need cols <= 1024");
  SUFHIP_REQUIRE(x_planes_ok(g.out_planes, size_t(g.rows) * size_t(g.cols)) &&
                     (!g.out_planes.planes || g.out_planes.cols == g.cols),
                 "sufhip_layernorm2: out_planes needs cols == the row length, rows and cols "
                 "multiples of 32, 16-byte alignment");
  SUFHIP_REQUIRE(triple_ok(g.sq) && triple_ok(g.norm), "sufhip_layernorm2: a triple is missing");
  SUFHIP_REQUIRE(g.rsqrt.kind == SUFHIP_CHAIN_RSQRT && g.rsqrt.n == size_t(g.rows),
                 "sufhip_layernorm2: the rsqrt chain must be RSQRT over rows elements");
  const size_t n = size_t(g.rows) * size_t(g.cols);
  LnArgs A{};
  if (int rc = make_chain_args(g.rsqrt, false, "sufhip_layernorm2 rsqrt", &A.rs)) return rc;
  if (int rc = table_epi(g.tr_mean, size_t(g.rows), "sufhip_layernorm2 tr_mean", &A.tr[kTrMean]))
    return rc;
  if (int rc = table_epi(g.tr_var[0], size_t(g.rows), "sufhip_layernorm2 tr_var", &A.tr[kTrVar0]))
    return rc;
  if (int rc = table_epi(g.tr_var[1], size_t(g.rows), "sufhip_layernorm2 tr_var", &A.tr[kTrVar1]))
    return rc;
  if (int rc = table_epi(g.tr_norm, n, "sufhip_layernorm2 tr_norm", &A.tr[kTrNorm])) return rc;
  if (g.in_slices) {
    if (int rc = make_epi(&g.tr_in, n, "sufhip_layernorm2 tr_in", &A.tr[kTrIn])) return rc;
    A.in_slices = g.in_slices;
    A.in_count = g.in_slice_count;
    A.mask[kTrIn] = g.in_mask;
  }
  A.x[0] = g.x[0];
  A.x[1] = g.x[1];
  A.rows = g.rows;
  A.cols = g.cols;
  A.inv_len = g.inv_len;
  A.eps = g.eps;
  A.mask[kTrMean] = g.mean_mask;
  A.mask[kTrVar0] = g.var_mask[0];
  A.mask[kTrVar1] = g.var_mask[1];
  A.mask[kTrNorm] = g.norm_mask;
  A.sq = g.sq;
  A.norm = g.norm;
  A.xp = g.out_planes;
  A.out[0] = g.out[0];
  A.out[1] = g.out[1];
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess)
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  const int grid = g.rows < cus * 8 ? g.rows : cus * 8;
  const int per = (g.cols + kLnBlock - 1) / kLnBlock;
  // More rows than CUs: 256 lanes per row leave the registers for two rows on
  // a CU, where 512 hold one (300 x 1001: 38 -> 25 us).  A row alone takes
  // about 1 us longer, so up to one row per CU keeps 512.
  const bool pair = g.rows > cus && per <= kLnMaxPer && !A.in_slices;
  const int block = (per <= kLnMaxPer || A.in_slices) && !pair ? kLnBlock : kLnWideBlock;
  A.row_groups = grid;
  // The walks: one workgroup per CU fits beside the rows' (the kernel's
  // registers allow one), so the CUs without a row hold one pass of them.
  // The 256-lane forms walk nothing themselves.
  size_t walk_lanes = 0;
  if (block == kLnBlock) {
    if (int rc = plan_hosted_walk(g.walk_prg_state, g.walk_jobs, g.walk_count,
                                  size_t(cus > grid ? cus - grid : 0) * size_t(block), stream,
                                  "sufhip_layernorm2 walk", A.w, &walk_lanes))
      return rc;
  } else if (g.walk_count > 0) {
    if (int rc = sufhip_trunc_prepare_batch(g.walk_prg_state, g.walk_jobs, g.walk_count, stream))
      return rc;
  }
  const size_t walk_groups = (walk_lanes + block - 1) / size_t(block);
  SUFHIP_REQUIRE(size_t(grid) + walk_groups <= 0x7fffffffu, "sufhip_layernorm2: grid too large");
  const dim3 launch(unsigned(size_t(grid) + walk_groups));
  hipStream_t s = as_stream(stream);
  auto rows512 = [&](auto per_c, auto in_c) {
    constexpr int kP = decltype(per_c)::value;
    constexpr bool kI = decltype(in_c)::value;
    if (walk_groups > 0)
      hipLaunchKernelGGL((layernorm2_kernel<kP, kI, kLnBlock, true>), launch, dim3(kLnBlock), 0,
                         s, A);
    else
      hipLaunchKernelGGL((layernorm2_kernel<kP, kI, kLnBlock, false>), launch, dim3(kLnBlock), 0,
                         s, A);
  };
  using PerOne = std::integral_constant<int, 1>;
  if (pair) {
    hipLaunchKernelGGL((layernorm2_kernel<kLnPairPer, false, kLnWideBlock, false>), launch,
                       dim3(kLnWideBlock), 0, s, A);
  } else if (A.in_slices) {
    if (per <= 1)
      rows512(PerOne{}, std::true_type{});
    else
      rows512(std::integral_constant<int, kLnMaxInPer>{}, std::true_type{});
  } else if (per <= 1) {
    rows512(PerOne{}, std::false_type{});
  } else if (per <= kLnMaxPer) {
    rows512(std::integral_constant<int, kLnMaxPer>{}, std::false_type{});
  } else {
    hipLaunchKernelGGL((layernorm2_kernel<kLnWidePer, false, kLnWideBlock, false>), launch,
                       dim3(kLnWideBlock), 0, s, A);
  }
  return check_launch("layernorm2_kernel");
}


int sufhip_softmax2(const sufhip_softmax2_args* args, void* stream) {
  SUFHIP_REQUIRE(args != nullptr, "sufhip_softmax2: null args");
  const sufhip_softmax2_args& g = *args;
  SUFHIP_REQUIRE(g.rows >= 0, "sufhip_softmax2: rows < 0");
  SUFHIP_REQUIRE(g.max_row >= 1 && g.max_row <= kSmMaxRow,
                 "sufhip_softmax2: rows of 1..512 elements");
  SUFHIP_REQUIRE(g.pre_truncs >= 0 && g.pre_truncs <= 2, "sufhip_softmax2: pre_truncs in [0, 2]");
  SmArgs A{};
  if (int rc = make_tree_keys<kSmRounds>(g.keys, g.rounds, g.max_row, "sufhip_softmax2", &A.keys))
    return rc;
  if (g.rows == 0) return SUFHIP_OK;
  SUFHIP_REQUIRE(g.d_row_offsets && (g.rounds == 0 || g.d_round_offsets),
                 "sufhip_softmax2: null offsets");
  SUFHIP_REQUIRE(g.nexp.kind == SUFHIP_CHAIN_CUBIC && g.recip.kind == SUFHIP_CHAIN_RECIP &&
                     g.recip.n == size_t(g.rows),
                 "sufhip_softmax2: nexp must be CUBIC and recip RECIP over rows elements");
  const size_t n = g.nexp.n;
  if (int rc = make_chain_args(g.nexp, false, "sufhip_softmax2 nexp", &A.nexp)) return rc;
  SUFHIP_REQUIRE(A.nexp.plain,
                 "sufhip_softmax2: the nExp chain's triples must be plain arrays (no index, "
                 "multiplier, shift or negation; stride 1 or 3)");
  if (int rc = make_chain_args(g.recip, false, "sufhip_softmax2 recip", &A.recip)) return rc;
  if (int rc = check_operand(g.x, n, "sufhip_softmax2 x")) return rc;
  SUFHIP_REQUIRE(g.x.t[0].p[0] != nullptr, "sufhip_softmax2: empty input operand");
  for (int q = 0; q < g.pre_truncs; ++q)
    if (int rc = table_epi(g.pre[q], n, "sufhip_softmax2 pre", &A.pre_tr[q])) return rc;
  SUFHIP_REQUIRE(triple_ok(g.norm), "sufhip_softmax2: the norm triple is missing");
  if (int rc = table_epi(g.tr_norm, n, "sufhip_softmax2 tr_norm", &A.tr_norm)) return rc;
  SUFHIP_REQUIRE((g.out[0] == nullptr) == (g.out[1] == nullptr),
                 "sufhip_softmax2: out needs both parties or neither");
  SUFHIP_REQUIRE(g.out[0] || g.d_dense, "sufhip_softmax2: no output");
  SUFHIP_REQUIRE(!g.d_dense || (g.dense_a[0] && g.dense_a[1] && g.dense_cols >= g.max_row),
                 "sufhip_softmax2: the dense open needs both a shares and dense_cols >= max_row");
  A.x = g.x;
  A.pre = g.pre_truncs;
  A.pre_mask[0] = g.pre_mask[0];
  A.pre_mask[1] = g.pre_mask[1];
  A.offs = g.d_row_offsets;
  A.round_off = g.d_round_offsets;
  A.rows = g.rows;
  A.max_row = g.max_row;
  A.norm = g.norm;
  A.norm_mask = g.norm_mask;
  A.out[0] = g.out[0];
  A.out[1] = g.out[1];
  A.dense = g.d_dense;
  A.dense_a[0] = g.dense_a[0];
  A.dense_a[1] = g.dense_a[1];
  A.dense_cols = g.d_dense ? g.dense_cols : 0;
  SUFHIP_REQUIRE(!g.dense_planes.planes ||
                     (g.d_dense && kb_planes_ok(g.dense_planes, size_t(g.rows) * g.dense_cols)),
                 "sufhip_softmax2: dense_planes need d_dense and cover rows x dense_cols");
  A.dkb = g.d_dense ? g.dense_planes : sufhip_kb_planes{};
  // Rows per workgroup: 8 while their scores fit kSmPer per lane (and their
  // level buffers the LDS), 6 of the longest.
  A.slots = g.max_row <= kSmThreads * kSmPer / kSmSlots ? kSmSlots : 6;
  const size_t dyn = size_t(A.slots) * tree_row_words(g.max_row) * sizeof(uint64_t);
  // Scores per lane at most: 1, 2 or kSmPer.
  const int scores = A.slots * g.max_row;
  const bool lds_ok = scores <= kSmThreads       ? sm_lds_allowed<1>()
                      : scores <= 2 * kSmThreads ? sm_lds_allowed<2>()
                                                 : sm_lds_allowed<kSmPer>();
  SUFHIP_REQUIRE(sizeof(SmStatic) + dyn <= kSmLdsCap && lds_ok,
                 "sufhip_softmax2: the kernel's LDS size was refused");
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess)
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  // Rows dealt evenly to whole passes of one workgroup per CU.
  const size_t passes = (size_t(g.rows) + size_t(A.slots) * cus - 1) / (size_t(A.slots) * cus);
  const size_t groups = passes * size_t(cus);
  A.groups = int(groups < size_t(g.rows) ? groups : size_t(g.rows));
  const int grid = A.groups < cus ? A.groups : cus;
  const hipStream_t s = as_stream(stream);
  if (scores <= kSmThreads)
    hipLaunchKernelGGL(softmax2_team_kernel<1>, dim3(grid), dim3(kSmThreads), dyn, s, A);
  else if (scores <= 2 * kSmThreads)
    hipLaunchKernelGGL(softmax2_team_kernel<2>, dim3(grid), dim3(kSmThreads), dyn, s, A);
  else
    hipLaunchKernelGGL(softmax2_team_kernel<kSmPer>, dim3(grid), dim3(kSmThreads), dyn, s, A);
  return check_launch("softmax2_team_kernel");
}

}  // extern "C"
