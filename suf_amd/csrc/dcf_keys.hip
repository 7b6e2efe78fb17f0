// Comparison bits of several broadcast DCF keys at the same public points, in
// launches of up to 64 keys (sufhip_dcf_eval_keys): the predicate and cut queries of a
// composite gate, which composite_eval_batch_backend evaluates one by one
// (include/gates/composite_fss.hpp:2132-2250).
//
// A workgroup takes one key and one tile of the points
// (dcf_forest_device.hpp).  22 keys at 4096 points of 15 bits take 72 us: 31
// of the common prefix's 47 levels, 8 of the expansion, 20 of the points' last
// 9 levels (5.8 ms as one launch per key, each on 4 of 256 CUs at 2.7 us a
// level).
#include <hip/hip_runtime.h>

#include <cstddef>

#include "dcf_forest_device.hpp"

namespace sufhip {
namespace {

constexpr int kKeysPerLaunch = 64;

struct DcfKeysArgs {
  DcfKeySel key_sel;
  const uint64_t* xs;
  size_t n;
  size_t tile;
  int depth;  // expansion depth of a tile
  int quad;   // points walk on 8 lanes each
  const uint8_t* key[kKeysPerLaunch];
  uint8_t* out[kKeysPerLaunch];
  uint8_t bits[kKeysPerLaunch];
};
static_assert(sizeof(DcfKeysArgs) <= 4096, "kernel argument block must fit in 4 KB");

__global__ void __launch_bounds__(kForestBlock) dcf_eval_keys_kernel(DcfKeysArgs a) {
  __shared__ ForestLds lds;
  const size_t first = size_t(blockIdx.x) * a.tile;
  const size_t count = a.n - first < a.tile ? a.n - first : a.tile;
  const uint64_t* xs = a.xs + first;
  const uint64_t x0 = xs[0];
  const uint64_t diff = xor_points(xs, count, x0);
  if (threadIdx.x < 2) lds.diff[threadIdx.x] = 0;
  SUFHIP_DCF_TABLE_SETUP();
  const KeySelPtr keys = kernarg_key_sel(offsetof(DcfKeysArgs, key_sel));
  const QuadKeys K = load_quad_keys(keys);
  const uint8_t* key = a.key[blockIdx.y];
  uint8_t* out = a.out[blockIdx.y] + first;
  const int in_bits = a.bits[blockIdx.y];
  const ForestTree tree[1] = {{key + 8, key[2] & 1u}};
  const int L = shared_levels(lds, diff, in_bits);
  const int D = a.depth < in_bits - L ? a.depth : in_bits - L;
  forest_build<kQuadBit, 1>(aes, K, tree, in_bits, x0, L, D, lds);
  const int from = L + D, buf = D & 1;
  if (a.quad) {
    for (size_t i = threadIdx.x >> 3; i < count; i += kForestBlock / 8) {
      const uint64_t x = xs[i];
      const int node = forest_node(x, in_bits - from, D);
      QuadState st = forest_get(lds, buf, node);
      quad_walk<kQuadBit, SUFHIP_GROUP_XOR>(aes, K, tree[0].chunk, in_bits, from, in_bits, x,
                                            tree[0].party, st);
      const U128 r = quad_finish<kQuadBit, SUFHIP_GROUP_XOR>(tree[0].chunk, in_bits,
                                                             tree[0].party, false, st);
      if ((threadIdx.x & 7u) == 4u) out[i] = uint8_t(r.lo);
    }
  } else {
    for (size_t i = threadIdx.x; i < count; i += kForestBlock) {
      const uint64_t x = xs[i];
      const int node = forest_node(x, in_bits - from, D);
      const uint4 sn = lds.s[buf][node];
      uint32_t s[4] = {sn.x, sn.y, sn.z, sn.w};
      out[i] = uint8_t(walk_bit_from(aes, keys, tree[0].chunk, in_bits, from, x, s,
                                     lds.t[buf][node], uint32_t(lds.v[buf][node])));
    }
  }
}

}  // namespace
}  // namespace sufhip

using namespace sufhip;

extern "C" {

int sufhip_dcf_eval_keys(const uint8_t* prg_state, const sufhip_dcf_key_job* jobs, int count,
                         const uint64_t* d_xs, size_t n, void* stream) {
  SUFHIP_REQUIRE(count >= 0 && (count == 0 || jobs), "sufhip_dcf_eval_keys: bad jobs");
  SUFHIP_REQUIRE(n < size_t(1) << 38, "sufhip_dcf_eval_keys: n too large");
  if (n == 0 || count == 0) return SUFHIP_OK;
  SUFHIP_REQUIRE(prg_state && d_xs, "sufhip_dcf_eval_keys: null pointer");
  for (int j = 0; j < count; ++j) {
    SUFHIP_REQUIRE(jobs[j].in_bits >= 1 && jobs[j].in_bits <= 64,
                   "sufhip_dcf_eval_keys: in_bits out of range");
    SUFHIP_REQUIRE(jobs[j].d_key && jobs[j].d_out, "sufhip_dcf_eval_keys: null key or output");
    SUFHIP_REQUIRE(jobs[j].key_bytes == sufhip_dcf_key_bytes(jobs[j].in_bits, 1),
                   "sufhip_dcf_eval_keys: key_bytes does not match (in_bits, 1-byte payload)");
  }
  int cus = 0;
  if (int rc = cu_count(&cus)) return rc;
  DcfKeysArgs a{};
  Prg4 prg;
  fill_prg4(prg_state, &prg);
  fill_key_sel(prg, &a.key_sel);
  a.xs = d_xs;
  a.n = n;
  // A launch gives every key the same number of equal tiles, as many as the
  // CUs hold.  From kForestBlock points per CU on, where a key alone fills the
  // chip, a launch's keys have one width and such a number that at most 1/16
  // of the CUs stay without a tile: points with no common prefix walk 56 levels
  // of a 64-bit key and 4 of a 12-bit one.  20 + 2 such keys at 2^18 points, us
  // in one launch / by width: no common prefix 6290 / 5115 (5940 as a launch
  // per key), points of 15 bits 1053 / 853.
  const bool whole = n >= size_t(kForestBlock) * size_t(cus);
  for (int bits = whole ? 64 : 1; bits >= 1; --bits) {
    const auto taken = [&](int j) { return !whole || jobs[j].in_bits == bits; };
    int left = 0;
    for (int j = 0; j < count; ++j) left += taken(j) ? 1 : 0;
    for (int j = 0, m = 0; left > 0; left -= m) {
      m = left < kKeysPerLaunch ? left : kKeysPerLaunch;
      if (whole)
        while (m <= cus && 16 * (cus / m * m) < 15 * cus) --m;
      // At least 8 points to a tile (one wave of quad walks).
      size_t tiles = size_t(cus / m > 0 ? cus / m : 1);
      a.tile = (n + tiles - 1) / tiles;
      if (a.tile < 8) a.tile = 8;
      tiles = (n + a.tile - 1) / a.tile;
      a.quad = a.tile <= 256;
      a.depth = forest_depth(a.tile, 1);
      for (int q = 0; q < m; ++j) {
        if (!taken(j)) continue;
        a.key[q] = jobs[j].d_key;
        a.out[q] = jobs[j].d_out;
        a.bits[q++] = uint8_t(jobs[j].in_bits);
      }
      hipLaunchKernelGGL(dcf_eval_keys_kernel, dim3(unsigned(tiles), unsigned(m)),
                         dim3(kForestBlock), 0, as_stream(stream), a);
      if (int rc = check_launch("dcf_eval_keys_kernel")) return rc;
    }
  }
  return SUFHIP_OK;
}

}  // extern "C"
