// DCF key generation (myl7 dcf_gen, third_party/myl7_fss/src/dcf.c:42-142,
// written in the adapter layout of include/proto/myl7_fss_backend.hpp:156-210)
// on 8 lanes per key: one of a level's eight PRG blocks per lane.
//
// Lane 4 p + b of a group computes AES_{K_b}(s_p) ^ s_p, p the party and b
// the output block (left seed, left value, right seed, right value).  A lane
// uses one key for the whole walk, so its 44 round-key words stay in
// registers and only table reads go through the LDS; the blocks then meet in
// DPP exchanges (the partner lane p ^ 1 for the differences of the two
// parties, the own quad for the correction words).  2^18 keys of 64 levels
// take 1.55 ms (2.5 ms with one key per lane: its eight blocks in turn, round
// keys in LDS, 144 bytes of scratch); the table reads are 85% of the LDS
// pipe's time at 2.2 clocks per wave read, and the VALU's share is as large.
// One key takes 82 us (835 before): 1.3 us a level, the serial chain of a
// block.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "dcf_device.hpp"

namespace sufhip {
namespace {

// Value of the lane four away in this lane's group of eight (lane ^ 4): the
// half-row mirror, then the quad's own mirror.
__device__ __forceinline__ uint32_t swap4(uint32_t v) {
  const uint32_t m = uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x141, 0xf, 0xf, true));
  return uint32_t(__builtin_amdgcn_update_dpp(0, int(m), 0x1b, 0xf, 0xf, true));
}

__device__ __forceinline__ U128 swap4_128(U128 v) {
  return mk(swap4(uint32_t(v.lo)), swap4(uint32_t(v.lo >> 32)), swap4(uint32_t(v.hi)),
            swap4(uint32_t(v.hi >> 32)));
}

// Lane c's value in the whole quad.  Bound control is on (as in swap4): the
// compiler then needs no register zeroed ahead of each exchange, about 40
// operations of a level.
template <int c>
__device__ __forceinline__ U128 quad_bcast128(U128 v) {
  const auto b = [](uint32_t w) {
    return uint32_t(__builtin_amdgcn_update_dpp(0, int(w), 0x55 * c, 0xf, 0xf, true));
  };
  return mk(b(uint32_t(v.lo)), b(uint32_t(v.lo >> 32)), b(uint32_t(v.hi)),
            b(uint32_t(v.hi >> 32)));
}

// The round keys of this lane's PRG key K_{lane & 3}; prg4 points at a Prg4
// in the kernel argument.
struct GenKeys {
  uint32_t k[44];
};

__device__ __forceinline__ GenKeys load_gen_keys(KeySelPtr prg4) {
  GenKeys K;
#pragma unroll
  for (int w = 0; w < 44; ++w) K.k[w] = prg4[(threadIdx.x & 3u) * 44u + w];
  return K;
}

// AES_K(s) ^ s with the round keys in registers.
__device__ __forceinline__ U128 gen_block(const AesLds4& aes, const GenKeys& K, U128 s) {
  const uint32_t in[4] = {uint32_t(s.lo), uint32_t(s.lo >> 32), uint32_t(s.hi),
                          uint32_t(s.hi >> 32)};
  uint32_t a[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) a[j] = in[j] ^ K.k[j];
#pragma unroll
  for (int r = 1; r < 10; ++r) {
    uint32_t ad[16], tv[16];
#pragma unroll
    for (int n = 0; n < 16; ++n)
      ad[n] = __builtin_amdgcn_perm(a[((n >> 2) + n) & 3], aes.base[n & 3], AesLds4::sel(n & 3));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < 16; ++n) tv[n] = lds_word(aes.lds, ad[n]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 4; ++c)
      a[c] = SUFHIP_BITOP3(SUFHIP_BITOP3(tv[4 * c], tv[4 * c + 1], tv[4 * c + 2], 0x96),
                           tv[4 * c + 3], K.k[4 * r + c], 0x96);
  }
  uint32_t o[4];
#pragma unroll
  for (int c = 0; c < 4; ++c)
    o[c] = aes.last_col(a[c], a[(c + 1) & 3], a[(c + 2) & 3], a[(c + 3) & 3], K.k[40 + c] ^ in[c]);
  return mk(o[0], o[1], o[2], o[3]);
}

// 8 bytes at any address (one unaligned store).
__device__ __forceinline__ void store8(uint8_t* p, uint64_t v) {
  __builtin_memcpy(p, &v, 8);
}

__device__ __forceinline__ U128 pick(bool c, U128 a, U128 b) {
  return U128{c ? a.lo : b.lo, c ? a.hi : b.hi};
}

// Chunk c of one key pair for f(x) = beta * 1[x < alpha], by the whole group
// of 8 lanes.  seeds: the chunk's 32 bytes (party-0 seed, party-1 seed); pay:
// the payload's payload_len bytes; out0, out1: the two keys.
template <int kGroup>
__device__ __forceinline__ void gen_chunk(const AesLds4& aes, const GenKeys& K, int nb, int chunks,
                                          int payload_len, int c, uint64_t alpha,
                                          const uint8_t* pay, const uint8_t* seeds, uint8_t* out0,
                                          uint8_t* out1) {
  const uint32_t l = threadIdx.x & 7u, b = l & 3u;
  const bool p1 = l >= 4;
  uint8_t* out = p1 ? out1 : out0;
  if (c == 0 && b == 0)
    store8(out, uint64_t(uint32_t(nb) | uint32_t(chunks) << 8 | uint32_t(p1) << 16) |
                    uint64_t(uint32_t(payload_len)) << 32);
  U128 beta{0, 0};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int at = 16 * c + i;
    if (at < payload_len) beta.lo |= uint64_t(pay[at]) << (8 * i);
    if (at + 8 < payload_len) beta.hi |= uint64_t(pay[at + 8]) << (8 * i);
  }
  beta.hi &= kMsbClear;
  U128 s{0, 0};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    s.lo |= uint64_t(seeds[16 * p1 + i]) << (8 * i);
    s.hi |= uint64_t(seeds[16 * p1 + 8 + i]) << (8 * i);
  }
  uint8_t* rec = out + 8 + size_t(c) * (32 + 33 * size_t(nb));
  if (b < 2) store8(rec + 8 * b, b ? s.hi : s.lo);
  rec += 16;
  s.hi &= kMsbClear;
  uint32_t t = p1 ? 1 : 0;
  U128 v{0, 0};
#pragma unroll 1
  for (int i = 0; i < nb; ++i, rec += 33) {
    const U128 own = gen_block(aes, K, s);
    const U128 oth = swap4_128(own);
    const bool ai = (alpha >> (nb - 1 - i)) & 1u;
    // The parties' t bits always differ on alpha's path.
    const bool t1 = (t != 0) == p1;
    const U128 x{own.lo ^ oth.lo, own.hi ^ oth.hi};
    // Party 1's block minus party 0's (the value lanes'; bit 127 dropped).
    U128 d;
    if constexpr (kGroup == SUFHIP_GROUP_XOR) {
      d = U128{x.lo, x.hi & kMsbClear};
    } else {
      U128 e0 = pick(p1, oth, own), e1 = pick(p1, own, oth);
      e0.hi &= kMsbClear;
      e1.hi &= kMsbClear;
      d = gadd<kGroup>(e1, gneg<kGroup>(e0));
    }
    // lose = side alpha does not take, keep = side it takes
    const U128 x0 = quad_bcast128<0>(x), x2 = quad_bcast128<2>(x);
    const U128 d1 = quad_bcast128<1>(d), d3 = quad_bcast128<3>(d);
    U128 s_cw = pick(ai, x0, x2);
    s_cw.hi &= kMsbClear;
    const U128 d_lose = pick(ai, d1, d3), d_keep = pick(ai, d3, d1);
    U128 v_cw = gadd<kGroup>(d_lose, gneg<kGroup>(v));
    if (ai) v_cw = gadd<kGroup>(v_cw, beta);
    // Negated with t1 (beta's sign then follows: -(d - v) - beta).
    if (t1) v_cw = gneg<kGroup>(v_cw);
    v = gadd<kGroup>(v, gneg<kGroup>(d_keep));
    v = gadd<kGroup>(v, t1 ? gneg<kGroup>(v_cw) : v_cw);
    const uint32_t tl_cw = uint32_t(x0.hi >> 63) ^ uint32_t(ai) ^ 1u;
    const uint32_t tr_cw = uint32_t(x2.hi >> 63) ^ uint32_t(ai);
    const U128 half = pick(b < 2, s_cw, v_cw);
    store8(rec + 8 * b, (b & 1u) ? half.hi : half.lo);
    if (b == 3) rec[32] = uint8_t(tl_cw << 1 | tr_cw);
    const U128 keep = pick(ai, quad_bcast128<2>(own), quad_bcast128<0>(own));
    const uint32_t tk = uint32_t(keep.hi >> 63);
    s.lo = keep.lo ^ (t ? s_cw.lo : 0);
    s.hi = (keep.hi & kMsbClear) ^ (t ? s_cw.hi : 0);
    t = tk ^ (t & (ai ? tr_cw : tl_cw));
  }
  const U128 so = swap4_128(s);
  U128 last = gadd<kGroup>(pick(p1, s, so), gneg<kGroup>(pick(p1, so, s)));
  last = gadd<kGroup>(last, gneg<kGroup>(v));
  if ((t != 0) == p1) last = gneg<kGroup>(last);
  if (b < 2) store8(rec + 8 * b, b ? last.hi : last.lo);
}

}  // namespace
}  // namespace sufhip
