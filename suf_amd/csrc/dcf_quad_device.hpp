// The myl7 DCF walk (third_party/myl7_fss/src/dcf.c:146-193) on 8 lanes, for
// batches too small to fill the chip with one walk per lane.
//
// Lanes 0-3 of a group compute the next-seed block AES_{K_{2b}}(s) and lanes
// 4-7 the value block AES_{K_{2b+1}}(s), one state column per lane
// (AesLds4::quad_terms' scheme).  A level is bounded by its serial
// chain -- ten rounds of table address, LDS read, three quad exchanges -- and
// a lane here issues 4 table reads a round where the one-lane walk issues 32,
// so the chain is 0.65 us a level against 2.1 us (measured at 300 to 8192
// keys, one or two waves per SIMD).  The exchanges make it 36 VALU operations
// per block and round instead of 28, so larger batches take fewer lanes per
// walk (two, at the end of this file, then one).
//
// A lane only ever needs one column of two keys, K_h and K_{2+h} (h its
// half), so the round keys live in 22 registers: nothing but table reads goes
// through the LDS, and the choice of key by the input bit is off the chain.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "dcf_device.hpp"

namespace sufhip {
namespace {

// Value of lane - 4 in this lane's row of 16 (lanes 4-7 and 12-15 of a row;
// the others hold nothing of use).
__device__ __forceinline__ uint32_t row_shr4(uint32_t v) {
  return uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0x114, 0xf, 0xf, false));
}

// Little-endian word at byte address p + 4 idx (any alignment; reads the
// aligned words idx and idx + 1 around it).
__device__ __forceinline__ uint32_t word_at(const uint8_t* p, int idx) {
  const uintptr_t a = reinterpret_cast<uintptr_t>(p);
  const uint32_t* w = reinterpret_cast<const uint32_t*>(a & ~uintptr_t(3));
  return __builtin_amdgcn_alignbyte(w[idx + 1], w[idx], uint32_t(a & 3));
}

// Round key column q of this lane's half: K_h and K_h ^ K_{2+h}.
struct QuadKeys {
  uint32_t k[11], d[11];
};

__device__ __forceinline__ QuadKeys load_quad_keys(KeySelPtr sel) {
  QuadKeys K;
  const uint32_t l = threadIdx.x & 7u;
  const uint32_t at = (l >> 2) * 8u + (l & 3u);
#pragma unroll
  for (int r = 0; r < 11; ++r) {
    K.k[r] = sel[16 * r + at];
    K.d[r] = sel[16 * r + at + 4];
  }
  return K;
}

// The same keys from a Prg4 in the kernel argument.
__device__ __forceinline__ QuadKeys load_quad_keys(const Prg4& prg) {
  QuadKeys K;
  const uint32_t h = (threadIdx.x >> 2) & 1u, q = threadIdx.x & 3u;
#pragma unroll
  for (int r = 0; r < 11; ++r) {
    K.k[r] = prg.rk[h][4 * r + q];
    K.d[r] = K.k[r] ^ prg.rk[2 + h][4 * r + q];
  }
  return K;
}

// AES_{K_{2b + h}} of N seeds in lockstep (column q of seed n in s[n]).
// N = 1: b = b0; else b = (b0 + n) & 1, with b0 known at compile time.
template <int N, class Aes>
__device__ __forceinline__ void quad_encrypt_n(const Aes& aes, const QuadKeys& K, uint32_t b0,
                                               uint32_t (&s)[N]) {
  const auto key = [&](int r, int n) {
    if (N == 1) return xor_and(K.k[r], 0u - b0, K.d[r]);
    return ((b0 + n) & 1u) ? K.k[r] ^ K.d[r] : K.k[r];
  };
#pragma unroll
  for (int n = 0; n < N; ++n) s[n] ^= key(0, n);
#pragma unroll
  for (int r = 1; r < 10; ++r) {
    uint32_t a[N][4];
#pragma unroll
    for (int n = 0; n < N; ++n) aes.quad_terms(s[n], a[n]);
#pragma unroll
    for (int n = 0; n < N; ++n)
      s[n] = a[n][0] ^ key(r, n) ^ quad_rot<1>(a[n][1]) ^ quad_rot<2>(a[n][2]) ^
             quad_rot<3>(a[n][3]);
  }
  uint32_t u[N][4];
#pragma unroll
  for (int n = 0; n < N; ++n) aes.quad_last(s[n], u[n]);
#pragma unroll
  for (int n = 0; n < N; ++n)
    s[n] = u[n][0] ^ key(10, n) ^ quad_rot<1>(u[n][1]) ^ quad_rot<2>(u[n][2]) ^
           quad_rot<3>(u[n][3]);
}

// What a walk accumulates: bit 0 of the share, its low 64 bits (additive
// group: + and - carry only upwards), or all 16 bytes.
enum QuadVal { kQuadBit, kQuadLow64, kQuadFull };

// A correction word record: the aligned words a lane needs of it, read a
// level ahead of their use.
template <int kVal>
struct QuadCw {
  static constexpr int kV = kVal == kQuadBit ? 1 : (kVal == kQuadLow64 ? 3 : 5);
  uint32_t s0, s1;  // words q and q + 1: s_cw column q
  uint32_t v[kV];   // words 4..: v_cw
  uint32_t tb;      // word 8: the t byte (bit mode and low 64)
  uint32_t sh;
};

template <int kVal>
__device__ __forceinline__ QuadCw<kVal> load_quad_cw(const uint8_t* p, uint32_t q) {
  const uintptr_t a = reinterpret_cast<uintptr_t>(p);
  GlobalWords w = (GlobalWords)(a & ~uintptr_t(3));
  QuadCw<kVal> c;
  c.s0 = w[q];
  c.s1 = w[q + 1];
#pragma unroll
  for (int j = 0; j < QuadCw<kVal>::kV; ++j) c.v[j] = w[4 + j];
  if constexpr (kVal == kQuadFull)
    c.tb = 0;
  else
    c.tb = w[8];
  c.sh = uint32_t(a & 3);
  return c;
}

// Seed word q (both halves), control bit (both halves), accumulated value
// (meaningful in the value half; kQuadBit: bit 0 of lane 4's lo).
struct QuadState {
  uint32_t s, t;
  U128 v;
};

template <int kVal, int kGroup>
__device__ __forceinline__ void quad_level(const AesLds4& aes, const QuadKeys& K,
                                           const QuadCw<kVal>& c, uint32_t xi, uint32_t party,
                                           QuadState& st) {
  const uint32_t l = threadIdx.x & 7u, q = l & 3u;
  uint32_t enc[1] = {st.s};
  quad_encrypt_n<1>(aes, K, xi, enc);
  uint32_t on = enc[0] ^ st.s;
  const uint32_t tmask = 0u - st.t;
  if constexpr (kVal == kQuadBit) {
    st.v.lo ^= (on ^ ((c.v[0] >> (8 * c.sh)) & tmask)) & 1u;
  } else if constexpr (kVal == kQuadLow64) {
    const uint64_t vd0 = uint64_t(quad_bcast<0>(on)) | uint64_t(quad_bcast<1>(on)) << 32;
    const uint64_t cv = uint64_t(__builtin_amdgcn_alignbyte(c.v[1], c.v[0], c.sh)) |
                        uint64_t(__builtin_amdgcn_alignbyte(c.v[2], c.v[1], c.sh)) << 32;
    const uint64_t vd = vd0 + (st.t ? cv : 0);
    st.v.lo += party ? 0 - vd : vd;
  } else {
    U128 vd = mk(quad_bcast<0>(on), quad_bcast<1>(on), quad_bcast<2>(on),
                 quad_bcast<3>(on) & 0x7fffffffu);
    const U128 cv = mk(__builtin_amdgcn_alignbyte(c.v[1], c.v[0], c.sh),
                       __builtin_amdgcn_alignbyte(c.v[2], c.v[1], c.sh),
                       __builtin_amdgcn_alignbyte(c.v[3], c.v[2], c.sh),
                       __builtin_amdgcn_alignbyte(c.v[4], c.v[3], c.sh));
    if (st.t) vd = gadd<kGroup>(vd, cv);
    if (party) vd = gneg<kGroup>(vd);
    st.v = gadd<kGroup>(st.v, vd);
  }
  const uint32_t tb = (kVal == kQuadFull ? c.v[QuadCw<kVal>::kV - 1] : c.tb) >> (8 * c.sh);
  uint32_t tn = quad_bcast<3>(on) >> 31;
  if (q == 3) on &= 0x7fffffffu;
  on ^= __builtin_amdgcn_alignbyte(c.s1, c.s0, c.sh) & tmask;
  tn ^= (xi ? tb : (tb >> 1)) & st.t & 1u;
  // The seed half's next seed and t move to the value half (lane - 4).
  const uint32_t os = row_shr4(on), ts = row_shr4(tn);
  st.s = l >= 4 ? os : on;
  st.t = l >= 4 ? ts : tn;
}

__device__ __forceinline__ QuadState quad_root(const uint8_t* chunk, uint32_t party) {
  const uint32_t q = threadIdx.x & 3u;
  uint32_t s = word_at(chunk, int(q));
  if (q == 3) s &= 0x7fffffffu;
  return QuadState{s, party, U128{0, 0}};
}

// Levels [from, to) of an in_bits-level walk at x, each record read a level
// ahead of its use.
template <int kVal, int kGroup>
__device__ __forceinline__ void quad_walk(const AesLds4& aes, const QuadKeys& K,
                                          const uint8_t* chunk, int in_bits, int from, int to,
                                          uint64_t x, uint32_t party, QuadState& st) {
  const uint32_t q = threadIdx.x & 3u;
  const uint8_t* cw = chunk + 16 + 33 * from;
  if (from >= to) return;
  QuadCw<kVal> c = load_quad_cw<kVal>(cw, q);
#pragma unroll 1
  for (int i = from; i < to; ++i) {
    // The last level's look-ahead reads its own record again.
    if (i + 1 < to) cw += 33;
    const QuadCw<kVal> next = load_quad_cw<kVal>(cw, q);
    quad_level<kVal, kGroup>(aes, K, c, uint32_t(x >> (in_bits - 1 - i)) & 1u, party, st);
    c = next;
  }
}

// Share after the last level: v + (-1)^party (s + t cw_np1), in the value
// half (kQuadBit: bit 0, in lane 4).
template <int kVal, int kGroup>
__device__ __forceinline__ U128 quad_finish(const uint8_t* chunk, int in_bits, uint32_t party,
                                            bool more_after, const QuadState& st) {
  const uint8_t* np1 = chunk + 16 + 33 * in_bits;
  if constexpr (kVal == kQuadBit) {
    return U128{(st.v.lo ^ st.s ^ (word_at(np1, 0) & st.t)) & 1u, 0};
  } else {
    uint32_t n[4];
    load16_bytes(np1, more_after, n);
    U128 sv = mk(quad_bcast<0>(st.s), quad_bcast<1>(st.s), quad_bcast<2>(st.s),
                 quad_bcast<3>(st.s));
    if constexpr (kVal == kQuadLow64) {
      const uint64_t s = sv.lo + (st.t ? mk(n[0], n[1], 0, 0).lo : 0);
      return U128{st.v.lo + (party ? 0 - s : s), 0};
    } else {
      if (st.t) sv = gadd<kGroup>(sv, mk(n[0], n[1], n[2], n[3]));
      if (party) sv = gneg<kGroup>(sv);
      return gadd<kGroup>(st.v, sv);
    }
  }
}

// ---------------------------------------------------------------------------
// The same walk on 2 lanes, for batches between the 8-lane walks' and a full
// chip of one-lane walks: the even lane forms the next-seed block, the odd
// lane the value block.  A lane's two keys K_h and K_{2+h} (h its parity) are
// 88 registers, so nothing but table reads goes through the LDS, and 512
// lanes per CU (two waves per SIMD) have the registers for them.
constexpr int kPairBlock = 512;

struct PairKeys {
  uint32_t k[44], d[44];  // K_h and K_h ^ K_{2+h}
};

__device__ __forceinline__ PairKeys load_pair_keys(KeySelPtr sel) {
  PairKeys K;
  const uint32_t at = (threadIdx.x & 1u) * 8u;
#pragma unroll
  for (int r = 0; r < 11; ++r)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      K.k[4 * r + j] = sel[16 * r + at + j];
      K.d[4 * r + j] = sel[16 * r + at + 4 + j];
    }
  return K;
}

// The even lane's value of each lane pair, in both.
__device__ __forceinline__ uint32_t pair_even(uint32_t v) {
  return uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0xa0, 0xf, 0xf, true));
}

// Walk of one chunk by a lane pair; the odd lane returns the 16-byte share.
template <int kGroup>
__device__ __forceinline__ U128 pair_walk(const AesLds4& aes, const PairKeys& K,
                                          const uint8_t* chunk, int in_bits, uint64_t x,
                                          uint32_t party, bool more_after) {
  uint32_t s[4];
  load16_bytes(chunk, true, s);
  s[3] &= 0x7fffffffu;
  uint32_t t = party;
  U128 v{0, 0};
  const uint8_t* cw = chunk + 16;
#pragma unroll 1
  for (int i = 0; i < in_bits; ++i, cw += 33) {
    const CwRawFull cr = load_cw_raw_full(cw);
    const uint32_t xi = uint32_t(x >> (in_bits - 1 - i)) & 1u;
    const uint32_t m = 0u - xi;
    uint32_t a[4], o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) a[j] = xor_and(s[j], m, K.d[j]) ^ K.k[j];
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
        a[c] = xor_and(SUFHIP_BITOP3(SUFHIP_BITOP3(tv[4 * c], tv[4 * c + 1], tv[4 * c + 2], 0x96),
                                     tv[4 * c + 3], K.k[4 * r + c], 0x96),
                       m, K.d[4 * r + c]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
      o[c] = xor_and(aes.last_col(a[c], a[(c + 1) & 3], a[(c + 2) & 3], a[(c + 3) & 3],
                                  K.k[40 + c] ^ s[c]),
                     m, K.d[40 + c]);
    const CwFull c = decode_cw_full(cr);
    const uint32_t tmask = 0u - t;
    // The odd lane's value; the even lane's v is not used.
    U128 vd = mk(o[0], o[1], o[2], o[3] & 0x7fffffffu);
    if (t) vd = gadd<kGroup>(vd, mk(c.v[0], c.v[1], c.v[2], c.v[3]));
    if (party) vd = gneg<kGroup>(vd);
    v = gadd<kGroup>(v, vd);
    // The even lane's next seed and control bit, to both.
    uint32_t tn = (o[3] >> 31) ^ ((xi ? c.tb : (c.tb >> 1)) & t & 1u);
    o[3] &= 0x7fffffffu;
#pragma unroll
    for (int j = 0; j < 4; ++j) s[j] = pair_even(o[j] ^ (c.s[j] & tmask));
    t = pair_even(tn);
  }
  uint32_t np1[4];
  load16_bytes(cw, more_after, np1);
  U128 sv = mk(s[0], s[1], s[2], s[3]);
  if (t) sv = gadd<kGroup>(sv, mk(np1[0], np1[1], np1[2], np1[3]));
  if (party) sv = gneg<kGroup>(sv);
  return gadd<kGroup>(v, sv);
}

}  // namespace
}  // namespace sufhip
