// Device building blocks of the myl7/fss v0.7.1 DCF shared by the batch
// kernels (dcf.hip) and the truncation gate (trunc_gate.hip): AES tables,
// correction-word loaders, the tree walks and the per-lane key writer.
#pragma once

#include <hip/hip_runtime.h>

#include "aes_lds.hpp"
#include "sufhip_internal.hpp"

namespace sufhip {
namespace {


// One workgroup per CU: the four replicated AES tables take 128 KB of the
// CU's 160 KB LDS.  Kernels loop over the batch in grid strides.
#ifndef SUFHIP_DCF_BLOCK
#define SUFHIP_DCF_BLOCK 512
#endif
constexpr int kDcfBlock = SUFHIP_DCF_BLOCK;

// AES tables for every DCF kernel: four rotated T tables, 32 copies each.
using DcfAes = AesLds4;

struct Prg4 {
  uint32_t rk[4][44];  // K_0..K_3: DCF uses PRG output blocks 0..3
};

struct U128 {
  uint64_t lo, hi;
};

__device__ __forceinline__ U128 mk(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3) {
  return U128{uint64_t(w0) | uint64_t(w1) << 32, uint64_t(w2) | uint64_t(w3) << 32};
}

constexpr uint64_t kMsbClear = 0x7fffffffffffffffull;

template <int kGroup>
__device__ __forceinline__ U128 gadd(U128 a, U128 b) {
  if constexpr (kGroup == SUFHIP_GROUP_XOR) {
    return U128{a.lo ^ b.lo, a.hi ^ b.hi};
  } else {
    uint64_t lo = a.lo + b.lo;
    uint64_t hi = a.hi + b.hi + (lo < a.lo ? 1 : 0);
    return U128{lo, hi & kMsbClear};
  }
}

template <int kGroup>
__device__ __forceinline__ U128 gneg(U128 a) {
  if constexpr (kGroup == SUFHIP_GROUP_XOR) {
    return a;
  } else {
    uint64_t lo = 0 - a.lo;
    uint64_t hi = ~a.hi + (lo == 0 ? 1 : 0);
    return U128{lo, hi & kMsbClear};
  }
}

// Per-level correction word fields needed by the bit modes:
// s_cw (16 bytes), v_cw byte 0, and the t byte (tl << 1 | tr).
struct CwBit {
  uint32_t s[4];
  uint32_t v0;
  uint32_t tb;
};

struct CwFull {
  uint32_t s[4];
  uint32_t v[4];
  uint32_t tb;
};


// Reads 16 bytes at p.  When p + 16 is the end of the key (`more` false) and
// p is not 4-byte aligned, the last sh bytes come from byte loads so that no
// word past the key is touched.
__device__ __forceinline__ void load16_bytes(const uint8_t* p, bool more, uint32_t (&w)[4]) {
  const uintptr_t a = reinterpret_cast<uintptr_t>(p);
  const uint32_t* q = reinterpret_cast<const uint32_t*>(a & ~uintptr_t(3));
  const uint32_t sh = uint32_t(a & 3);
  uint32_t r0 = q[0], r1 = q[1], r2 = q[2], r3 = q[3];
  uint32_t r4 = 0;
  if (sh != 0) {
    if (more) {
      r4 = q[4];
    } else {
      const uint8_t* tail = reinterpret_cast<const uint8_t*>(q + 4);
      for (uint32_t k = 0; k < sh; ++k) r4 |= uint32_t(tail[k]) << (8 * k);
    }
  }
  w[0] = __builtin_amdgcn_alignbyte(r1, r0, sh);
  w[1] = __builtin_amdgcn_alignbyte(r2, r1, sh);
  w[2] = __builtin_amdgcn_alignbyte(r3, r2, sh);
  w[3] = __builtin_amdgcn_alignbyte(r4, r3, sh);
}

// ---------------------------------------------------------------------------
// Bit-mode walk (share byte 0 & 1) with the round keys in scalar registers.
//
// At level i every lane needs K_{2 x_i} (next seed) and K_{2 x_i + 1} (value
// block), x_i being its own input bit.  With m = -x_i (all ones or zero) they
// are K_0 ^ (m & (K_0 ^ K_2)) and K_1 ^ (m & (K_1 ^ K_3)): the four uniform
// words of each pair come from the kernel argument through the scalar unit,
// and the per-lane choice is one 3-input bit operation per key word.  Reading
// the chosen keys from LDS instead costs 20 ds_read_b128 per level (about 4
// LDS clocks each) on the pipe that bounds the walk, and 80 VGPRs.
//
// DcfKeySel row r: K_0[r], (K_0 ^ K_2)[r], K_1[r], (K_1 ^ K_3)[r].
struct DcfKeySel {
  uint32_t w[11][16];
};

void fill_key_sel(const Prg4& p, DcfKeySel* k) {
  for (int r = 0; r < 11; ++r)
    for (int j = 0; j < 4; ++j) {
      k->w[r][j] = p.rk[0][4 * r + j];
      k->w[r][4 + j] = p.rk[0][4 * r + j] ^ p.rk[2][4 * r + j];
      k->w[r][8 + j] = p.rk[1][4 * r + j];
      k->w[r][12 + j] = p.rk[1][4 * r + j] ^ p.rk[3][4 * r + j];
    }
}

// A DcfKeySel inside the kernel's by-value argument, addressed through the
// constant (kernel-argument) address space so that its loads are scalar.
typedef const __attribute__((address_space(4))) uint32_t* KeySelPtr;

__device__ __forceinline__ KeySelPtr kernarg_key_sel(size_t field) {
  return (KeySelPtr)((const __attribute__((address_space(4))) uint8_t*)
                         __builtin_amdgcn_kernarg_segment_ptr() + field);
}

#define SUFHIP_BITOP3(a, b, c, f) __builtin_amdgcn_bitop3_b32((a), (b), (c), (f))
// x ^ (m & d) as one v_bitop3 (truth table over src0 = 0xf0, src1 = 0xcc,
// src2 = 0xaa).
__device__ __forceinline__ uint32_t xor_and(uint32_t x, uint32_t m, uint32_t d) {
  return SUFHIP_BITOP3(x, m, d, 0x78);
}

__device__ __forceinline__ uint32_t lds_word(const uint32_t* lds, uint32_t byte_addr) {
  return *reinterpret_cast<const uint32_t*>(reinterpret_cast<const uint8_t*>(lds) + byte_addr);
}

// One middle round of the seed block A and of columns [0, kB) of the value
// block B, in three groups: every table address, then every table read with
// the round's key loads, then the combines.  The scheduling barriers keep the
// compiler from interleaving reads with their uses (each read's latency
// would then be paid in turn).
template <int kB>
__device__ __forceinline__ void key_sel_round(const AesLds4& aes, KeySelPtr q, uint32_t m,
                                              uint32_t (&A)[4], uint32_t (&B)[4]) {
  constexpr int kN = 16 + 4 * kB;
  uint32_t ad[kN];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      ad[4 * c + j] = __builtin_amdgcn_perm(A[(c + j) & 3], aes.base[j], AesLds4::sel(j));
      if (c < kB)
        ad[16 + 4 * c + j] = __builtin_amdgcn_perm(B[(c + j) & 3], aes.base[j], AesLds4::sel(j));
    }
  __builtin_amdgcn_sched_barrier(0);
  uint32_t tv[kN];
#pragma unroll
  for (int n = 0; n < kN; ++n) tv[n] = lds_word(aes.lds, ad[n]);
  uint32_t kq[16];
#pragma unroll
  for (int n = 0; n < 8; ++n) kq[n] = q[n];
#pragma unroll
  for (int c = 0; c < kB; ++c) {
    kq[8 + c] = q[8 + c];
    kq[12 + c] = q[12 + c];
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int c = 0; c < 4; ++c)
    A[c] = xor_and(SUFHIP_BITOP3(SUFHIP_BITOP3(tv[4 * c], tv[4 * c + 1], tv[4 * c + 2], 0x96),
                                 tv[4 * c + 3], kq[c], 0x96),
                   m, kq[4 + c]);
#pragma unroll
  for (int c = 0; c < kB; ++c)
    B[c] = xor_and(SUFHIP_BITOP3(SUFHIP_BITOP3(tv[16 + 4 * c], tv[17 + 4 * c], tv[18 + 4 * c], 0x96),
                                 tv[19 + 4 * c], kq[8 + c], 0x96),
                   m, kq[12 + c]);
}

// The aligned words of a 33-byte correction-word record that hold s_cw,
// byte 0 of v_cw and the t byte (words 0..4 and 8), read with global loads:
// a flat load also counts on the LDS wait counter, so every LDS wait of the
// level would wait for it too.
struct CwRaw {
  uint32_t r[6];
  uint32_t sh;
};

typedef const __attribute__((address_space(1))) uint32_t* GlobalWords;

__device__ __forceinline__ CwRaw load_cw_raw(const uint8_t* p) {
  const uintptr_t a = reinterpret_cast<uintptr_t>(p);
  GlobalWords q = (GlobalWords)(a & ~uintptr_t(3));
  CwRaw c;
  c.r[0] = q[0];
  c.r[1] = q[1];
  c.r[2] = q[2];
  c.r[3] = q[3];
  c.r[4] = q[4];
  c.r[5] = q[8];
  c.sh = uint32_t(a & 3);
  return c;
}

__device__ __forceinline__ CwBit decode_cw(const CwRaw& w) {
  CwBit c;
  c.s[0] = __builtin_amdgcn_alignbyte(w.r[1], w.r[0], w.sh);
  c.s[1] = __builtin_amdgcn_alignbyte(w.r[2], w.r[1], w.sh);
  c.s[2] = __builtin_amdgcn_alignbyte(w.r[3], w.r[2], w.sh);
  c.s[3] = __builtin_amdgcn_alignbyte(w.r[4], w.r[3], w.sh);
  c.v0 = (w.r[4] >> (8 * w.sh)) & 0xffu;
  c.tb = (w.r[5] >> (8 * w.sh)) & 0xffu;
  return c;
}

// Bit-mode walk of one chunk: returns share byte 0 & 1.  The seed block is
// AES_{K_{2 x_i}}(s) ^ s in full; of the value block only byte 0 is formed
// (round 9 column 0, then one final S-box byte).
// walk_bit_from continues at level `from` with seed s, control bit t and
// accumulated bit v.
__device__ __forceinline__ uint32_t walk_bit_from(const AesLds4& aes, KeySelPtr keys,
                                                  const uint8_t* chunk, int in_bits, int from,
                                                  uint64_t x, uint32_t (&s)[4], uint32_t t,
                                                  uint32_t v) {
  const uint8_t* cw = chunk + 16 + 33 * from;
  for (int i = from; i < in_bits; ++i, cw += 33) {
    const uint32_t xi = uint32_t(x >> (in_bits - 1 - i)) & 1u;
    const uint32_t m = 0u - xi;
    const CwRaw cr = load_cw_raw(cw);
    // An opaque copy of the key pointer per level: the compiler would
    // otherwise hoist all 176 key words out of the level loop into scalar
    // registers it does not have.
    KeySelPtr k = keys;
    asm volatile("" : "+s"(k));
    uint32_t A[4], B[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      A[j] = xor_and(s[j], m, k[4 + j]) ^ k[j];
      B[j] = xor_and(s[j], m, k[12 + j]) ^ k[8 + j];
    }
#pragma unroll
    for (int r = 1; r < 9; ++r) key_sel_round<4>(aes, k + 16 * r, m, A, B);
    key_sel_round<1>(aes, k + 16 * 9, m, A, B);
    // Final round of the seed block: S(x) is byte 0 of T3[x], bytes 1 and 2
    // of T0[x] and byte 3 of T1[x]; byte 0 of the value block from T3.
    uint32_t ad[17];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      ad[4 * c + 0] = __builtin_amdgcn_perm(A[c], aes.base[3], AesLds4::sel(0));
      ad[4 * c + 1] = __builtin_amdgcn_perm(A[(c + 1) & 3], aes.base[0], AesLds4::sel(1));
      ad[4 * c + 2] = __builtin_amdgcn_perm(A[(c + 2) & 3], aes.base[0], AesLds4::sel(2));
      ad[4 * c + 3] = __builtin_amdgcn_perm(A[(c + 3) & 3], aes.base[1], AesLds4::sel(3));
    }
    ad[16] = __builtin_amdgcn_perm(B[0], aes.base[3], AesLds4::sel(0));
    __builtin_amdgcn_sched_barrier(0);
    uint32_t tv[17];
#pragma unroll
    for (int n = 0; n < 17; ++n) tv[n] = lds_word(aes.lds, ad[n]);
    const KeySelPtr q = k + 160;
    uint32_t kq[10];
#pragma unroll
    for (int n = 0; n < 8; ++n) kq[n] = q[n];
    kq[8] = q[8];
    kq[9] = q[12];
    __builtin_amdgcn_sched_barrier(0);
    uint32_t o[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const uint32_t lo = __builtin_amdgcn_perm(tv[4 * c + 1], tv[4 * c], 0x0c0c0500u);
      const uint32_t hi = __builtin_amdgcn_perm(tv[4 * c + 3], tv[4 * c + 2], 0x07020c0cu);
      // ((lo | hi) ^ s) ^ K_sel: the Matyas-Meyer-Oseas output of the seed block.
      o[c] = xor_and(SUFHIP_BITOP3(lo, hi, s[c], 0x56) ^ kq[c], m, kq[4 + c]);
    }
    const uint32_t vb = xor_and(tv[16] ^ s[0] ^ kq[8], m, kq[9]) & 1u;
    const CwBit c = decode_cw(cr);
    uint32_t tn = o[3] >> 31;
    o[3] &= 0x7fffffffu;
    const uint32_t tmask = 0u - t;
#pragma unroll
    for (int j = 0; j < 4; ++j) s[j] = o[j] ^ (c.s[j] & tmask);
    tn ^= ((xi ? c.tb : (c.tb >> 1)) & 1u) & t;
    v ^= vb ^ (c.v0 & t & 1u);
    t = tn;
  }
  uint32_t np1[4];
  load16_bytes(cw, false, np1);
  return (v ^ s[0] ^ (np1[0] & t)) & 1u;
}

__device__ __forceinline__ uint32_t walk_bit(const AesLds4& aes, KeySelPtr keys,
                                             const uint8_t* chunk, int in_bits, uint64_t x,
                                             uint32_t party) {
  uint32_t seed[4];
  load16_bytes(chunk, true, seed);
  uint32_t s[4] = {seed[0], seed[1], seed[2], seed[3] & 0x7fffffffu};
  return walk_bit_from(aes, keys, chunk, in_bits, 0, x, s, party, 0);
}

// The aligned words 0..8 around a 33-byte correction-word record (s_cw,
// v_cw, the t byte), read with global loads at the start of a level and
// decoded after its AES (as CwRaw for the bit walk).
struct CwRawFull {
  uint32_t r[9];
  uint32_t sh;
};

__device__ __forceinline__ CwRawFull load_cw_raw_full(const uint8_t* p) {
  const uintptr_t a = reinterpret_cast<uintptr_t>(p);
  GlobalWords q = (GlobalWords)(a & ~uintptr_t(3));
  CwRawFull c;
#pragma unroll
  for (int j = 0; j < 9; ++j) c.r[j] = q[j];
  c.sh = uint32_t(a & 3);
  return c;
}

__device__ __forceinline__ CwFull decode_cw_full(const CwRawFull& w) {
  CwFull c;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    c.s[j] = __builtin_amdgcn_alignbyte(w.r[j + 1], w.r[j], w.sh);
    c.v[j] = __builtin_amdgcn_alignbyte(w.r[j + 5], w.r[j + 4], w.sh);
  }
  c.tb = (w.r[8] >> (8 * w.sh)) & 0xffu;
  return c;
}

// Both blocks of a level, as walk_bit forms them (round keys chosen per lane
// from scalar registers, grouped rounds): o = AES_{K_{2b}}(s) ^ s and the
// first kW words (2 or 4) of AES_{K_{2b+1}}(s) ^ s in ob, m = -b.
template <int kW>
__device__ __forceinline__ void sel_blocks(const AesLds4& aes, KeySelPtr keys, uint32_t m,
                                           const uint32_t (&s)[4], uint32_t (&o)[4],
                                           uint32_t (&ob)[kW]) {
  KeySelPtr k = keys;
  asm volatile("" : "+s"(k));
  uint32_t A[4], B[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    A[j] = xor_and(s[j], m, k[4 + j]) ^ k[j];
    B[j] = xor_and(s[j], m, k[12 + j]) ^ k[8 + j];
  }
#pragma unroll
  for (int r = 1; r < 10; ++r) key_sel_round<4>(aes, k + 16 * r, m, A, B);
  // Final round of both blocks: S(x) is byte 0 of T3[x], bytes 1 and 2 of
  // T0[x] and byte 3 of T1[x].
  constexpr int kN = 16 + 4 * kW;
  uint32_t ad[kN];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    ad[4 * c + 0] = __builtin_amdgcn_perm(A[c], aes.base[3], AesLds4::sel(0));
    ad[4 * c + 1] = __builtin_amdgcn_perm(A[(c + 1) & 3], aes.base[0], AesLds4::sel(1));
    ad[4 * c + 2] = __builtin_amdgcn_perm(A[(c + 2) & 3], aes.base[0], AesLds4::sel(2));
    ad[4 * c + 3] = __builtin_amdgcn_perm(A[(c + 3) & 3], aes.base[1], AesLds4::sel(3));
    if (c < kW) {
      ad[16 + 4 * c + 0] = __builtin_amdgcn_perm(B[c], aes.base[3], AesLds4::sel(0));
      ad[16 + 4 * c + 1] = __builtin_amdgcn_perm(B[(c + 1) & 3], aes.base[0], AesLds4::sel(1));
      ad[16 + 4 * c + 2] = __builtin_amdgcn_perm(B[(c + 2) & 3], aes.base[0], AesLds4::sel(2));
      ad[16 + 4 * c + 3] = __builtin_amdgcn_perm(B[(c + 3) & 3], aes.base[1], AesLds4::sel(3));
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  uint32_t tv[kN];
#pragma unroll
  for (int n = 0; n < kN; ++n) tv[n] = lds_word(aes.lds, ad[n]);
  const KeySelPtr q = k + 160;
  uint32_t kq[16];
#pragma unroll
  for (int n = 0; n < 16; ++n) kq[n] = q[n];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const uint32_t lo = __builtin_amdgcn_perm(tv[4 * c + 1], tv[4 * c], 0x0c0c0500u);
    const uint32_t hi = __builtin_amdgcn_perm(tv[4 * c + 3], tv[4 * c + 2], 0x07020c0cu);
    o[c] = xor_and(SUFHIP_BITOP3(lo, hi, s[c], 0x56) ^ kq[c], m, kq[4 + c]);
    if (c < kW) {
      const uint32_t lb = __builtin_amdgcn_perm(tv[16 + 4 * c + 1], tv[16 + 4 * c], 0x0c0c0500u);
      const uint32_t hb =
          __builtin_amdgcn_perm(tv[16 + 4 * c + 3], tv[16 + 4 * c + 2], 0x07020c0cu);
      ob[c < kW ? c : 0] = xor_and(SUFHIP_BITOP3(lb, hb, s[c], 0x56) ^ kq[8 + c], m, kq[12 + c]);
    }
  }
}

// Full-block walk of one chunk (any group): returns the 16-byte share.
template <int kGroup>
__device__ __forceinline__ U128 walk_full(const AesLds4& aes, KeySelPtr keys, const uint8_t* chunk,
                                          int in_bits, uint64_t x, uint32_t party,
                                          bool more_after) {
  uint32_t seed[4];
  load16_bytes(chunk, true, seed);
  uint32_t s[4] = {seed[0], seed[1], seed[2], seed[3] & 0x7fffffffu};
  uint32_t t = party;
  U128 v{0, 0};
  const uint8_t* cw = chunk + 16;
  for (int i = 0; i < in_bits; ++i, cw += 33) {
    const uint32_t xi = uint32_t(x >> (in_bits - 1 - i)) & 1u;
    const CwRawFull cr = load_cw_raw_full(cw);
    uint32_t o[4], ob[4];
    sel_blocks<4>(aes, keys, 0u - xi, s, o, ob);
    const CwFull c = decode_cw_full(cr);
    U128 vd = mk(ob[0], ob[1], ob[2], ob[3] & 0x7fffffffu);
    uint32_t tn = o[3] >> 31;
    o[3] &= 0x7fffffffu;
    if (t) {
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] ^= c.s[j];
      tn ^= (xi ? c.tb : (c.tb >> 1)) & 1u;
      vd = gadd<kGroup>(vd, mk(c.v[0], c.v[1], c.v[2], c.v[3]));
    }
    if (party) vd = gneg<kGroup>(vd);
    v = gadd<kGroup>(v, vd);
#pragma unroll
    for (int j = 0; j < 4; ++j) s[j] = o[j];
    t = tn;
  }
  uint32_t np1[4];
  load16_bytes(cw, more_after, np1);
  U128 sv = mk(s[0], s[1], s[2], s[3]);
  if (t) sv = gadd<kGroup>(sv, mk(np1[0], np1[1], np1[2], np1[3]));
  if (party) sv = gneg<kGroup>(sv);
  return gadd<kGroup>(v, sv);
}

// Additive-group walk that keeps only the low 64 bits of the 16-byte
// value: + mod 2^127 and negation never carry from bit 63 upward into the
// low word, so the low 8 bytes of the share are exact.  Used for DCF keys
// with an 8-byte payload (SUF's AddU64 predicates).
struct Add64State {
  uint32_t s0, s1, s2, s3;  // seed, MSB cleared
  uint32_t t;
  uint64_t v;  // accumulated value, low 64 bits
};

// Correction word fields for the low-64 walk: s_cw, v_cw bytes 0..7, t byte.
struct CwAdd64 {
  uint32_t s[4];
  uint64_t v;
  uint32_t tb;
};

__device__ __forceinline__ CwAdd64 load_cw_add64(const uint8_t* p) {
  const uintptr_t a = reinterpret_cast<uintptr_t>(p);
  const uint32_t* q = reinterpret_cast<const uint32_t*>(a & ~uintptr_t(3));
  const uint32_t sh = uint32_t(a & 3);
  // Words 0..6 and 8 of the aligned window: bytes [0, 24) and byte 32 of
  // the 33-byte record (word 8 may reach into the next record or cw_np1,
  // both inside the key).
  const uint32_t r0 = q[0], r1 = q[1], r2 = q[2], r3 = q[3], r4 = q[4], r5 = q[5], r6 = q[6],
                 r8 = q[8];
  CwAdd64 c;
  c.s[0] = __builtin_amdgcn_alignbyte(r1, r0, sh);
  c.s[1] = __builtin_amdgcn_alignbyte(r2, r1, sh);
  c.s[2] = __builtin_amdgcn_alignbyte(r3, r2, sh);
  c.s[3] = __builtin_amdgcn_alignbyte(r4, r3, sh);
  c.v = uint64_t(__builtin_amdgcn_alignbyte(r5, r4, sh)) |
        uint64_t(__builtin_amdgcn_alignbyte(r6, r5, sh)) << 32;
  c.tb = (r8 >> (8 * sh)) & 0xffu;
  return c;
}

// State at the root of one chunk (chunk = key + 8: seed, CWs, cw_np1).
__device__ __forceinline__ Add64State add64_root(const uint8_t* chunk, uint32_t party) {
  uint32_t seed[4];
  load16_bytes(chunk, true, seed);
  return Add64State{seed[0], seed[1], seed[2], seed[3] & 0x7fffffffu, party, 0};
}

// Levels [from, to) of an in_bits-level walk at x (only bits in_bits-1-i used).
__device__ __forceinline__ void add64_walk(const DcfAes& aes, const uint4* rkl,
                                           const uint8_t* chunk, int in_bits, int from, int to,
                                           uint64_t x, uint32_t party, Add64State& st) {
  const uint8_t* cw = chunk + 16 + 33 * from;
  for (int i = from; i < to; ++i, cw += 33) {
    const uint32_t xi = uint32_t(x >> (in_bits - 1 - i)) & 1u;
    const CwAdd64 c = load_cw_add64(cw);
    const uint4* ks = rkl + 22 * xi;
    const uint4* kv = ks + 11;
    uint32_t a0 = st.s0, a1 = st.s1, a2 = st.s2, a3 = st.s3;
    uint32_t b0, b1;
    aes.encrypt(a0, a1, a2, a3, ks);
    aes.encrypt_lo2(st.s0, st.s1, st.s2, st.s3, kv, b0, b1);
    uint64_t vd = uint64_t(b0 ^ st.s0) | uint64_t(b1 ^ st.s1) << 32;
    a0 ^= st.s0;
    a1 ^= st.s1;
    a2 ^= st.s2;
    a3 ^= st.s3;
    uint32_t tn = a3 >> 31;
    a3 &= 0x7fffffffu;
    if (st.t) {
      a0 ^= c.s[0];
      a1 ^= c.s[1];
      a2 ^= c.s[2];
      a3 ^= c.s[3];
      tn ^= (xi ? c.tb : (c.tb >> 1)) & 1u;
      vd += c.v;
    }
    st.v += party ? 0 - vd : vd;
    st.s0 = a0;
    st.s1 = a1;
    st.s2 = a2;
    st.s3 = a3;
    st.t = tn;
  }
}

// add64_walk with the round keys in scalar registers (sel_blocks), for 1024
// lanes per CU.
__device__ __forceinline__ void walk_low64(const DcfAes& aes, KeySelPtr keys,
                                           const uint8_t* chunk, int in_bits, int from, int to,
                                           uint64_t x, uint32_t party, Add64State& st) {
  const uint8_t* cw = chunk + 16 + 33 * from;
  for (int i = from; i < to; ++i, cw += 33) {
    const uint32_t xi = uint32_t(x >> (in_bits - 1 - i)) & 1u;
    const CwRawFull cr = load_cw_raw_full(cw);
    const uint32_t s[4] = {st.s0, st.s1, st.s2, st.s3};
    uint32_t o[4], ob[2];
    sel_blocks<2>(aes, keys, 0u - xi, s, o, ob);
    const CwFull c = decode_cw_full(cr);
    uint64_t vd = uint64_t(ob[0]) | uint64_t(ob[1]) << 32;
    uint32_t tn = o[3] >> 31;
    o[3] &= 0x7fffffffu;
    if (st.t) {
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] ^= c.s[j];
      tn ^= (xi ? c.tb : (c.tb >> 1)) & 1u;
      vd += uint64_t(c.v[0]) | uint64_t(c.v[1]) << 32;
    }
    st.v += party ? 0 - vd : vd;
    st.s0 = o[0];
    st.s1 = o[1];
    st.s2 = o[2];
    st.s3 = o[3];
    st.t = tn;
  }
}

// Share after the last level: v + (-1)^party (s + t * cw_np1), low 64 bits.
__device__ __forceinline__ uint64_t add64_finish(const uint8_t* chunk, int in_bits,
                                                 uint32_t party, const Add64State& st) {
  uint32_t np1[4];
  load16_bytes(chunk + 16 + 33 * in_bits, false, np1);
  uint64_t s = uint64_t(st.s0) | uint64_t(st.s1) << 32;
  if (st.t) s += uint64_t(np1[0]) | uint64_t(np1[1]) << 32;
  return st.v + (party ? 0 - s : s);
}

// Stages the replicated tables in LDS (the bit-mode walk's setup).
#define SUFHIP_DCF_TABLE_SETUP()                                   \
  __shared__ __align__(16) uint32_t tabs[DcfAes::kWords];          \
  __shared__ uint32_t tstage[256];                                 \
  DcfAes::fill(tabs, tstage, kTDev.v);                             \
  __syncthreads();                                                 \
  const DcfAes aes = DcfAes::make(tabs)

// Stages the replicated tables and the K_0..K_3 round keys in LDS.
#define SUFHIP_DCF_LDS_SETUP(PRG)                                  \
  __shared__ __align__(16) uint32_t tabs[DcfAes::kWords];          \
  __shared__ uint32_t tstage[256];                                 \
  __shared__ uint4 rkl[4 * 11];                                    \
  DcfAes::fill(tabs, tstage, kTDev.v);                             \
  fill_round_keys(rkl, (PRG).rk, 4);                               \
  __syncthreads();                                                 \
  const DcfAes aes = DcfAes::make(tabs)

// K_0..K_3 expanded (FIPS-197 word order).
void fill_prg4(const uint8_t* state, Prg4* p) {
  for (int j = 0; j < 4; ++j) {
    aes128_expand_words(state + 16 * j, p->rk[j]);
  }
}

int cu_count(int* cus) {
  int dev = 0;
  SUFHIP_CHECK(hipGetDevice(&dev), "hipGetDevice");
  SUFHIP_CHECK(hipDeviceGetAttribute(cus, hipDeviceAttributeMultiprocessorCount, dev),
               "hipDeviceGetAttribute(CU count)");
  return SUFHIP_OK;
}

}  // namespace
}  // namespace sufhip
