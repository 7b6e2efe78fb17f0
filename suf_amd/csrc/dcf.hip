// myl7/fss v0.7.1 DCF (lambda = 16, AES-128-MMO PRG) on CDNA4: batched key
// generation and evaluation over SUF's myl7 adapter key blobs.
//
// Evaluation (third_party/myl7_fss/src/dcf.c:146-193) walks the tree from
// bit in_bits-1 down to bit 0.  At each level the reference expands the seed
// into four blocks (sl, vl, sr, vr) with four AES calls, then keeps only the
// side selected by the input bit.  Here each lane computes just the two
// blocks on that side -- AES_{K_{2b}} for the next seed and AES_{K_{2b+1}}
// for the value block, b = x_i -- which halves the AES work without changing
// any output byte.  When only share byte 0 bit 0 is needed (the
// eval_dcf_many_u64 contract, include/proto/myl7_fss_backend.hpp:88-99), the
// value block is reduced to its first byte: bit 0 of a sum or XOR depends
// only on bit 0 of the terms, and bit 0 of -v equals bit 0 of v, so this
// holds for both output groups.
//
// Batches of more than 384 walks per CU: one walk per lane, a walk being one
// 16-byte chunk of one element's payload; each lane streams its own key front
// to back (33 bytes per level), so successive levels hit the same cache lines.
//
// The evaluation kernels run 1024 lanes per CU (four waves per SIMD): their
// walks keep the round keys in scalar registers and fit in the 128 VGPRs
// that allows, and the table lookups that bound them overlap better with
// more waves.
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstring>

#include "dcf_device.hpp"
#include "dcf_gen_device.hpp"
#include "dcf_quad_device.hpp"

namespace sufhip {
namespace {

struct DcfEvalArgs {
  const uint8_t* keys;
  const uint64_t* xs;
  void* out;
  size_t key_bytes;
  size_t n;
  int broadcast;
  int in_bits;
  int chunks;     // chunks to evaluate (1 for the bit modes)
  int out_bytes;  // bytes per element (OUT_BYTES)
  DcfKeySel key_sel;  // the round keys (scalar loads)
};

constexpr int kDcfBitBlock = 1024;

// First walk of this wave in the pass that starts at `pass`.  A full pass
// gives each workgroup 1024 neighbouring keys; the last one deals its walks
// out 64 at a time, so that what does not fill the chip spreads over every CU
// (100000 keys of 64 levels: 318 -> 184 us) instead of filling the first ones.
// Dealing the full passes out too made 2^20 keys 4% slower (the keys in flight
// on a CU then span the whole 2 GB).
__device__ __forceinline__ size_t wave_base(size_t pass, size_t n) {
  const size_t wave = threadIdx.x >> 6;
  return n - pass >= size_t(gridDim.x) * kDcfBitBlock
             ? pass + size_t(blockIdx.x) * kDcfBitBlock + wave * 64
             : pass + (size_t(blockIdx.x) + size_t(gridDim.x) * wave) * 64;
}

template <int kMode>
__global__ void __launch_bounds__(kDcfBitBlock) dcf_eval_bit_kernel(DcfEvalArgs a) {
  SUFHIP_DCF_TABLE_SETUP();
  const KeySelPtr keys = kernarg_key_sel(offsetof(DcfEvalArgs, key_sel));
  const size_t stride = size_t(gridDim.x) * kDcfBitBlock;
  for (size_t pass = 0; pass < a.n; pass += stride) {
    const size_t e = wave_base(pass, a.n) + (threadIdx.x & 63);
    uint32_t bit = 0;
    if (e < a.n) {
      const uint8_t* key = a.broadcast ? a.keys : a.keys + e * a.key_bytes;
      const uint32_t party = key[2] & 1u;
      uint64_t x = a.xs[e];
      if (a.in_bits < 64) x &= (uint64_t(1) << a.in_bits) - 1;
      bit = walk_bit(aes, keys, key + 8, a.in_bits, x, party);
    }
    if constexpr (kMode == SUFHIP_DCF_OUT_BIT) {
      if (e < a.n) static_cast<uint8_t*>(a.out)[e] = uint8_t(bit);
    } else {
      // Waves cover 64 consecutive elements starting at a multiple of 64.
      const uint64_t word = __ballot(bit != 0);
      if ((threadIdx.x & 63) == 0 && e < a.n) static_cast<uint64_t*>(a.out)[e >> 6] = word;
    }
  }
}

// A lane that ran an element's chunks in turn left the chip to few elements of
// many chunks: 1562 of 64 chunks of 16 levels took 2431 us, 58 this way.
template <int kGroup>
__global__ void __launch_bounds__(kDcfBitBlock) dcf_eval_bytes_kernel(DcfEvalArgs a) {
  SUFHIP_DCF_TABLE_SETUP();
  const KeySelPtr keys = kernarg_key_sel(offsetof(DcfEvalArgs, key_sel));
  const size_t stride = size_t(gridDim.x) * kDcfBitBlock;
  const size_t chunk_bytes = 32 + 33 * size_t(a.in_bits);
  const size_t walks = a.n * size_t(a.chunks);
  for (size_t pass = 0; pass < walks; pass += stride) {
    const size_t w = wave_base(pass, walks) + (threadIdx.x & 63);
    if (w >= walks) continue;
    const size_t e = w / size_t(a.chunks);
    const int c = int(w - e * size_t(a.chunks));
    const uint8_t* key = a.broadcast ? a.keys : a.keys + e * a.key_bytes;
    uint64_t x = a.xs[e];
    if (a.in_bits < 64) x &= (uint64_t(1) << a.in_bits) - 1;
    const bool more = size_t(c + 1) * chunk_bytes + 8 < a.key_bytes;
    const U128 r = walk_full<kGroup>(aes, keys, key + 8 + size_t(c) * chunk_bytes, a.in_bits, x,
                                     key[2] & 1u, more);
    uint8_t* out = static_cast<uint8_t*>(a.out) + e * size_t(a.out_bytes) + 16 * c;
    const int take = a.out_bytes - 16 * c < 16 ? a.out_bytes - 16 * c : 16;
    for (int b = 0; b < take; ++b) out[b] = uint8_t((b < 8 ? r.lo : r.hi) >> (8 * (b & 7)));
  }
}

// Small batches: 8 lanes per walk (dcf_quad_device.hpp), a walk being one
// chunk of one element.  A wave takes 8 consecutive elements' walks; passes
// deal waves to the workgroups in turn.
template <int kMode>
__global__ void __launch_bounds__(kDcfBitBlock) dcf_eval_quad_bit_kernel(DcfEvalArgs a) {
  SUFHIP_DCF_TABLE_SETUP();
  const QuadKeys K = load_quad_keys(kernarg_key_sel(offsetof(DcfEvalArgs, key_sel)));
  // Packed outputs are whole words: the last word's missing elements are 0.
  const size_t octets = kMode == SUFHIP_DCF_OUT_BIT ? (a.n + 7) / 8 : (a.n + 63) / 64 * 8;
  const size_t stride = size_t(gridDim.x) * (kDcfBitBlock / 64);
  const uint32_t lane = threadIdx.x & 63u;
  for (size_t o = size_t(blockIdx.x) + size_t(gridDim.x) * (threadIdx.x >> 6); o < octets;
       o += stride) {
    const size_t e = 8 * o + (lane >> 3);
    const size_t ec = e < a.n ? e : a.n - 1;  // whole groups of 8 lanes keep walking
    const uint8_t* key = a.broadcast ? a.keys : a.keys + ec * a.key_bytes;
    const uint32_t party = key[2] & 1u;
    const uint64_t x = a.xs[ec];
    QuadState st = quad_root(key + 8, party);
    quad_walk<kQuadBit, SUFHIP_GROUP_XOR>(aes, K, key + 8, a.in_bits, 0, a.in_bits, x, party, st);
    const uint32_t bit = uint32_t(
        quad_finish<kQuadBit, SUFHIP_GROUP_XOR>(key + 8, a.in_bits, party, false, st).lo);
    const bool mine = (lane & 7u) == 4u && e < a.n;
    if constexpr (kMode == SUFHIP_DCF_OUT_BIT) {
      if (mine) static_cast<uint8_t*>(a.out)[e] = uint8_t(bit);
    } else {
      // Bit 8 g + 4 of the ballot is element g of the octet; the product
      // gathers the eight bits in its top byte.
      const uint64_t b = __ballot(mine && bit != 0) >> 4;
      if (lane == 0)
        static_cast<uint8_t*>(a.out)[o] = uint8_t((b * 0x0102040810204080ull) >> 56);
    }
  }
}

template <int kGroup>
__global__ void __launch_bounds__(kDcfBitBlock) dcf_eval_quad_bytes_kernel(DcfEvalArgs a) {
  SUFHIP_DCF_TABLE_SETUP();
  const QuadKeys K = load_quad_keys(kernarg_key_sel(offsetof(DcfEvalArgs, key_sel)));
  const size_t chunk_bytes = 32 + 33 * size_t(a.in_bits);
  const size_t walks = a.n * size_t(a.chunks);
  const size_t stride = size_t(gridDim.x) * (kDcfBitBlock / 8);
  for (size_t w = (size_t(blockIdx.x) + size_t(gridDim.x) * (threadIdx.x >> 6)) * 8 +
                  ((threadIdx.x & 63u) >> 3);
       w < walks; w += stride) {
    const size_t e = w / size_t(a.chunks);
    const int c = int(w - e * size_t(a.chunks));
    const uint8_t* key = a.broadcast ? a.keys : a.keys + e * a.key_bytes;
    const uint8_t* chunk = key + 8 + size_t(c) * chunk_bytes;
    const uint32_t party = key[2] & 1u;
    const uint64_t x = a.xs[e];
    const bool more = size_t(c + 1) * chunk_bytes + 8 < a.key_bytes;
    QuadState st = quad_root(chunk, party);
    quad_walk<kQuadFull, kGroup>(aes, K, chunk, a.in_bits, 0, a.in_bits, x, party, st);
    const U128 r = quad_finish<kQuadFull, kGroup>(chunk, a.in_bits, party, more, st);
    // Lane q of the value half writes word q of the chunk.
    const uint32_t l = threadIdx.x & 7u, q = l & 3u;
    const uint64_t half = q < 2 ? r.lo : r.hi;
    const uint32_t word = uint32_t(half >> (32 * (q & 1u)));
    uint8_t* out = static_cast<uint8_t*>(a.out) + e * size_t(a.out_bytes) + 16 * c + 4 * q;
    const int left = a.out_bytes - 16 * c - 4 * int(q);
    if (l >= 4)
      for (int b = 0; b < 4 && b < left; ++b) out[b] = uint8_t(word >> (8 * b));
  }
}

// Middling batches: 2 lanes per walk (dcf_quad_device.hpp).  The group only
// matters for the bits past bit 0.
template <int kMode, int kGroup>
__global__ void __launch_bounds__(kPairBlock) dcf_eval_pair_kernel(DcfEvalArgs a) {
  SUFHIP_DCF_TABLE_SETUP();
  const PairKeys K = load_pair_keys(kernarg_key_sel(offsetof(DcfEvalArgs, key_sel)));
  const size_t chunk_bytes = 32 + 33 * size_t(a.in_bits);
  const size_t walks = a.n * size_t(a.chunks);
  const size_t stride = size_t(gridDim.x) * (kPairBlock / 2);
  const uint32_t lane = threadIdx.x & 63u;
  // A wave takes 32 consecutive walks (a half word of packed bits); the last
  // packed word's missing elements are 0.
  const size_t end = kMode == SUFHIP_DCF_OUT_PACKED ? (walks + 63) / 64 * 64 : walks;
  for (size_t base = (size_t(blockIdx.x) + size_t(gridDim.x) * (threadIdx.x >> 6)) * 32;
       base < end; base += stride) {
    const size_t w = base + (lane >> 1);
    const bool in = w < walks;
    const size_t wc = in ? w : walks - 1;  // whole lane pairs keep walking
    const size_t e = wc / size_t(a.chunks);
    const int c = int(wc - e * size_t(a.chunks));
    const uint8_t* key = a.broadcast ? a.keys : a.keys + e * a.key_bytes;
    const uint8_t* chunk = key + 8 + size_t(c) * chunk_bytes;
    const bool more = size_t(c + 1) * chunk_bytes + 8 < a.key_bytes;
    const U128 r =
        pair_walk<kGroup>(aes, K, chunk, a.in_bits, a.xs[e], key[2] & 1u, more);
    const bool mine = in && (lane & 1u);
    if constexpr (kMode == SUFHIP_DCF_OUT_BIT) {
      if (mine) static_cast<uint8_t*>(a.out)[e] = uint8_t(r.lo & 1u);
    } else if constexpr (kMode == SUFHIP_DCF_OUT_PACKED) {
      // Bit 2 g + 1 of the ballot is element g: the odd bits, gathered.
      uint64_t b = (__ballot(mine && (r.lo & 1u)) >> 1) & 0x5555555555555555ull;
      b = (b | b >> 1) & 0x3333333333333333ull;
      b = (b | b >> 2) & 0x0f0f0f0f0f0f0f0full;
      b = (b | b >> 4) & 0x00ff00ff00ff00ffull;
      b = (b | b >> 8) & 0x0000ffff0000ffffull;
      b = (b | b >> 16) & 0xffffffffull;
      if (lane == 0) static_cast<uint32_t*>(a.out)[base >> 5] = uint32_t(b);
    } else {
      uint8_t* out = static_cast<uint8_t*>(a.out) + e * size_t(a.out_bytes) + 16 * c;
      const int take = a.out_bytes - 16 * c < 16 ? a.out_bytes - 16 * c : 16;
      if (mine)
        for (int b = 0; b < take; ++b) out[b] = uint8_t((b < 8 ? r.lo : r.hi) >> (8 * (b & 7)));
    }
  }
}

// ---------------------------------------------------------------- keygen --

struct DcfGenArgs {
  Prg4 prg;
  const uint64_t* alpha;
  const uint8_t* payload;
  const uint8_t* seeds;
  uint8_t* keys0;
  uint8_t* keys1;
  size_t key_bytes;
  size_t n;
  int payload_bcast;
  int payload_len;
  int in_bits;
  int chunks;
};

// Key generation: 8 lanes per chunk of a key pair (dcf_gen_device.hpp).  A
// wave takes 8 consecutive walks; passes deal waves to the workgroups in turn.
template <int kGroup>
__global__ void __launch_bounds__(kDcfBitBlock) dcf_gen_kernel(DcfGenArgs a) {
  SUFHIP_DCF_TABLE_SETUP();
  const GenKeys K = load_gen_keys(kernarg_key_sel(offsetof(DcfGenArgs, prg)));
  const size_t walks = a.n * size_t(a.chunks);
  const size_t stride = size_t(gridDim.x) * (kDcfBitBlock / 8);
  for (size_t w = (size_t(blockIdx.x) + size_t(gridDim.x) * (threadIdx.x >> 6)) * 8 +
                  ((threadIdx.x & 63u) >> 3);
       w < walks; w += stride) {
    const size_t e = w / size_t(a.chunks);
    const int c = int(w - e * size_t(a.chunks));
    const uint8_t* pay = a.payload_bcast ? a.payload : a.payload + e * size_t(a.payload_len);
    gen_chunk<kGroup>(aes, K, a.in_bits, a.chunks, a.payload_len, c, a.alpha[e], pay,
                      a.seeds + w * 32, a.keys0 + e * a.key_bytes, a.keys1 + e * a.key_bytes);
  }
}

constexpr size_t kMaxElems = size_t(1) << 38;

}  // namespace
}  // namespace sufhip

using namespace sufhip;

extern "C" {

size_t sufhip_dcf_key_bytes(int in_bits, int payload_len) {
  if (in_bits <= 0 || in_bits > 64 || payload_len <= 0) return 0;
  const size_t chunks = (size_t(payload_len) + 15) / 16;
  if (chunks > 255) return 0;
  return 8 + chunks * (32 + 33 * size_t(in_bits));
}

int sufhip_dcf_gen(int group, int in_bits, const uint8_t* prg_state, const uint64_t* d_alpha,
                   const uint8_t* d_payload, int payload_len, int payload_broadcast,
                   const uint8_t* d_seeds, size_t n, uint8_t* d_keys0, uint8_t* d_keys1,
                   void* stream) {
  SUFHIP_REQUIRE(group == SUFHIP_GROUP_XOR || group == SUFHIP_GROUP_ADD,
                 "sufhip_dcf_gen: unknown group");
  SUFHIP_REQUIRE(in_bits >= 1 && in_bits <= 64, "sufhip_dcf_gen: in_bits out of range");
  SUFHIP_REQUIRE(payload_len >= 1 && payload_len <= 255 * 16,
                 "sufhip_dcf_gen: payload_len out of range");
  if (n == 0) return SUFHIP_OK;
  SUFHIP_REQUIRE(n < kMaxElems, "sufhip_dcf_gen: n too large");
  SUFHIP_REQUIRE(prg_state && d_alpha && d_payload && d_seeds && d_keys0 && d_keys1,
                 "sufhip_dcf_gen: null pointer");
  DcfGenArgs a{};
  fill_prg4(prg_state, &a.prg);
  a.alpha = d_alpha;
  a.payload = d_payload;
  a.seeds = d_seeds;
  a.keys0 = d_keys0;
  a.keys1 = d_keys1;
  a.key_bytes = sufhip_dcf_key_bytes(in_bits, payload_len);
  a.n = n;
  a.payload_bcast = payload_broadcast ? 1 : 0;
  a.payload_len = payload_len;
  a.in_bits = in_bits;
  a.chunks = (payload_len + 15) / 16;
  int cus = 0;
  if (int rc = cu_count(&cus)) return rc;
  const size_t waves = (n * size_t(a.chunks) + 7) / 8;
  const dim3 grid(unsigned(waves < size_t(cus) ? waves : size_t(cus))), block(kDcfBitBlock);
  if (group == SUFHIP_GROUP_XOR)
    hipLaunchKernelGGL((dcf_gen_kernel<SUFHIP_GROUP_XOR>), grid, block, 0, as_stream(stream), a);
  else
    hipLaunchKernelGGL((dcf_gen_kernel<SUFHIP_GROUP_ADD>), grid, block, 0, as_stream(stream), a);
  return check_launch("dcf_gen_kernel");
}

int sufhip_dcf_eval(int group, int in_bits, int payload_len, const uint8_t* prg_state,
                    const uint8_t* d_keys, size_t key_bytes, int key_broadcast,
                    const uint64_t* d_xs, size_t n, int out_mode, int out_bytes, void* d_out,
                    void* stream) {
  SUFHIP_REQUIRE(group == SUFHIP_GROUP_XOR || group == SUFHIP_GROUP_ADD,
                 "sufhip_dcf_eval: unknown group");
  SUFHIP_REQUIRE(in_bits >= 1 && in_bits <= 64, "sufhip_dcf_eval: in_bits out of range");
  SUFHIP_REQUIRE(payload_len >= 1 && payload_len <= 255 * 16,
                 "sufhip_dcf_eval: payload_len out of range");
  SUFHIP_REQUIRE(key_bytes == sufhip_dcf_key_bytes(in_bits, payload_len),
                 "sufhip_dcf_eval: key_bytes does not match (in_bits, payload_len)");
  SUFHIP_REQUIRE(out_mode == SUFHIP_DCF_OUT_BIT || out_mode == SUFHIP_DCF_OUT_BYTES ||
                     out_mode == SUFHIP_DCF_OUT_PACKED,
                 "sufhip_dcf_eval: unknown out_mode");
  if (out_mode == SUFHIP_DCF_OUT_BYTES)
    SUFHIP_REQUIRE(out_bytes >= 1 && out_bytes <= payload_len,
                   "sufhip_dcf_eval: out_bytes must be in [1, payload_len]");
  if (n == 0) return SUFHIP_OK;
  SUFHIP_REQUIRE(n < kMaxElems, "sufhip_dcf_eval: n too large");
  SUFHIP_REQUIRE(prg_state && d_keys && d_xs && d_out, "sufhip_dcf_eval: null pointer");
  DcfEvalArgs a{};
  Prg4 prg;
  fill_prg4(prg_state, &prg);
  fill_key_sel(prg, &a.key_sel);
  a.keys = d_keys;
  a.xs = d_xs;
  a.out = d_out;
  a.key_bytes = key_bytes;
  a.n = n;
  a.broadcast = key_broadcast ? 1 : 0;
  a.in_bits = in_bits;
  a.chunks = 1;
  a.out_bytes = out_mode == SUFHIP_DCF_OUT_BYTES ? out_bytes : 1;
  hipStream_t s = as_stream(stream);
  if (out_mode == SUFHIP_DCF_OUT_BYTES) a.chunks = (out_bytes + 15) / 16;
  const size_t walks = n * size_t(a.chunks);
  int cus = 0;
  if (int rc = cu_count(&cus)) return rc;
  // Lanes per walk by walks per CU: 8 up to 160, 2 up to 384, then one; bits
  // take 8 lanes again from 256 to 320.  Fewer lanes do less exchange per
  // walk, more have a shorter serial chain; a full pass is 128, 256 or 1024
  // walks per CU, and just past one the next is as long.  Us on 256 CUs of
  // 64-level keys with 8 / 2 / 1 lanes, bits and 8-byte additive shares:
  //    40000 walks   88 /  93 / 151     93 / 100 / 168
  //    50021        108 / 100 / 152    125 / 107 / 172
  //    65536        132 / 101 / 154    152 / 108 / 184
  //    65600        138 / 151 / 168    161 / 160 / 186
  //    80000        150 / 156 / 174    174 / 168 / 191
  //    98304        196 / 158 / 173    226 / 168 / 186
  //   110000        215 / 192 / 185    249 / 205 / 206
  //   131072        271 / 200 / 187    302 / 211 / 210
  // 16-byte shares, payloads of 2 and 64 chunks (a walk is one chunk) and 16-
  // and 32-level keys give the same choice; XOR byte shares lie between the
  // columns (the choice costs them 4% at most).
  const size_t full = size_t(cus);
  const bool bytes = out_mode == SUFHIP_DCF_OUT_BYTES;
  const bool quad =
      walks <= 160 * full || (!bytes && walks > 256 * full && walks <= 320 * full);
  const bool pair = !quad && walks <= 384 * full;
  // Waves of 64, 8 or 32 walks, one workgroup per CU at most.
  const size_t per = quad ? 8 : (pair ? 32 : 64);
  const size_t waves = (walks + per - 1) / per;
  const dim3 grid(unsigned(waves < full ? waves : full));
  const dim3 block(unsigned(pair ? kPairBlock : kDcfBitBlock));
  const bool xor_group = group == SUFHIP_GROUP_XOR;
  SUFHIP_REQUIRE(out_mode != SUFHIP_DCF_OUT_PACKED || (reinterpret_cast<uintptr_t>(d_out) & 7) == 0,
                 "sufhip_dcf_eval: packed output must be 8-byte aligned");
#define SUFHIP_DCF_LAUNCH(...) hipLaunchKernelGGL((__VA_ARGS__), grid, block, 0, s, a)
  if (out_mode == SUFHIP_DCF_OUT_BIT) {
    if (quad)
      SUFHIP_DCF_LAUNCH(dcf_eval_quad_bit_kernel<SUFHIP_DCF_OUT_BIT>);
    else if (pair)
      SUFHIP_DCF_LAUNCH(dcf_eval_pair_kernel<SUFHIP_DCF_OUT_BIT, SUFHIP_GROUP_XOR>);
    else
      SUFHIP_DCF_LAUNCH(dcf_eval_bit_kernel<SUFHIP_DCF_OUT_BIT>);
  } else if (out_mode == SUFHIP_DCF_OUT_PACKED) {
    if (quad)
      SUFHIP_DCF_LAUNCH(dcf_eval_quad_bit_kernel<SUFHIP_DCF_OUT_PACKED>);
    else if (pair)
      SUFHIP_DCF_LAUNCH(dcf_eval_pair_kernel<SUFHIP_DCF_OUT_PACKED, SUFHIP_GROUP_XOR>);
    else
      SUFHIP_DCF_LAUNCH(dcf_eval_bit_kernel<SUFHIP_DCF_OUT_PACKED>);
  } else if (xor_group) {
    if (quad)
      SUFHIP_DCF_LAUNCH(dcf_eval_quad_bytes_kernel<SUFHIP_GROUP_XOR>);
    else if (pair)
      SUFHIP_DCF_LAUNCH(dcf_eval_pair_kernel<SUFHIP_DCF_OUT_BYTES, SUFHIP_GROUP_XOR>);
    else
      SUFHIP_DCF_LAUNCH(dcf_eval_bytes_kernel<SUFHIP_GROUP_XOR>);
  } else {
    if (quad)
      SUFHIP_DCF_LAUNCH(dcf_eval_quad_bytes_kernel<SUFHIP_GROUP_ADD>);
    else if (pair)
      SUFHIP_DCF_LAUNCH(dcf_eval_pair_kernel<SUFHIP_DCF_OUT_BYTES, SUFHIP_GROUP_ADD>);
    else
      SUFHIP_DCF_LAUNCH(dcf_eval_bytes_kernel<SUFHIP_GROUP_ADD>);
  }
#undef SUFHIP_DCF_LAUNCH
  return check_launch("dcf_eval kernel");
}

}  // extern "C"
