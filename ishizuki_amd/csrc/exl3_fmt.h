// EXL3 trellis tiles as the gfx950 kernels read them: where a weight's state lies in its tile's bit
// ring, and the codebook images (EXL3Tensor, Sources/IshizukiKit/Core/EXL3.swift:9-77, 136-147).
#pragma once
#include "common.h"

namespace ishz {

// exl3_decode (EXL3.swift:136-147): 3INST / MCG / MUL1 codebooks, fp16 single rounding.
DEV _Float16 exl3_decode(uint32_t s, int cb) {
  if (cb == 2) {
    const uint32_t x = s * 0x83DCD12Du;
    const uint32_t p = (x & 0x00ff00ffu) + ((x >> 8) & 0x00ff00ffu);
    const _Float16 h = __builtin_bit_cast(_Float16, (uint16_t)((p & 0xffffu) + (p >> 16) + 0x6400u));
    return __builtin_fmaf16(h, __builtin_bit_cast(_Float16, (uint16_t)0x1eee),
                            __builtin_bit_cast(_Float16, (uint16_t)0xc931));
  }
  uint32_t x = cb == 1 ? s * 0xCBAC1FEDu : s * 89226354u + 64248484u;
  x = (x & 0x8fff8fffu) ^ 0x3b603b60u;
  return __builtin_bit_cast(_Float16, (uint16_t)x) + __builtin_bit_cast(_Float16, (uint16_t)(x >> 16));
}

// Where the states lie in a tile's bit ring. At an integer rate of KA bits per weight, position p
// consumes KA bits and its state ends at ring bit KA (p + 1). At a half rate (KA + 1/2 bits) an
// even/odd pair consumes 2 KA + 1 bits, the even position KA of them and the odd one KA + 1. A
// state is the 16 ring bits ending there, read MSB first (bit 0 is the top bit of word 0), so it
// reaches back into the bits of earlier positions and wraps around the ring.
template <int KA, bool HALF>
struct Trellis {
  static constexpr int RING = HALF ? 128 * (2 * KA + 1) : 256 * KA;  // bits per 16x16 tile
  static constexpr int WORDS = RING / 32;
  static __host__ __device__ constexpr int bit_end(int p) {
    return HALF ? (p / 2) * (2 * KA + 1) + KA + (p % 2) * (KA + 1) : (p + 1) * KA;
  }
  // First ring bit of position p's state.
  static DEV int first_bit(int p) { return (bit_end(p) + RING - 16) % RING; }
  // Start of the state of position p0 + i relative to that of p0 (p0 even).
  static constexpr int offset(int i) { return bit_end(i) - bit_end(0); }
  // The 16-bit state starting at ring bit b: the 32 bits from b are one funnel shift of the word
  // holding b and the next word (b on a word boundary: that word alone); the state is the top half.
  static DEV uint32_t state(const uint32_t *tile, int b) {
    const int w = b >> 5, o = b & 31;
    const uint32_t hi = tile[w];
    const uint32_t bits32 = o ? __builtin_amdgcn_alignbit(hi, tile[(w + 1) % WORDS], 32 - o) : hi;
    return bits32 >> 16;
  }
  // The four weights at positions p0 .. p0 + 3, as two packed fp16 pairs.
  static DEV u2 decode4(const uint32_t *tile, int p0, int cb) {
    uint32_t h[4];
#pragma unroll
    for (int i = 0; i < 4; i++)
      h[i] = __builtin_bit_cast(uint16_t, exl3_decode(state(tile, (first_bit(p0) + offset(i)) % RING), cb));
    return u2{h[0] | h[1] << 16, h[2] | h[3] << 16};
  }
};

// Rates whose four lane states span at most 32 bits: a lane's window is one funnel shift of two
// tile words, each state one bit-field extract.
template <int KA, bool HALF>
struct Trellis32 {
  using TR = Trellis<KA, HALF>;
  static constexpr bool FITS = TR::offset(3) <= 16;  // the four states within 32 bits
  // The lane's 32-bit window (from the first bit of p0's state): words ja, jb funnel-shifted by amt.
  struct Win {
    int ja, jb, amt;
  };
  static DEV Win window(int p0) {
    const int b = TR::first_bit(p0), w = b >> 5, o = b & 31;
    return o ? Win{w, (w + 1) % TR::WORDS, 32 - o} : Win{w, w, 0};
  }
  // Bit-field offset of state i inside the window.
  static constexpr int field(int i) { return 16 - TR::offset(i); }
};

// Codebook images of two states, packed as fp16 (a in the low half): exl3_decode, pairwise.
template <int CB>
DEV uint32_t exl3_decode2(uint32_t sa, uint32_t sb) {
  if constexpr (CB == 2) {
    auto p = [](uint32_t s) {
      const uint32_t x = s * 0x83DCD12Du;
      const uint32_t q = (x & 0x00ff00ffu) + ((x >> 8) & 0x00ff00ffu);
      return ((q & 0xffffu) + (q >> 16) + 0x6400u) & 0xffffu;
    };
    const h2 h = as_h2(p(sa) | p(sb) << 16);
    const h2 m = as_h2(0x1eee1eeeu), c = as_h2(0xc931c931u);
    return __builtin_bit_cast(uint32_t, (h2)__builtin_elementwise_fma(h, m, c));
  } else {
    auto x = [](uint32_t s) {
      const uint32_t v = CB == 1 ? s * 0xCBAC1FEDu : s * 89226354u + 64248484u;
      return (v & 0x8fff8fffu) ^ 0x3b603b60u;
    };
    const uint32_t xa = x(sa), xb = x(sb);
    const uint32_t lo = __builtin_amdgcn_perm(xb, xa, 0x05040100u), hi = __builtin_amdgcn_perm(xb, xa, 0x07060302u);
    return __builtin_bit_cast(uint32_t, as_h2(lo) + as_h2(hi));
  }
}

// 3INST / MCG image of one state as the two fp16 halves whose sum is the weight (exl3_decode
// before its final add). The M = 1 matvec multiplies them by (x, x) as two MFMA k-entries: the
// halves meet x in fp32, so the weight's fp16 rounding of their sum is skipped (a difference of
// at most half an fp16 ulp per weight, inside the matmul tolerance; dequantization keeps the
// exact decode).
template <int CB>
DEV uint32_t exl3_halves(uint32_t s) {
  static_assert(CB != 2, "MUL1 decodes to one fp16 directly");
  const uint32_t v = CB == 1 ? s * 0xCBAC1FEDu : s * 89226354u + 64248484u;
  return (v & 0x8fff8fffu) ^ 0x3b603b60u;
}
DEV uint32_t dup_lo(uint32_t p) { return __builtin_amdgcn_perm(p, p, 0x01000100u); }
DEV uint32_t dup_hi(uint32_t p) { return __builtin_amdgcn_perm(p, p, 0x03020302u); }

}  // namespace ishz
