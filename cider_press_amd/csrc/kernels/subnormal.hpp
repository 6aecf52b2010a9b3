// Vote-free exact dequantization: packed values as f16 subnormals.
//
// A value q < 2^bits left at bit position p of a 16-bit half (p + bits <= 10)
// reads as the f16 subnormal q * 2^(p - 24): no conversion, the field is only
// masked.  v_fma_mix_f32 takes that f16 as one operand, so
//   fma(s * 2^(24 - p), q * 2^(p - 24), b) == fmaf(s, q, b)
// with one rounding.  s * 2^(24 - p) is exact in fp32 for every f16 scale and
// for every bf16 scale with a biased exponent below 231 (|s| < 2^104); larger
// ones (and Inf, NaN) overflow, so callers track sub_over() and use
// dequant_chunk for them.  Compared on an MI355X with fmaf(s, q, b) over all
// 65536 scale patterns of either type x 64 biases x q = 0..255: no
// difference outside that range.  Against the 1024 + q form of
// dequant_slice_nat this needs no group check up front and no b - 1024 s.
#pragma once

#include "common.hpp"

namespace cpq {
namespace dev {

// Largest scale pattern (sign cleared) that sub_chunk takes, plus one.
template <typename TT>
constexpr uint32_t kSubScaleLimit = Sig16<TT>::bf16 ? 231u << 7 : 0x10000u;

// Element E of a chunk's 8-element group (`bits` bytes): byte and bit of its
// first bit.
template <int BITS, int E>
constexpr int kByte = (BITS * E) >> 3;
template <int BITS, int E>
constexpr int kBit = (BITS * E) & 7;

// Bytes kByte(E), kByte(E) + 1 of a group at byte BASE, from the word pair
// (lo: word BASE/4, hi: the next), as two v_perm selector bytes; a byte the
// element does not reach is zero (selector 0x0c).
template <int BITS, int BASE, int E>
constexpr uint32_t sub_sel() {
  constexpr int b = (BASE & 3) + kByte<BITS, E>;
  constexpr uint32_t hi = kBit<BITS, E> + BITS > 8 ? (uint32_t)(b + 1) : 0x0cu;
  static_assert(b < 8 && (hi < 8 || hi == 0x0cu), "the element lies in one word pair");
  return (uint32_t)b | (hi << 8);
}

// Elements E0 (low half) and E1 (high half) of 8-element group G, each
// masked and SHR bits below its place in its first byte.
template <int BITS, int G, int E0, int E1, int SHR>
__device__ __forceinline__ uint32_t sub_pair(const uint32_t* w) {
  constexpr int base = BITS * G, wi = base >> 2;
  constexpr int s0 = kBit<BITS, E0> - SHR, s1 = kBit<BITS, E1> - SHR;
  static_assert(s0 >= 0 && s1 >= 0 && s0 + BITS <= 10 && s1 + BITS <= 10, "field inside a subnormal's 10 bits");
  constexpr uint32_t one = (1u << BITS) - 1u, mask = (one << s0) | (one << s1) << 16;
  constexpr uint32_t sel = sub_sel<BITS, base, E0>() | sub_sel<BITS, base, E1>() << 16;
  uint32_t t = __builtin_amdgcn_perm(w[wi + 1 < BITS ? wi + 1 : wi], w[wi], sel);
  if constexpr (SHR != 0) t >>= SHR;
  return t & mask;
}

// A chunk's scale (times 2^24) and bias, and the scale for a field SH bits up.
struct SubCst {
  float s24, b;
  template <int SH>
  __device__ __forceinline__ float s() const {
    return s24 * (1.0f / (float)(1 << SH));
  }
};

// 8-element group G (0..3) of a chunk as 4 packed T pairs in element order.
template <typename TT, int BITS, int G>
__device__ __forceinline__ u32x4 sub_group(const uint32_t* w, const SubCst& c) {
  if constexpr (BITS == 4) {
    const uint32_t v = w[G], v8 = v >> 8;
    const uint32_t p0 = v & 0x000F000Fu, p1 = v & 0x00F000F0u;    // (e0, e4), (e1, e5) 4 up
    const uint32_t p2 = v8 & 0x000F000Fu, p3 = v8 & 0x00F000F0u;  // (e2, e6), (e3, e7) 4 up
    const float s0 = c.s24, s4 = c.template s<4>();
    return u32x4{TT::pack2(fmaf(s0, f16lo(p0), c.b), fmaf(s4, f16lo(p1), c.b)),
                 TT::pack2(fmaf(s0, f16lo(p2), c.b), fmaf(s4, f16lo(p3), c.b)),
                 TT::pack2(fmaf(s0, f16hi(p0), c.b), fmaf(s4, f16hi(p1), c.b)),
                 TT::pack2(fmaf(s0, f16hi(p2), c.b), fmaf(s4, f16hi(p3), c.b))};
  } else if constexpr (BITS == 8) {
    u32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t p = __builtin_amdgcn_perm(0u, w[2 * G + (j >> 1)], (j & 1) ? 0x0c030c02u : 0x0c010c00u);
      o[j] = TT::pack2(fmaf(c.s24, f16lo(p), c.b), fmaf(c.s24, f16hi(p), c.b));
    }
    return o;
  } else if constexpr (BITS == 2) {
    // A group is one 16-bit half of a word: element e at its bit 2e.
    const uint32_t v = (G & 1) ? w[G >> 1] >> 16 : w[G >> 1];
    const uint32_t p01 = (v & 0x0003u) | ((v << 16) & 0x000C0000u);           // e0, e1 (2 up)
    const uint32_t p23 = (v & 0x0030u) | ((v << 16) & 0x00C00000u);           // e2 (4), e3 (6)
    const uint32_t u = v >> 8;
    const uint32_t p45 = (u & 0x0003u) | ((u << 16) & 0x000C0000u);
    const uint32_t p67 = (u & 0x0030u) | ((u << 16) & 0x00C00000u);
    const float s0 = c.s24, s2 = c.template s<2>(), s4 = c.template s<4>(), s6 = c.template s<6>();
    return u32x4{TT::pack2(fmaf(s0, f16lo(p01), c.b), fmaf(s2, f16hi(p01), c.b)),
                 TT::pack2(fmaf(s4, f16lo(p23), c.b), fmaf(s6, f16hi(p23), c.b)),
                 TT::pack2(fmaf(s0, f16lo(p45), c.b), fmaf(s2, f16hi(p45), c.b)),
                 TT::pack2(fmaf(s4, f16lo(p67), c.b), fmaf(s6, f16hi(p67), c.b))};
  } else if constexpr (BITS == 3) {
    const uint32_t p0 = sub_pair<3, G, 0, 1, 0>(w), p1 = sub_pair<3, G, 2, 3, 0>(w);
    const uint32_t p2 = sub_pair<3, G, 4, 5, 0>(w), p3 = sub_pair<3, G, 6, 7, 0>(w);
    return u32x4{TT::pack2(fmaf(c.template s<0>(), f16lo(p0), c.b), fmaf(c.template s<3>(), f16hi(p0), c.b)),
                 TT::pack2(fmaf(c.template s<6>(), f16lo(p1), c.b), fmaf(c.template s<1>(), f16hi(p1), c.b)),
                 TT::pack2(fmaf(c.template s<4>(), f16lo(p2), c.b), fmaf(c.template s<7>(), f16hi(p2), c.b)),
                 TT::pack2(fmaf(c.template s<2>(), f16lo(p3), c.b), fmaf(c.template s<5>(), f16hi(p3), c.b))};
  } else if constexpr (BITS == 5) {
    const uint32_t p0 = sub_pair<5, G, 0, 1, 0>(w), p1 = sub_pair<5, G, 2, 4, 0>(w);
    const uint32_t p2 = sub_pair<5, G, 5, 7, 0>(w), p3 = sub_pair<5, G, 3, 6, 2>(w);
    const float e0 = fmaf(c.template s<0>(), f16lo(p0), c.b), e1 = fmaf(c.template s<5>(), f16hi(p0), c.b);
    const float e2 = fmaf(c.template s<2>(), f16lo(p1), c.b), e4 = fmaf(c.template s<4>(), f16hi(p1), c.b);
    const float e5 = fmaf(c.template s<1>(), f16lo(p2), c.b), e7 = fmaf(c.template s<3>(), f16hi(p2), c.b);
    const float e3 = fmaf(c.template s<5>(), f16lo(p3), c.b), e6 = fmaf(c.template s<4>(), f16hi(p3), c.b);
    return u32x4{TT::pack2(e0, e1), TT::pack2(e2, e3), TT::pack2(e4, e5), TT::pack2(e6, e7)};
  } else {
    static_assert(BITS == 6, "2, 3, 4, 5, 6 or 8 bits");
    const uint32_t p0 = sub_pair<6, G, 0, 4, 0>(w), p1 = sub_pair<6, G, 1, 5, 2>(w);
    const uint32_t p2 = sub_pair<6, G, 2, 6, 0>(w), p3 = sub_pair<6, G, 3, 7, 0>(w);
    const float s0 = c.s24, s4 = c.template s<4>(), s2 = c.template s<2>();
    return u32x4{TT::pack2(fmaf(s0, f16lo(p0), c.b), fmaf(s4, f16lo(p1), c.b)),
                 TT::pack2(fmaf(s4, f16lo(p2), c.b), fmaf(s2, f16lo(p3), c.b)),
                 TT::pack2(fmaf(s0, f16hi(p0), c.b), fmaf(s4, f16hi(p1), c.b)),
                 TT::pack2(fmaf(s4, f16hi(p2), c.b), fmaf(s2, f16hi(p3), c.b))};
  }
}

}  // namespace dev
}  // namespace cpq
