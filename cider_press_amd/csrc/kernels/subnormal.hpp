// Vote-free exact dequantization: packed values as f16 subnormals.
//
// A value q < 2^bits left at bit position p of a 16-bit half (p + bits <= 10)
// reads as the f16 subnormal q * 2^(p - 24): no conversion, the field is only
// masked.  v_fma_mix_f32 takes that f16 as one operand, so
//   fma(s * 2^(24 - p), q * 2^(p - 24), b) == fmaf(s, q, b)
// with one rounding.  s * 2^(24 - p) is exact in fp32 for every f16 scale and
// for every bf16 scale with a biased exponent below 231 (|s| < 2^104); larger
// ones (and Inf, NaN) overflow, so callers compare the scales they meet with
// kSubScaleLimit and use BigCst for them.  Checked on the host for every scale
// pattern, value and place (tests/test_subnormal.py); the fields' extraction on
// the GPU against the oracle's weights, bit for bit, for every width
// (tests/test_exact_weights.py).  Against the 1024 + q form of
// dequant_slice_nat this needs no group check up front and no b - 1024 s.
#pragma once

#include "common.hpp"

namespace cpq {
namespace dev {

typedef __amdgpu_buffer_rsrc_t Rsrc;

// The words of the chunk at byte `off` (4-byte aligned).
template <int BITS>
__device__ __forceinline__ void load_words(Rsrc r, uint32_t off, uint32_t* w) {
  if constexpr (BITS == 2) {
    const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
    w[0] = v.x; w[1] = v.y;
  } else if constexpr (BITS == 3) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b96(r, off, 0, 0);
    w[0] = v[0]; w[1] = v[1]; w[2] = v[2];
  } else {
    const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
    w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
    if constexpr (BITS == 5) w[4] = __builtin_amdgcn_raw_buffer_load_b32(r, off + 16, 0, 0);
    if constexpr (BITS == 6) {
      const u32x2 u = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, off + 16, 0, 0));
      w[4] = u.x; w[5] = u.y;
    }
    if constexpr (BITS == 8) {
      const u32x4 u = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off + 16, 0, 0));
      w[4] = u.x; w[5] = u.y; w[6] = u.z; w[7] = u.w;
    }
  }
}

// Largest scale pattern (sign cleared) that SubCst takes, plus one.
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

// A chunk's constants: val<SH>(h) is fmaf(s, q, b) of a field SH bits up, read
// as the f16 subnormal h.
struct SubCst {
  float s24, b;  // s * 2^24
  template <int SH>
  __device__ __forceinline__ float val(float h) const {
    return fmaf(s24 * (1.0f / (float)(1 << SH)), h, b);
  }
};

// The same for scales past kSubScaleLimit: the field scaled to q first.
struct BigCst {
  float s, b;
  template <int SH>
  __device__ __forceinline__ float val(float h) const {
    return fmaf(s, h * (16777216.0f / (float)(1 << SH)), b);
  }
};

// 8-element group G (0..3) of a chunk as 4 packed T pairs in element order.
template <typename TT, int BITS, int G, typename C>
__device__ __forceinline__ u32x4 sub_group(const uint32_t* w, const C& c) {
  if constexpr (BITS == 4) {
    const uint32_t v = w[G], v8 = v >> 8;
    const uint32_t p0 = v & 0x000F000Fu, p1 = v & 0x00F000F0u;    // (e0, e4), (e1, e5) 4 up
    const uint32_t p2 = v8 & 0x000F000Fu, p3 = v8 & 0x00F000F0u;  // (e2, e6), (e3, e7) 4 up
    return u32x4{TT::pack2(c.template val<0>(f16lo(p0)), c.template val<4>(f16lo(p1))),
                 TT::pack2(c.template val<0>(f16lo(p2)), c.template val<4>(f16lo(p3))),
                 TT::pack2(c.template val<0>(f16hi(p0)), c.template val<4>(f16hi(p1))),
                 TT::pack2(c.template val<0>(f16hi(p2)), c.template val<4>(f16hi(p3)))};
  } else if constexpr (BITS == 8) {
    u32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t p = __builtin_amdgcn_perm(0u, w[2 * G + (j >> 1)], (j & 1) ? 0x0c030c02u : 0x0c010c00u);
      o[j] = TT::pack2(c.template val<0>(f16lo(p)), c.template val<0>(f16hi(p)));
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
    return u32x4{TT::pack2(c.template val<0>(f16lo(p01)), c.template val<2>(f16hi(p01))),
                 TT::pack2(c.template val<4>(f16lo(p23)), c.template val<6>(f16hi(p23))),
                 TT::pack2(c.template val<0>(f16lo(p45)), c.template val<2>(f16hi(p45))),
                 TT::pack2(c.template val<4>(f16lo(p67)), c.template val<6>(f16hi(p67)))};
  } else if constexpr (BITS == 3) {
    const uint32_t p0 = sub_pair<3, G, 0, 1, 0>(w), p1 = sub_pair<3, G, 2, 3, 0>(w);
    const uint32_t p2 = sub_pair<3, G, 4, 5, 0>(w), p3 = sub_pair<3, G, 6, 7, 0>(w);
    return u32x4{TT::pack2(c.template val<0>(f16lo(p0)), c.template val<3>(f16hi(p0))),
                 TT::pack2(c.template val<6>(f16lo(p1)), c.template val<1>(f16hi(p1))),
                 TT::pack2(c.template val<4>(f16lo(p2)), c.template val<7>(f16hi(p2))),
                 TT::pack2(c.template val<2>(f16lo(p3)), c.template val<5>(f16hi(p3)))};
  } else if constexpr (BITS == 5) {
    const uint32_t p0 = sub_pair<5, G, 0, 1, 0>(w), p1 = sub_pair<5, G, 2, 4, 0>(w);
    const uint32_t p2 = sub_pair<5, G, 5, 7, 0>(w), p3 = sub_pair<5, G, 3, 6, 2>(w);
    const float e0 = c.template val<0>(f16lo(p0)), e1 = c.template val<5>(f16hi(p0));
    const float e2 = c.template val<2>(f16lo(p1)), e4 = c.template val<4>(f16hi(p1));
    const float e5 = c.template val<1>(f16lo(p2)), e7 = c.template val<3>(f16hi(p2));
    const float e3 = c.template val<5>(f16lo(p3)), e6 = c.template val<4>(f16hi(p3));
    return u32x4{TT::pack2(e0, e1), TT::pack2(e2, e3), TT::pack2(e4, e5), TT::pack2(e6, e7)};
  } else {
    static_assert(BITS == 6, "2, 3, 4, 5, 6 or 8 bits");
    const uint32_t p0 = sub_pair<6, G, 0, 4, 0>(w), p1 = sub_pair<6, G, 1, 5, 2>(w);
    const uint32_t p2 = sub_pair<6, G, 2, 6, 0>(w), p3 = sub_pair<6, G, 3, 7, 0>(w);
    return u32x4{TT::pack2(c.template val<0>(f16lo(p0)), c.template val<4>(f16lo(p1))),
                 TT::pack2(c.template val<4>(f16lo(p2)), c.template val<2>(f16lo(p3))),
                 TT::pack2(c.template val<0>(f16hi(p0)), c.template val<4>(f16hi(p1))),
                 TT::pack2(c.template val<4>(f16hi(p2)), c.template val<2>(f16hi(p3)))};
  }
}

}  // namespace dev
}  // namespace cpq
