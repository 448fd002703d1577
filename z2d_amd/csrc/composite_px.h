// composite_px.h - one pixel through one draw: the coverage mask, then the
// draw's operator (src/internal/raster/shared.zig:9-117, compositeOpaque and
// compositeOpacity, for the pixel the raster loops hand it).  Compiled for
// the device by render.hip and, with Z2D_HOST_PIXEL, for the host by the CPU
// harness that runs it under the sanitizers against the oracle.
#pragma once

#include "render.h"

namespace z2d {

Z2D_PX __forceinline__ int32_t clampi(int32_t v, int32_t lo, int32_t hi) {
  return v < lo ? lo : (v > hi ? hi : v);
}

// The supersample mask's alpha for k covered samples of 16 at `bits` bits
// (supersample.zig's packed alpha mask, scaled back to 8 bits).
Z2D_PX __forceinline__ uint32_t ssaa_mask(int k, int bits) {
  switch (bits) {
    case 4: return ((15u * (uint32_t)k) / 16u) * 17u;
    case 2: return ((3u * (uint32_t)k) / 16u) * 85u;
    case 1: return ((1u * (uint32_t)k) / 16u) * 255u;
    default: return (255u * (uint32_t)k) / 16u;
  }
}

// One pixel through one draw, given its sample coverage k (of kfull): the
// paint masked by the coverage (DST_IN), then the draw's operator.  The
// supersample mode masks every pixel of its box, even at zero coverage; the
// solid fast path of painter.fill stays in integer precision.
Z2D_PX __forceinline__ uint32_t composite_cov(uint32_t raw, uint32_t fmt, int k, int kfull,
                                              const DevDraw &D, const DevPaint &P,
                                              const StopView &sv, const uint16_t *bn, int x,
                                              int y) {
  uint32_t mask_a = 255;
  bool masked = true;
  if (D.mode == MODE_SSAA) {
    mask_a = ssaa_mask(k, D.mask_bits);
  } else {
    if (k == 0) return raw;
    if (D.op == Z2D_OP_CLEAR) return pack(I4{0, 0, 0, 0}, fmt);
    if (k >= kfull) {
      if (D.flags & DRAW_FAST_SRC) return pack(P.px, fmt);
      masked = false;
    } else {
      mask_a = (uint32_t)clampi(k * 16 - 1, 0, 255);
    }
  }
  const bool int_path = D.precision == Z2D_PRECISION_INTEGER ||
                        (D.mode != MODE_SSAA && (D.flags & DRAW_FAST_SRC));
  if (int_path) {
    I4 src = P.kind == Z2D_PATTERN_OPAQUE ? P.px : paint_int(P, sv, bn, x, y);
    if (masked) src = op_int(Z2D_OP_DST_IN, src, I4{0, 0, 0, mask_a});
    return pack(op_int(D.op, unpack(raw, fmt), src), fmt);
  }
  F4 src = P.kind == Z2D_PATTERN_OPAQUE ? decode_raw(P.px) : paint_float(P, sv, bn, x, y);
  if (masked) src = op_float(Z2D_OP_DST_IN, src, decode_raw(I4{0, 0, 0, mask_a}));
  return pack(encode_raw(op_float(D.op, decode_raw(unpack(raw, fmt)), src)), fmt);
}

// Channels of s (each <= 255) masked by coverage count k.
Z2D_PX __forceinline__ I4 mask_coverage(I4 s, int k) {
  const uint32_t a = (uint32_t)clampi(k * 16 - 1, 0, 255);
  return I4{imul8(s.r, a), imul8(s.g, a), imul8(s.b, a), imul8(s.a, a)};
}
// s: the paint already masked by the pixel's coverage (channels <= 255).
Z2D_PX __forceinline__ uint32_t composite_src_over(uint32_t raw, uint32_t fmt, I4 s) {
  const I4 d = unpack(raw, fmt);
  const uint32_t sa = s.a, na = 255u - sa;
  const I4 o{u16(s.r + imul8(d.r, na)), u16(s.g + imul8(d.g, na)), u16(s.b + imul8(d.b, na)),
             u16(sa + d.a - imul8(sa, d.a))};
  return pack(o, fmt);
}

// The same two steps on RGBA8 words (red in the low byte), two channels at
// a time in the 16-bit halves of a word, with packed 16-bit arithmetic.  For
// x = a * b <= 255 * 255, floor(x / 255) is (y + (y >> 8)) >> 8 with
// y = x + 1, and ceil(x / 255) the same with y = x + 255 (floor((x + 254) /
// 255)); y + (y >> 8) stays below 2^16 in both, so each is a multiply-add, a
// shift, an add and a shift, the last shared by what is added next.
typedef unsigned short z_u16x2 __attribute__((ext_vector_type(2)));
Z2D_PX __forceinline__ z_u16x2 as_u16x2(uint32_t v) { return __builtin_bit_cast(z_u16x2, v); }
Z2D_PX __forceinline__ uint32_t as_u32(z_u16x2 v) { return __builtin_bit_cast(uint32_t, v); }
// 256 * (a * m + c - 1 divided by 255, rounded down) per half, plus a low
// byte below 256 (a, m <= 255; c 1 or 255)
Z2D_PX __forceinline__ z_u16x2 div255_hi(z_u16x2 a, z_u16x2 m, z_u16x2 c) {
  const z_u16x2 y = a * m + c;
  return y + (y >> (unsigned short)8);
}

// A pixel in the strip worker's registers: red and blue, green and alpha, one
// channel in the low byte of each 16-bit half.
struct Px2 {
  uint32_t rb, ga;
};
Z2D_PX __forceinline__ Px2 px2_rgba8(uint32_t raw) {
  return Px2{raw & 0x00FF00FFu, (raw >> 8) & 0x00FF00FFu};
}
Z2D_PX __forceinline__ uint32_t px2_to_rgba8(Px2 p) { return p.rb | (p.ga << 8); }
Z2D_PX __forceinline__ Px2 px2_unpack(uint32_t raw, uint32_t fmt) {
  const I4 v = unpack(raw, fmt);
  return Px2{v.r | (v.b << 16), v.g | (v.a << 16)};
}
Z2D_PX __forceinline__ uint32_t px2_pack(Px2 p, uint32_t fmt) {
  return pack(I4{p.rb & 0xFFFFu, p.ga & 0xFFFFu, p.rb >> 16, p.ga >> 16}, fmt);
}
// src_over of the RGBA8 word s: per channel s + floor(d * (255 - sa) / 255),
// truncated to a byte; alpha s + d - floor(s * d / 255), which is
// s + ceil(d * (255 - s) / 255).  The sum of 256 times the quotient and 256
// times the source holds the truncated byte in its high byte.
Z2D_PX __forceinline__ Px2 px2_src_over(Px2 d, uint32_t s) {
  const uint32_t na = 0x00FF00FFu - (s >> 24) * 0x00010001u;
  const uint32_t s_rb = (s << 8) & 0xFF00FF00u, s_ga = s & 0xFF00FF00u;
  const z_u16x2 rb = div255_hi(as_u16x2(d.rb), as_u16x2(na), as_u16x2(0x00010001u)) + as_u16x2(s_rb);
  const z_u16x2 ga = div255_hi(as_u16x2(d.ga), as_u16x2(na), as_u16x2(0x00FF0001u)) + as_u16x2(s_ga);
  return Px2{as_u32(rb >> (unsigned short)8), as_u32(ga >> (unsigned short)8)};
}
// mask_coverage on an RGBA8 word.  Full coverage (k = 16) leaves the word as
// it is and none gives 0, whose src_over leaves the destination as it is.
Z2D_PX __forceinline__ uint32_t mask_coverage_rgba8(uint32_t s, int k) {
  const uint32_t a = (uint32_t)clampi(k * 16 - 1, 0, 255) * 0x00010001u;
  const z_u16x2 rb = div255_hi(as_u16x2(s & 0x00FF00FFu), as_u16x2(a), as_u16x2(0x00010001u));
  const z_u16x2 ga = div255_hi(as_u16x2((s >> 8) & 0x00FF00FFu), as_u16x2(a), as_u16x2(0x00010001u));
  return ((as_u32(rb) >> 8) & 0x00FF00FFu) | (as_u32(ga) & 0xFF00FF00u);
}
// composite_src_over on an RGBA8 surface word d and RGBA8 source s
Z2D_PX __forceinline__ uint32_t src_over_rgba8(uint32_t d, uint32_t s) {
  return px2_to_rgba8(px2_src_over(px2_rgba8(d), s));
}

}  // namespace z2d
