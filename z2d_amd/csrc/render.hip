// render.hip - gfx950 kernels of the fill/stroke/composite hot path.
//
// Pipeline for one job (any number of surfaces and draws, one stream):
//   k_edge_build  flattened nodes -> Polygon edges + extents + draw setup
//                 (fill_plotter.plot, Polygon.addEdge/inBox and the raster
//                 entry logic of src/internal/raster/{direct,multisample,
//                 supersample}.zig), and the edges counted per (draw, band)
//                 entry
//   k_rowprog     serial row emulation, only for draws whose coverage depends
//                 on the reference's sort order (unbalanced contours) or whose
//                 direct-mode unbounded clears depend on whole rows
//   k_edge_bins / scan
//                 per (draw, band) entry, the draw's edges that meet the band
//   k_band_pass / scan
//                 ordered per-band lists of entries (band_h-row bins, draw
//                 order kept)
//   k_strip_pass / scan
//                 per strip (TILE_W x ROWS_PER_THREAD pixels), the band
//                 entries whose composite region meets it, in draw order
//   k_render      strip workers, one wave per strip: the strip stays in
//                 registers while each draw of its list is
//                 rasterized (exact f64 intercepts accumulated as winding
//                 deltas in LDS, wave prefix scans for per-sample winding) and
//                 composited in draw order; HBM sees one read and one write
//                 per strip pixel
//   k_composite   SurfaceCompositor.run batches (src/compositor.zig:302-440)
#include <hip/hip_runtime.h>

#include "composite_px.h"
#include "render.h"

namespace z2d {

// ---------------------------------------------------------------------------
// surface memory
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t load_raw(const DevSurface &s, int64_t idx) {
  switch (s.fmt) {
    case Z2D_FORMAT_ALPHA8: return s.data[idx];
    case Z2D_FORMAT_ALPHA4:
    case Z2D_FORMAT_ALPHA2:
    case Z2D_FORMAT_ALPHA1: {
      int bits = fmt_bits(s.fmt);
      uint64_t bit = (uint64_t)idx * bits;
      return (s.data[bit >> 3] >> (bit & 7)) & ((1u << bits) - 1u);
    }
    default: return reinterpret_cast<const uint32_t *>(s.data)[idx];
  }
}

// Packed alpha rows are not byte aligned, so neighbouring tiles can share a
// byte: packed stores go through 32-bit atomics on the containing word.
__device__ __forceinline__ void store_raw(const DevSurface &s, int64_t idx, uint32_t v) {
  switch (s.fmt) {
    case Z2D_FORMAT_ALPHA8: s.data[idx] = (uint8_t)v; break;
    case Z2D_FORMAT_ALPHA4:
    case Z2D_FORMAT_ALPHA2:
    case Z2D_FORMAT_ALPHA1: {
      int bits = fmt_bits(s.fmt);
      uint64_t bit = (uint64_t)idx * bits;
      uint32_t *word = reinterpret_cast<uint32_t *>(s.data) + (bit >> 5);
      uint32_t sh = (uint32_t)(bit & 31);
      uint32_t mask = ((1u << bits) - 1u) << sh;
      atomicAnd(word, ~mask);
      atomicOr(word, (v << sh) & mask);
    } break;
    default: reinterpret_cast<uint32_t *>(s.data)[idx] = v; break;
  }
}


// Inclusive prefix sum over the 64 lanes of a wave (DPP row shifts within
// 16-lane rows, then row broadcasts across rows), one DPP add per step: a
// shift reads 0 past the row's start (bound_ctrl), a broadcast leaves the
// rows outside its row mask as they were.  Written out because the
// compiler keeps some of the builtin form's steps as a DPP move and an add.
// Each step reads the previous one's result through DPP, which needs two
// wait states after the VALU write (s_nop 1); the first covers the
// caller's write of x.  Every lane of the wave must be active.
__device__ __forceinline__ int32_t wave_incl_scan(int32_t x) {
  asm("s_nop 1\n\t"
      "v_add_u32_dpp %0, %0, %0 row_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "s_nop 1\n\t"
      "v_add_u32_dpp %0, %0, %0 row_shr:2 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "s_nop 1\n\t"
      "v_add_u32_dpp %0, %0, %0 row_shr:4 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "s_nop 1\n\t"
      "v_add_u32_dpp %0, %0, %0 row_shr:8 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "s_nop 1\n\t"
      "v_add_u32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_add_u32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf"
      : "+v"(x));
  return x;
}

// Minimum / maximum over the 64 lanes of a wave as a wave-uniform value.
// The DPP steps have no bound_ctrl, so a lane whose source lies outside its
// row (or outside the broadcast's row mask) is not written and keeps its
// value; lane 63 ends with the extreme of the whole wave.  Every lane of
// the wave must be active.
__device__ __forceinline__ int32_t wave_min_i32(int32_t x) {
  asm("s_nop 1\n\t"
      "v_min_i32_dpp %0, %0, %0 row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_min_i32_dpp %0, %0, %0 row_shr:2 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_min_i32_dpp %0, %0, %0 row_shr:4 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_min_i32_dpp %0, %0, %0 row_shr:8 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_min_i32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_min_i32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf"
      : "+v"(x));
  return __builtin_amdgcn_readlane(x, 63);
}
__device__ __forceinline__ int32_t wave_max_i32(int32_t x) {
  asm("s_nop 1\n\t"
      "v_max_i32_dpp %0, %0, %0 row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_max_i32_dpp %0, %0, %0 row_shr:2 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_max_i32_dpp %0, %0, %0 row_shr:4 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_max_i32_dpp %0, %0, %0 row_shr:8 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_max_i32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_max_i32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf"
      : "+v"(x));
  return __builtin_amdgcn_readlane(x, 63);
}

// ---------------------------------------------------------------------------
// Edges and extents (k_edge_build).
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool pt_eq(double ax, double ay, double bx, double by) {
  return ax == bx && ay == by;
}

struct ExtAcc {
  uint32_t n;
  double top, bottom, left, right;
};

// Polygon.addEdge (src/internal/tess/Polygon.zig:61-109).
__device__ __forceinline__ void add_edge(z2d_edge *out, ExtAcc &acc, double scale, double x0,
                                         double y0, double x1, double y1) {
  double ax = x0 * scale, ay = y0 * scale, bx = x1 * scale, by = y1 * scale;
  z2d_edge e;
  if (ay < by) {
    e.y0 = ay; e.y1 = by; e.x_start = ax; e.x_inc = (bx - ax) / (by - ay);
  } else if (ay > by) {
    e.y0 = ay; e.y1 = by; e.x_start = bx; e.x_inc = (ax - bx) / (ay - by);
  } else {
    return;
  }
  double top = e.y0 < e.y1 ? e.y0 : e.y1, bottom = e.y0 < e.y1 ? e.y1 : e.y0;
  double left = ax < bx ? ax : bx, right = ax < bx ? bx : ax;
  if (acc.n == 0) {
    acc.top = top; acc.bottom = bottom; acc.left = left; acc.right = right;
  } else {
    if (top < acc.top) acc.top = top;
    if (bottom > acc.bottom) acc.bottom = bottom;
    if (left < acc.left) acc.left = left;
    if (right > acc.right) acc.right = right;
  }
  out[acc.n++] = e;
}

// Polygon.inBox (src/internal/tess/Polygon.zig:142-201).
__device__ bool in_box(const double *ext, double scale, int32_t w, int32_t h) {
  double top = ext[0], bottom = ext[1], left = ext[2], right = ext[3];
  if (!isfinite(left) || !isfinite(top) || !isfinite(right) || !isfinite(bottom)) return false;
  if (w < 1 || h < 1) return false;
  if (right < 0.0 || bottom < 0.0) return false;
  int32_t sx = (int32_t)floor(left / scale), sy = (int32_t)floor(top / scale);
  int32_t ex = (int32_t)ceil(right / scale), ey = (int32_t)ceil(bottom / scale);
  int32_t pw = ex - sx, ph = ey - sy;
  if (pw <= 0 || ph <= 0) return false;
  if (sx + pw < 0 || sy + ph < 0) return false;
  if (sx >= w || sy >= h) return false;
  return true;
}

// Inclusive max over the lanes of a wave up to this one, by the DPP steps
// of wave_incl_scan with a max (no bound_ctrl: a lane without a source keeps
// its value).  Every lane of the wave must be active.
__device__ __forceinline__ int32_t wave_max_scan(int32_t v) {
  asm("s_nop 1\n\t"
      "v_max_i32_dpp %0, %0, %0 row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_max_i32_dpp %0, %0, %0 row_shr:2 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_max_i32_dpp %0, %0, %0 row_shr:4 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_max_i32_dpp %0, %0, %0 row_shr:8 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_max_i32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_max_i32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf"
      : "+v"(v));
  return v;
}
// Orders this wave's LDS accesses before and after the call (lanes of one
// wave exchanging data through LDS).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// A lane's value read by every lane (src wave-uniform).
__device__ __forceinline__ uint32_t lane_u32(uint32_t v, uint32_t src) {
  return __builtin_amdgcn_readlane(v, src);
}
__device__ __forceinline__ double lane_f64(double v, uint32_t src) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, src);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), src);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
// The value of the lane below (DPP wave_shr:1); lane 0, which has none,
// gets `first`.
__device__ __forceinline__ uint32_t lane_prev_u32(uint32_t v, uint32_t first) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)first, (int)v, 0x138, 0xF, 0xF, false);
}
__device__ __forceinline__ double lane_prev_f64(double v, double first) {
  const uint64_t u = (uint64_t)__double_as_longlong(v), f = (uint64_t)__double_as_longlong(first);
  const uint32_t lo = lane_prev_u32((uint32_t)u, (uint32_t)f);
  const uint32_t hi = lane_prev_u32((uint32_t)(u >> 32), (uint32_t)(f >> 32));
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
// v from the lane `k` below within the lane's row of 16 (DPP row_shr:k);
// the first k lanes of each row get `fill`.
template <int K>
__device__ __forceinline__ double row_shr_f64(double v, double fill) {
  const uint64_t u = (uint64_t)__double_as_longlong(v), f = (uint64_t)__double_as_longlong(fill);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)f, (int)(uint32_t)u,
                                                            0x110 + K, 0xF, 0xF, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(
      (int)(uint32_t)(f >> 32), (int)(uint32_t)(u >> 32), 0x110 + K, 0xF, 0xF, false);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
// fmin / fmax of a double over the 64 lanes as a wave-uniform value: a
// prefix within each row of 16, then the four rows' last lanes.  (fmin and
// fmax drop NaN operands in any order, so the order of the steps does not
// change the result.)  Every lane of the wave must be active.
__device__ __forceinline__ double wave_fmin_f64(double v) {
  const double inf = __builtin_huge_val();
  v = fmin(v, row_shr_f64<1>(v, inf));
  v = fmin(v, row_shr_f64<2>(v, inf));
  v = fmin(v, row_shr_f64<4>(v, inf));
  v = fmin(v, row_shr_f64<8>(v, inf));
  return fmin(fmin(lane_f64(v, 15), lane_f64(v, 31)), fmin(lane_f64(v, 47), lane_f64(v, 63)));
}
__device__ __forceinline__ double wave_fmax_f64(double v) {
  const double ninf = -__builtin_huge_val();
  v = fmax(v, row_shr_f64<1>(v, ninf));
  v = fmax(v, row_shr_f64<2>(v, ninf));
  v = fmax(v, row_shr_f64<4>(v, ninf));
  v = fmax(v, row_shr_f64<8>(v, ninf));
  return fmax(fmax(lane_f64(v, 15), lane_f64(v, 31)), fmax(lane_f64(v, 47), lane_f64(v, 63)));
}

// A double as an unsigned key in the same order (never 0 for a number), and
// back.
__device__ __forceinline__ unsigned long long f64_key(double v) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  return (u >> 63) ? ~u : (u | (1ull << 63));
}
__device__ __forceinline__ double key_f64(unsigned long long k) {
  return __longlong_as_double((long long)((k >> 63) ? (k & ~(1ull << 63)) : ~k));
}

// The fast renderer's paint class of a paint (FAST_PAINT_NONE: the general
// renderer's).
__device__ __forceinline__ uint32_t fast_paint(const DevPaint &P) {
  if (P.kind == Z2D_PATTERN_OPAQUE) return FAST_PAINT_SOLID;
  if (P.kind == Z2D_PATTERN_GRADIENT && P.gradient) {
    const DevGradient &G = *P.gradient;
    if (G.method == Z2D_INTERP_LINEAR_RGB && G.n_stops <= FAST_STOPS && G.type <= 2u)
      return FAST_PAINT_LINEAR + G.type;
  }
  return FAST_PAINT_NONE;
}

// A solid paint's RGBA8 word (FastDraw::px) masked by coverage count k
// (mask_coverage; k = 16: the paint itself), FastDraw::srctab[k].
__device__ __forceinline__ uint32_t fast_srctab_entry(const DevPaint &P, uint32_t k) {
  const uint32_t praw = P.px.r | (P.px.g << 8) | (P.px.b << 16) | (P.px.a << 24);
  const I4 p_px{praw & 0xFFu, (praw >> 8) & 0xFFu, (praw >> 16) & 0xFFu, praw >> 24};
  const I4 m = k >= 16 ? p_px : mask_coverage(p_px, (int)k);
  return m.r | (m.g << 8) | (m.b << 16) | (m.a << 24);
}

// A gradient's constants in a fast draw's block.
__device__ void write_fast_gradient(FastDraw &F, const DevGradient &G, uint32_t pf) {
  F.n_stops = G.n_stops;
  F.identity = G.identity;
  F.gx = G.geom[0];
  F.gy = G.geom[1];
  for (int i = 0; i < 6; i++) F.m[i] = G.m[i];
  for (int i = 0; i < 8; i++) F.p[i] = 0.0;
  if (pf == FAST_PAINT_LINEAR) {
    F.p[0] = G.lin_dx;
    F.p[1] = G.lin_dy;
    F.p[2] = G.lin_inv;
    F.p[3] = G.lin_degenerate ? 1.0 : 0.0;
  } else if (pf == FAST_PAINT_RADIAL) {
    F.p[0] = G.r1;
    F.p[1] = G.r2;
    F.p[2] = G.cdx;
    F.p[3] = G.cdy;
    F.p[4] = G.dr;
    F.p[5] = G.min_dr;
    F.p[6] = G.a;
    F.p[7] = G.inv_a;
  } else {
    F.p[0] = G.conic_angle;
  }
  for (uint32_t i = 0; i < FAST_STOPS; i++) {
    F.offs[i] = i < G.n_stops ? G.offs[i] : __builtin_inff();
    F.pre[i] = i < G.n_stops ? G.pre[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
}

// A fast draw's block: its region and rule, and the paint's constants
// (the solid paint's table is written by the draw's lanes 0..16 before).
__device__ void write_fast_draw(FastDraw &F, const DevDraw &D, const DevPaint &P, uint32_t pf) {
  F.rx0 = D.rx0;
  F.rx1 = D.rx1;
  F.ry0 = D.ry0;
  F.ry1 = D.ry1;
  F.rule = D.rule;
  F.paint = pf;
  F.n_stops = 0;
  F.identity = 1;
  if (pf >= FAST_PAINT_LINEAR && pf <= FAST_PAINT_CONIC) write_fast_gradient(F, *P.gradient, pf);
}

// The copy of the work counters that workgroup (or draw) i adds to.
__device__ __forceinline__ uint32_t *stat_slot(const JobView &J, uint32_t i) {
  return J.counters + 16 + (i % STAT_SLOTS) * STAT_WORDS;
}

// The set-up of draw d once its edges are built (one lane): the raster entry
// logic, visibility, draw window and composite region, and the fast
// renderer's block.
__device__ void draw_setup(const JobView &J, uint32_t d, uint32_t flags, const ExtAcc &acc) {
  DevDraw &D = J.draws[d];
  const DevSurface S = J.surfaces[D.surface];
  const double scale = D.mode == MODE_DIRECT ? 1.0 : 4.0;
  J.draw_rows[d] = make_int2(0, 0);  // not visible unless set below
  D.ext[0] = acc.top; D.ext[1] = acc.bottom; D.ext[2] = acc.left; D.ext[3] = acc.right;

  const int32_t W = S.w, H = S.h;
  const bool bounded = op_is_bounded(D.op);
  if (!bounded) flags |= DRAW_UNBOUNDED;
  if (acc.n > 0) flags |= DRAW_HAS_EDGES;
  const DevPaint &P = J.paints[D.paint];
  if (P.kind == Z2D_PATTERN_OPAQUE &&
      (D.op == Z2D_OP_SRC || (D.op == Z2D_OP_SRC_OVER && P.px_opaque)))
    flags |= DRAW_FAST_SRC;
  D.rx0 = D.ry0 = D.rx1 = D.ry1 = 0;
  D.sx = D.ex = D.sy = D.ey = 0;
  D.mask_bits = 8;
  if (!in_box(D.ext, scale, W, H)) {
    D.flags = flags & ~DRAW_VISIBLE;
    return;
  }
  if (D.mode == MODE_MSAA) {
    // multisample.run (src/internal/raster/multisample.zig:46-80)
    int32_t sy = clampi((int32_t)floor(acc.top / 4.0), 0, H - 1);
    int32_t ey = clampi((int32_t)ceil(acc.bottom / 4.0), sy, H - 1);
    int32_t sx = clampi((int32_t)floor(acc.left / 4.0), 0, W - 1);
    int32_t ex = clampi((int32_t)ceil(acc.right / 4.0), sx, W);
    D.sx = sx; D.ex = ex; D.sy = sy; D.ey = ey;
    if (bounded) {
      D.rx0 = sx; D.rx1 = ex; D.ry0 = sy; D.ry1 = ey + 1;
    } else {
      D.rx0 = 0; D.rx1 = W; D.ry0 = 0; D.ry1 = H;
    }
    D.row_y0 = 4 * sy;
    D.row_n = 4 * (ey - sy + 1);
  } else if (D.mode == MODE_SSAA) {
    // supersample.run (src/internal/raster/supersample.zig:48-184)
    int32_t x0 = bounded ? (int32_t)floor(acc.left / 4.0) : 0;
    int32_t y0 = bounded ? (int32_t)floor(acc.top / 4.0) : 0;
    int32_t x1 = bounded ? (int32_t)ceil(acc.right / 4.0) : W;
    int32_t y1 = bounded ? (int32_t)ceil(acc.bottom / 4.0) : H;
    int32_t bx0 = clampi(x0 * 4, 0, W * 4 - 1), by0 = clampi(y0 * 4, 0, H * 4 - 1);
    int32_t bx1 = clampi(x1 * 4, bx0, W * 4 - 1), by1 = clampi(y1 * 4, by0, H * 4 - 1);
    int32_t dmw = (bx1 + 1 - bx0) / 4, dmh = (by1 + 1 - by0) / 4;
    int32_t cx = x0 > 0 ? x0 : 0, cy = y0 > 0 ? y0 : 0;
    int32_t cw = (dmw + cx > W) ? W - cx : dmw, ch = (dmh + cy > H) ? H - cy : dmh;
    if (cw <= 0 || ch <= 0) {
      D.flags = flags & ~DRAW_VISIBLE;
      return;
    }
    D.rx0 = cx; D.rx1 = cx + cw; D.ry0 = cy; D.ry1 = cy + ch;
    D.mask_bits = (S.fmt == Z2D_FORMAT_ALPHA4) ? 4 : (S.fmt == Z2D_FORMAT_ALPHA2) ? 2
                : (S.fmt == Z2D_FORMAT_ALPHA1) ? 1 : 8;
    D.row_y0 = by0;
    D.row_n = 4 * ch;
  } else {
    // direct.run (src/internal/raster/direct.zig:38-49)
    int32_t psy = bounded ? (int32_t)floor(acc.top) : 0;
    int32_t pey = bounded ? (int32_t)ceil(acc.bottom) : H - 1;
    int32_t sy = clampi(psy, 0, H - 1), ey = clampi(pey, sy, H - 1);
    D.sy = sy; D.ey = ey;
    if (bounded) {
      int32_t lx = (int32_t)floor(acc.left), rx = (int32_t)ceil(acc.right) + 1;
      D.rx0 = clampi(lx, 0, W); D.rx1 = clampi(rx, 0, W);
      D.ry0 = sy; D.ry1 = ey + 1;
      if (D.rx1 <= D.rx0) {
        D.flags = flags & ~DRAW_VISIBLE;
        return;
      }
    } else {
      D.rx0 = 0; D.rx1 = W; D.ry0 = 0; D.ry1 = H;
      flags |= DRAW_ROWPROG;
    }
    D.row_y0 = sy;
    D.row_n = ey - sy + 1;
  }
  D.flags = flags | DRAW_VISIBLE;
  J.draw_rows[d] = make_int2(D.ry0, D.ry1);
  if (J.fast) {
    // (a solid src and a clear do not depend on the precision)
    uint32_t pf = FAST_PAINT_NONE;
    if (D.op == Z2D_OP_SRC_OVER && D.precision == Z2D_PRECISION_INTEGER)
      pf = fast_paint(P);
    else if (D.op == Z2D_OP_CLEAR || (D.op == Z2D_OP_SRC && P.kind == Z2D_PATTERN_OPAQUE))
      pf = FAST_PAINT_REPLACE;
    if (pf != FAST_PAINT_NONE && D.mode == MODE_MSAA &&
        !(D.flags & (DRAW_ROWPROG | DRAW_UNBALANCED | DRAW_UNBOUNDED))) {
      D.flags |= DRAW_FAST;
      write_fast_draw(J.fast[d], D, P, pf);
    }
  }
}

// A draw's edge slots: built by k_edge_build, or the caller's edges where they
// are.
__device__ __forceinline__ const z2d_edge *draw_edges(const JobView &J, const DevDraw &D) {
  return D.input_edges ? J.in_edges + D.in_edge_off : J.edges + D.node_off;
}

// ---------------------------------------------------------------------------
// k_rowprog: the reference's serial scanline loop for one draw per thread
// (WorkingEdgeSet rescan/inc/sort/filter, src/internal/tess/Polygon.zig:
// 275-353), on a private copy of the edges.  Rescanning every sub-row is
// equivalent to rescanning at breakpoints (the set only changes there and a
// rescan of an unchanged set moves nothing), so the order history matches.
// ---------------------------------------------------------------------------
__global__ void k_rowprog(JobView J, const uint32_t *draw_list, uint32_t n_list,
                          z2d_edge *scratch_edges, int32_t *scratch_x,
                          const uint32_t *scratch_off) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_list) return;
  DevDraw &D = J.draws[draw_list[i]];
  if (!(D.flags & DRAW_VISIBLE) || !(D.flags & DRAW_ROWPROG)) return;
  const DevSurface S = J.surfaces[D.surface];
  z2d_edge *E = scratch_edges + scratch_off[i];
  int32_t *X = scratch_x + scratch_off[i];
  uint32_t n_all = 0;
  for (uint32_t k = 0; k < D.edge_cnt; k++) {
    const z2d_edge e = draw_edges(J, D)[k];
    if (D.input_edges || e.y0 != e.y1) E[n_all++] = e;  // (not a slot without an edge)
  }
  RowRec *R = J.rows + D.row_off;
  const bool direct_unbounded = D.mode == MODE_DIRECT && (D.flags & DRAW_UNBOUNDED);
  const int32_t W = S.w;
  for (int32_t r = 0; r < D.row_n; r++) {
    const int32_t ys = D.row_y0 + r;
    const double mid = (double)ys + 0.5;
    // rescan
    uint32_t to = 0;
    for (uint32_t from = 0; from < n_all; from++) {
      double top = E[from].y0 < E[from].y1 ? E[from].y0 : E[from].y1;
      double bot = E[from].y0 < E[from].y1 ? E[from].y1 : E[from].y0;
      if (top < mid && bot >= mid) {
        if (from != to) {
          z2d_edge t = E[to];
          E[to] = E[from];
          E[from] = t;
        }
        to++;
      }
    }
    // inc
    for (uint32_t k = 0; k < to; k++) {
      double top = E[k].y0 < E[k].y1 ? E[k].y0 : E[k].y1;
      X[k] = round_i32(E[k].x_start + (E[k].x_inc * (mid - top)));
    }
    // sort (insertion, stable)
    for (uint32_t a = 1; a < to; a++) {
      uint32_t b = a;
      while (b > 0 && X[b] < X[b - 1]) {
        int32_t tx = X[b]; X[b] = X[b - 1]; X[b - 1] = tx;
        z2d_edge te = E[b]; E[b] = E[b - 1]; E[b - 1] = te;
        b--;
      }
    }
    // filter
    uint32_t nf = to;
    if (D.rule == Z2D_FILL_NON_ZERO) {
      int32_t wn = 0;
      nf = 0;
      for (uint32_t from = 0; from < to; from++) {
        int dir = E[from].y0 < E[from].y1 ? -1 : 1;
        X[nf] = X[from];
        if (wn == 0) {
          wn += dir;
          nf++;
        } else {
          wn += dir;
          if (wn == 0) nf++;
        }
      }
    }
    RowRec rec;
    rec.cutoff = (nf & 1u) ? X[nf - 1] : INT32_MAX;
    rec.kind = 1;
    rec.s = rec.e = 0;
    if (direct_unbounded) {
      if (nf == 0) {
        rec.kind = 0;
      } else {
        uint32_t m = 0;
        int32_t sm = 0, em = 0;
        for (uint32_t p = 0; p < nf / 2; p++) {
          int32_t st = X[2 * p] > 0 ? X[2 * p] : 0;
          if (st >= W) break;
          int32_t en = clampi(X[2 * p + 1], st, W);
          m++;
          sm = st;
          em = en;
        }
        if (m > 0) {
          rec.kind = (m == 1) ? 2 : 3;
          rec.s = sm;
          rec.e = em;
        }
      }
    }
    R[r] = rec;
  }
}

// ---------------------------------------------------------------------------
// Flattening: the fill plotter's node walk with Spline decomposition
// (src/internal/tess/Spline.zig:37-165, fill_plotter.zig:52-118) on the
// device.  A curve starts at its predecessor's end point, so its subdivision
// is independent of the rest of the draw: k_curve_tasks splits each curve's
// recursion into FLAT_TASKS subtrees (one thread each) and k_curve_combine
// turns their counts into offsets and the curve's bounds.  The count pass
// (once per prepared batch, k_flatten_wave, one wave per fill draw and one lane
// per raw node: wave scans give the output offsets and the contour state)
// returns the number of flattened nodes, the contour-balance and
// line-after-close flags, the (edge, band) bound and the bounding box of the
// tracked points, and stores each raw node's output offset; the emit pass
// (every render, k_flatten_nodes and k_curve_tasks) writes the nodes.  Draws
// whose point-buffer state needs the whole walk (FLAT_NONSIMPLE) go through
// k_flatten_serial in both, one thread per draw.  The recursion is walked
// depth-first with the knots of a piece halved from its parent when descending
// and recomputed from the curve by its path of halvings when moving to a
// sibling, which reproduces the recursion's values exactly.
// ---------------------------------------------------------------------------
struct FPt {
  double x, y;
};
__device__ __forceinline__ bool fpeq(FPt a, FPt b) { return a.x == b.x && a.y == b.y; }
__device__ __forceinline__ FPt fhalf(FPt a, FPt b) {
  return FPt{a.x + ((b.x - a.x) / 2.0), a.y + ((b.y - a.y) / 2.0)};
}
struct FKnots {
  FPt a, b, c, d;
};
// Spline.Knots.errorSq (src/internal/tess/Spline.zig:83-123)
__device__ __forceinline__ double knots_err_sq(const FKnots &k) {
  double bx = k.b.x - k.a.x, by = k.b.y - k.a.y, cx = k.c.x - k.a.x, cy = k.c.y - k.a.y;
  if (k.a.x != k.d.x || k.a.y != k.d.y) {
    const double dx = k.d.x - k.a.x, dy = k.d.y - k.a.y;
    const double dd = dx * dx + dy * dy;
    const double bd = bx * dx + by * dy;
    if (bd >= dd) {
      bx -= dx;
      by -= dy;
    } else {
      bx -= bd / dd * dx;
      by -= bd / dd * dy;
    }
    const double cd = cx * dx + cy * dy;
    if (cd >= dd) {
      cx -= dx;
      cy -= dy;
    } else {
      cx -= cd / dd * dx;
      cy -= cd / dd * dy;
    }
  }
  const double be = bx * bx + by * by, ce = cx * cx + cy * cy;
  return be > ce ? be : ce;
}
// deCasteljau at the midpoint: the first (right = false) or second half
__device__ __forceinline__ FKnots knots_half(const FKnots &k, bool right) {
  const FPt ab = fhalf(k.a, k.b), bc = fhalf(k.b, k.c), cd = fhalf(k.c, k.d);
  const FPt abbc = fhalf(ab, bc), bccd = fhalf(bc, cd), fin = fhalf(abbc, bccd);
  return right ? FKnots{fin, bccd, cd, k.d} : FKnots{k.a, ab, abbc, fin};
}

constexpr uint32_t FLAT_MAX_VISITS = 1u << 20;  // per curve

__device__ __forceinline__ double flat_band_span(double a, double b, uint32_t nbands,
                                                 uint32_t band_h) {
  const double lo = fmin(a, b), hi = fmax(a, b);
  if (!isfinite(lo) || !isfinite(hi)) return (double)nbands;
  const double s = floor(hi / band_h) - floor(lo / band_h) + 1.0;
  return fmin(s, (double)nbands);
}

// Spline.decompose from start point a: depth-first over the halvings, leaves
// give their first point unless it is the curve's start, then d; pieces
// deeper than 64 halvings are leaves.  `pt` receives each line_to point.
template <class F>
__device__ __forceinline__ void spline_points(FPt a, FPt b, FPt c, FPt d, double tol_sq,
                                              uint32_t &flags, F &&pt) {
  if (fpeq(a, b) && fpeq(c, d)) {
    pt(d);
    return;
  }
  const FKnots root{a, b, c, d};
  uint32_t depth = 0;
  uint64_t path = 0;  // bit (depth - 1 - i): the half taken at level i
  uint32_t visits = 0;
  FKnots k = root;  // the visited piece: a first half from its parent when
                    // descending, else recomputed from the root by its path
  for (;;) {
    bool leaf = knots_err_sq(k) < tol_sq || depth > 64;
    bool runaway = false;
    if (++visits > FLAT_MAX_VISITS) {
      flags |= FLAT_RUNAWAY;
      runaway = true;
      leaf = true;
    }
    if (!leaf && depth == 64) {
      // both halves are leaves (depth 65): their first points
      if (!fpeq(k.a, a)) pt(k.a);
      const FKnots r = knots_half(k, true);
      if (!fpeq(r.a, a)) pt(r.a);
      leaf = true;
    } else if (leaf) {
      if (!fpeq(k.a, a)) pt(k.a);
    }
    if (leaf) {
      while (depth > 0 && (path & 1u)) {
        path >>= 1;
        depth--;
      }
      if (depth == 0 || runaway) break;
      path |= 1u;  // the second half of the same parent
      k = root;
      for (uint32_t i = 0; i < depth; i++) k = knots_half(k, (path >> (depth - 1 - i)) & 1u);
    } else {
      depth++;
      path <<= 1;
      k = knots_half(k, false);
    }
  }
  pt(d);
}

template <bool EMIT>
struct DevFlattener {
  FNode *out;
  uint32_t n = 0, flags = 0;
  uint64_t pairs = 0;
  uint32_t nbands, band_h;
  double cur_y = 0.0, init_y = 0.0;
  uint32_t last_tag = 0xFFFFFFFFu;
  FPt buf[3];
  int len = 0;
  double box[4] = {INFINITY, -INFINITY, INFINITY, -INFINITY};

  __device__ void track(FPt p) {
    box[0] = fmin(box[0], p.x);
    box[1] = fmax(box[1], p.x);
    box[2] = fmin(box[2], p.y);
    box[3] = fmax(box[3], p.y);
  }
  __device__ void emit(uint32_t tag, FPt p, bool closes = false) {
    if (EMIT) out[n] = FNode{p.x, p.y, tag, closes ? 1u : 0u};
    n++;
    // the (edge, band) bound over the emitted stream, as the host computes it
    if (tag == Z2D_NODE_MOVE_TO) {
      cur_y = init_y = p.y;
    } else if (tag == Z2D_NODE_LINE_TO) {
      pairs += (uint64_t)flat_band_span(cur_y, p.y, nbands, band_h);
      cur_y = p.y;
      if (last_tag == Z2D_NODE_CLOSE_PATH) flags |= FLAT_SERIAL;
    } else if (tag == Z2D_NODE_CLOSE_PATH) {
      pairs += (uint64_t)flat_band_span(cur_y, init_y, nbands, band_h);
      cur_y = init_y;
    }
    last_tag = tag;
  }
  __device__ void add(FPt p) {
    if (len < 3) {
      buf[len++] = p;
    } else {
      buf[1] = buf[2];
      buf[2] = p;
    }
  }
  __device__ void line_to(FPt p) {
    emit(Z2D_NODE_LINE_TO, p);
    track(p);
    if (!fpeq(buf[len - 1], p)) add(p);
  }
  __device__ void curve(FPt b, FPt c, FPt d, double tol_sq) {
    spline_points(buf[len - 1], b, c, d, tol_sq, flags, [&](FPt p) { line_to(p); });
  }
};

// The per-draw walk, for the draws k_flatten_wave marked FLAT_NONSIMPLE
// (count pass) or the host marked serial (emit pass).
template <bool EMIT>
__global__ void k_flatten_serial(const z2d_path_node *__restrict__ raw,
                                 const FlatJob *__restrict__ jobs, uint32_t n_jobs, FNode *out,
                                 FlatResult *res) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n_jobs) return;
  const FlatJob J = jobs[j];
  if (EMIT ? !J.serial : !(res[j].flags & FLAT_NONSIMPLE)) return;
  DevFlattener<EMIT> f;
  f.out = out + J.node_off;
  f.nbands = J.nbands;
  f.band_h = J.band_h;
  const z2d_path_node *nodes = raw + J.raw_off;
  const uint32_t n = J.raw_cnt;
  bool balanced = true;
  // the node walk of the host's checks (tags and first move already
  // validated): fill_plotter.plot with PointBuffer(1, 3)
  for (uint32_t i = 0; i < n; i++) {
    const z2d_path_node nd = nodes[i];
    const FPt p{nd.v[0], nd.v[1]};
    if (nd.tag == Z2D_NODE_MOVE_TO) {
      if (i == n - 1) {
        f.emit(Z2D_NODE_MOVE_TO, p);
        break;
      }
      if (f.len > 0 && !fpeq(f.buf[f.len - 1], f.buf[0])) balanced = false;
      f.len = 0;
      f.add(p);
      f.emit(Z2D_NODE_MOVE_TO, p);
      f.track(p);
    } else if (nd.tag == Z2D_NODE_LINE_TO) {
      f.line_to(p);
    } else if (nd.tag == Z2D_NODE_CURVE_TO) {
      const FPt b{nd.v[0], nd.v[1]}, c{nd.v[2], nd.v[3]}, d{nd.v[4], nd.v[5]};
      f.track(b);
      f.track(c);
      f.curve(b, c, d, J.tol_sq);
    } else {  // close
      const bool closes = f.len >= 3 && !fpeq(f.buf[f.len - 1], f.buf[0]);
      f.emit(Z2D_NODE_CLOSE_PATH, f.len ? f.buf[0] : FPt{0.0, 0.0}, closes);
      if (closes) f.add(f.buf[0]);
    }
  }
  if (f.len > 0 && !fpeq(f.buf[f.len - 1], f.buf[0])) balanced = false;
  if (!EMIT) {
    FlatResult r;
    r.n_nodes = f.n;
    r.flags = f.flags | (balanced ? 0u : FLAT_UNBALANCED) | FLAT_NONSIMPLE;
    r.edge_pairs = f.pairs;
    for (int i = 0; i < 4; i++) r.box[i] = f.box[i];
    res[j] = r;
  }
}

__device__ __forceinline__ void box_track(double *box, FPt p) {
  box[0] = fmin(box[0], p.x);
  box[1] = fmax(box[1], p.x);
  box[2] = fmin(box[2], p.y);
  box[3] = fmax(box[3], p.y);
}

// One wave per draw, one lane per raw node (64 at a time).  For the draws it
// keeps (every close is the last node or followed by a move, comes after a
// move, and ends a contour of at least 3 distinct points), the point buffer
// before a line or curve ends at its predecessor's end point, a close always
// returns the contour to its start, and a contour without a close is
// balanced exactly when it ends at its move point.  The distinct-point count
// is taken over the end points (a curve counted by its end point only), a
// lower bound of the buffer's length, so a draw kept here has at least 3.
__global__ void __launch_bounds__(256) k_flatten_wave(const z2d_path_node *__restrict__ raw,
                                                      const FlatJob *__restrict__ jobs,
                                                      uint32_t n_jobs, FlatResult *res,
                                                      uint32_t *rel, uint32_t *mvi,
                                                      const FlatCurve *__restrict__ cv) {
  constexpr uint32_t NONE = 0xFFFFFFFFu;
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t j = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (j >= n_jobs) return;
  const FlatJob J = jobs[j];
  const z2d_path_node *nodes = raw + J.raw_off;
  uint32_t *rl = rel + J.raw_off;
  const uint32_t n = J.raw_cnt;
  const uint64_t below = (1ull << lane) - 1ull;
  // carried from the previous 64 nodes (wave-uniform)
  uint32_t c_tag = NONE, c_S = 0, c_out = 0, c_mvS = 0, c_mvi = 0, c_cur = J.curve_base;
  FPt c_pt{0.0, 0.0}, c_mv{0.0, 0.0};
  bool c_mv_ok = false;
  // per lane, reduced at the end
  uint64_t pairs = 0;
  uint32_t flags = 0;
  double box[4] = {INFINITY, -INFINITY, INFINITY, -INFINITY};
  for (uint32_t base = 0; base < n; base += 64) {
    const uint32_t i = base + lane;
    const bool act = i < n;
    z2d_path_node nd;
    uint32_t tag = NONE;
    FPt p{0.0, 0.0};
    if (act) {
      nd = nodes[i];
      tag = nd.tag;
      if (tag == Z2D_NODE_MOVE_TO || tag == Z2D_NODE_LINE_TO) p = FPt{nd.v[0], nd.v[1]};
      else if (tag == Z2D_NODE_CURVE_TO) p = FPt{nd.v[4], nd.v[5]};
    }
    // the predecessor's tag and end point
    const uint32_t ptag = lane_prev_u32(tag, c_tag);
    const FPt pp{lane_prev_f64(p.x, c_pt.x), lane_prev_f64(p.y, c_pt.y)};
    const uint32_t ntag = (act && i + 1 < n) ? nodes[i + 1].tag : NONE;
    // S: running count of lines/curves whose end point differs from the
    // previous end point
    uint32_t S = ((tag == Z2D_NODE_LINE_TO || tag == Z2D_NODE_CURVE_TO) && !fpeq(p, pp)) ? 1u : 0u;
    S = (uint32_t)wave_incl_scan((int32_t)S) + c_S;
    // the contour's move: the last move at or before this node, and the last
    // one before it
    const uint64_t mv_mask = __ballot(tag == Z2D_NODE_MOVE_TO);
    const uint64_t at = mv_mask & (below | (1ull << lane)), before = mv_mask & below;
    const int src_at = at ? 63 - __builtin_clzll(at) : 0;
    const int src_bf = before ? 63 - __builtin_clzll(before) : 0;
    FPt mv{__shfl(p.x, src_at, 64), __shfl(p.y, src_at, 64)};
    uint32_t mvS = __shfl(S, src_at, 64);
    FPt mvb{__shfl(p.x, src_bf, 64), __shfl(p.y, src_bf, 64)};
    bool mv_ok = true;
    if (!at) {
      mv = c_mv;
      mvS = c_mvS;
      mv_ok = c_mv_ok;
    }
    if (!before) mvb = c_mv;
    uint32_t cnt = 0;
    if (tag == Z2D_NODE_MOVE_TO) {
      cnt = 1;
      if (i != n - 1) box_track(box, p);
      // the previous contour ends at the predecessor
      if ((ptag == Z2D_NODE_LINE_TO || ptag == Z2D_NODE_CURVE_TO) && !fpeq(pp, mvb))
        flags |= FLAT_UNBALANCED;
    } else if (tag == Z2D_NODE_LINE_TO) {
      cnt = 1;
      box_track(box, p);
      pairs += (uint64_t)flat_band_span(pp.y, p.y, J.nbands, J.band_h);
    } else if (tag == Z2D_NODE_CLOSE_PATH) {
      cnt = 1;
      pairs += (uint64_t)flat_band_span(pp.y, mv.y, J.nbands, J.band_h);
      mvi[J.raw_off + i] = J.raw_off + (at ? base + (uint32_t)src_at : c_mvi);
      if (!mv_ok || (ntag != NONE && ntag != Z2D_NODE_MOVE_TO) || 1u + S - mvS < 3u)
        flags |= FLAT_NONSIMPLE;
    }
    if ((tag == Z2D_NODE_LINE_TO || tag == Z2D_NODE_CURVE_TO) && i == n - 1 && !fpeq(p, mv))
      flags |= FLAT_UNBALANCED;
    // output offsets from the node counts (a curve's from k_curve_combine)
    const uint64_t cm = __ballot(tag == Z2D_NODE_CURVE_TO);
    if (tag == Z2D_NODE_CURVE_TO) {
      const FlatCurve &r = cv[c_cur + (uint32_t)__popcll(cm & below)];
      cnt = r.cnt;
      flags |= r.flags;
      pairs += r.pairs;
      box[0] = fmin(box[0], r.box[0]);
      box[1] = fmax(box[1], r.box[1]);
      box[2] = fmin(box[2], r.box[2]);
      box[3] = fmax(box[3], r.box[3]);
    }
    c_cur += (uint32_t)__popcll(cm);
    const uint32_t x = (uint32_t)wave_incl_scan((int32_t)cnt);
    if (act) rl[i] = c_out + x - cnt;
    c_out += lane_u32(x, 63);
    c_tag = lane_u32(tag, 63);
    c_pt = FPt{lane_f64(p.x, 63), lane_f64(p.y, 63)};
    c_S = lane_u32(S, 63);
    if (mv_mask) {
      const uint32_t last = 63u - (uint32_t)__builtin_clzll(mv_mask);
      c_mv = FPt{lane_f64(p.x, last), lane_f64(p.y, last)};
      c_mvS = lane_u32(S, last);
      c_mvi = base + last;
      c_mv_ok = true;
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    pairs += __shfl_xor(pairs, off, 64);
    flags |= __shfl_xor(flags, off, 64);
    box[0] = fmin(box[0], __shfl_xor(box[0], off, 64));
    box[1] = fmax(box[1], __shfl_xor(box[1], off, 64));
    box[2] = fmin(box[2], __shfl_xor(box[2], off, 64));
    box[3] = fmax(box[3], __shfl_xor(box[3], off, 64));
  }
  if (lane == 0) {
    FlatResult r;
    r.n_nodes = c_out;
    r.flags = flags;
    r.edge_pairs = pairs;
    for (int q = 0; q < 4; q++) r.box[q] = box[q];
    res[j] = r;
  }
}

// Emit pass, one lane per raw node, 64 of a draw per wave: the nodes other
// than curves (k_curve_tasks writes those) at the offsets of the count pass.
// A close gets its contour's move point (mvi), and leads there: a draw kept by
// k_flatten_wave closes only contours of at least two lines that move.  The
// wave per draw of the count pass took 40 us for the 2,300 nodes of a page's
// lines here, a chunk of 64 after the other; this form 7.
__global__ void __launch_bounds__(256) k_flatten_nodes(const z2d_path_node *__restrict__ raw,
                                                       const FlatJob *__restrict__ jobs,
                                                       const uint2 *__restrict__ groups,
                                                       uint32_t n_groups, FNode *out,
                                                       const uint32_t *__restrict__ rel,
                                                       const uint32_t *__restrict__ mvi,
                                                       FillSet fill) {
  // the render's per-step resets (none of them is read by the flattening),
  // here instead of a launch of their own
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint32_t f = 0; f < fill.count; f++)
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < fill.n[f]; i += stride)
      fill.p[f][i] = fill.v[f];
  const uint32_t g = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (g >= n_groups) return;
  const uint2 e = groups[g];  // job, first node
  const FlatJob &J = jobs[e.x];
  const uint32_t i = e.y + (threadIdx.x & 63);
  if (J.serial || i >= J.raw_cnt) return;
  const uint32_t r = J.raw_off + i, tag = raw[r].tag;
  if (tag == Z2D_NODE_CURVE_TO) return;
  const bool close = tag == Z2D_NODE_CLOSE_PATH;
  const z2d_path_node &p = raw[close ? mvi[r] : r];
  out[J.node_off + rel[r]] = FNode{p.v[0], p.v[1], tag, close ? 1u : 0u};
}

// One piece of a curve's Spline walk (task t of FLAT_TASKS): the subtree at
// depth FLAT_TASK_DEPTH along t's bits, depth-first, or the leaf above that
// depth when t is the leftmost piece under it.  Concatenated in t order, the
// pieces give spline_points' leaf points (without the final d).
template <class F>
__device__ __forceinline__ void spline_task(FPt a, FPt b, FPt c, FPt d, double tol_sq, uint32_t t,
                                            uint32_t &flags, F &&pt) {
  const FKnots root{a, b, c, d};
  FKnots k = root;
  for (uint32_t l = 0; l < FLAT_TASK_DEPTH; l++) {
    if (knots_err_sq(k) < tol_sq) {
      if ((t & ((1u << (FLAT_TASK_DEPTH - l)) - 1u)) == 0u && !fpeq(k.a, a)) pt(k.a);
      return;
    }
    k = knots_half(k, (t >> (FLAT_TASK_DEPTH - 1 - l)) & 1u);
  }
  uint32_t depth = FLAT_TASK_DEPTH;
  uint64_t path = t;
  uint32_t visits = 0;
  // the visited piece's parent (set once the walk is below the task's
  // root): a first half's sibling is the parent's second half, the same
  // value the recomputation from the root gives
  FKnots par = k;
  for (;;) {
    bool leaf = knots_err_sq(k) < tol_sq || depth > 64;
    bool runaway = false;
    if (++visits > FLAT_MAX_VISITS) {
      flags |= FLAT_RUNAWAY;
      runaway = true;
      leaf = true;
    }
    if (!leaf && depth == 64) {
      if (!fpeq(k.a, a)) pt(k.a);
      const FKnots r = knots_half(k, true);
      if (!fpeq(r.a, a)) pt(r.a);
      leaf = true;
    } else if (leaf) {
      if (!fpeq(k.a, a)) pt(k.a);
    }
    if (leaf) {
      if (depth > FLAT_TASK_DEPTH && !(path & 1u)) {
        if (runaway) break;
        path |= 1u;  // the second half of the same parent
        k = knots_half(par, true);
        continue;
      }
      while (depth > FLAT_TASK_DEPTH && (path & 1u)) {
        path >>= 1;
        depth--;
      }
      if (depth == FLAT_TASK_DEPTH || runaway) break;
      path |= 1u;
      k = root;
      for (uint32_t i = 0; i < depth; i++) {
        if (i + 1 == depth) par = k;
        k = knots_half(k, (path >> (depth - 1 - i)) & 1u);
      }
    } else {
      depth++;
      path <<= 1;
      par = k;
      k = knots_half(k, false);
    }
  }
}

__device__ __forceinline__ void curve_points(const z2d_path_node *raw, uint32_t i, FPt &a, FPt &b,
                                             FPt &c, FPt &d) {
  // a curve of a per-node draw follows a move, line or curve
  const z2d_path_node nd = raw[i], pv = raw[i - 1];
  a = pv.tag == Z2D_NODE_CURVE_TO ? FPt{pv.v[4], pv.v[5]} : FPt{pv.v[0], pv.v[1]};
  b = FPt{nd.v[0], nd.v[1]};
  c = FPt{nd.v[2], nd.v[3]};
  d = FPt{nd.v[4], nd.v[5]};
}

// One thread per curve piece.  Count pass: the piece's point count, its
// first and last y, the (edge, band) bound between its points and its box.
// Emit pass: its points at the offset k_curve_combine gave it; the last
// piece adds the curve's end point.
template <bool EMIT>
__global__ void __launch_bounds__(256) k_curve_tasks(const z2d_path_node *__restrict__ raw,
                                                     const FlatJob *__restrict__ jobs,
                                                     const uint2 *__restrict__ curves,
                                                     uint32_t n_curves, FlatTask *tasks,
                                                     const uint32_t *__restrict__ toff,
                                                     const uint32_t *__restrict__ rel,
                                                     FNode *out) {
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t ci = g / FLAT_TASKS, t = g % FLAT_TASKS;
  if (ci >= n_curves) return;
  const uint2 e = curves[ci];
  const FlatJob &J = jobs[e.x];
  if (EMIT && J.serial) return;
  FPt a, b, c, d;
  curve_points(raw, e.y, a, b, c, d);
  const bool degenerate = fpeq(a, b) && fpeq(c, d);  // the curve is one line to d
  uint32_t flags = 0;
  if (EMIT) {
    FNode *o = out + J.node_off + rel[e.y] + toff[g];
    uint32_t k = 0;
    if (!degenerate)
      spline_task(a, b, c, d, J.tol_sq, t, flags,
                  [&](FPt q) { o[k++] = FNode{q.x, q.y, Z2D_NODE_LINE_TO, 0u}; });
    if (t == FLAT_TASKS - 1) o[k] = FNode{d.x, d.y, Z2D_NODE_LINE_TO, 0u};
  } else {
    FlatTask r;
    r.cnt = 0;
    r.pairs = 0;
    r.fy = r.ly = 0.0;
    r.box[0] = r.box[2] = INFINITY;
    r.box[1] = r.box[3] = -INFINITY;
    if (!degenerate)
      spline_task(a, b, c, d, J.tol_sq, t, flags, [&](FPt q) {
        if (r.cnt) r.pairs += (uint64_t)flat_band_span(r.ly, q.y, J.nbands, J.band_h);
        else r.fy = q.y;
        r.ly = q.y;
        r.cnt++;
        box_track(r.box, q);
      });
    r.flags = flags;
    tasks[g] = r;
  }
}

// Count pass, one thread per curve: piece offsets, and the curve's point
// count (pieces + its end point), (edge, band) bound from its start point
// along all its points, box (control points and points) and flags.
__global__ void __launch_bounds__(256) k_curve_combine(const z2d_path_node *__restrict__ raw,
                                                       const FlatJob *__restrict__ jobs,
                                                       const uint2 *__restrict__ curves,
                                                       uint32_t n_curves,
                                                       const FlatTask *__restrict__ tasks,
                                                       uint32_t *toff, FlatCurve *cv) {
  const uint32_t ci = blockIdx.x * blockDim.x + threadIdx.x;
  if (ci >= n_curves) return;
  const uint2 e = curves[ci];
  const FlatJob &J = jobs[e.x];
  FPt a, b, c, d;
  curve_points(raw, e.y, a, b, c, d);
  FlatCurve r;
  r.cnt = 0;
  r.flags = 0;
  r.pairs = 0;
  r.box[0] = r.box[2] = INFINITY;
  r.box[1] = r.box[3] = -INFINITY;
  box_track(r.box, b);
  box_track(r.box, c);
  double cy = a.y;
  for (uint32_t t = 0; t < FLAT_TASKS; t++) {
    const FlatTask &T = tasks[ci * FLAT_TASKS + t];
    toff[ci * FLAT_TASKS + t] = r.cnt;
    r.flags |= T.flags;
    if (!T.cnt) continue;
    r.pairs += (uint64_t)flat_band_span(cy, T.fy, J.nbands, J.band_h) + T.pairs;
    cy = T.ly;
    r.cnt += T.cnt;
    r.box[0] = fmin(r.box[0], T.box[0]);
    r.box[1] = fmax(r.box[1], T.box[1]);
    r.box[2] = fmin(r.box[2], T.box[2]);
    r.box[3] = fmax(r.box[3], T.box[3]);
  }
  r.pairs += (uint64_t)flat_band_span(cy, d.y, J.nbands, J.band_h);
  box_track(r.box, d);
  r.cnt += 1;
  cv[ci] = r;
}

// ---------------------------------------------------------------------------
// Running sums over the workgroups of a launch, in one pass (decoupled
// look-back): the workgroups are numbered by a ticket taken when they start,
// so each waits only on workgroups already running.  A workgroup publishes
// its aggregate, then its inclusive prefix, in its status word
// (flag << 32 | value); its first wave sums its predecessors' words, 64 at a
// time, back to the nearest inclusive prefix.  stat[0] is the ticket and
// stat[1 + b] the status of workgroup b, all zero at launch.  A wait that
// outlasts SCAN_SPIN_LIMIT polls (never expected) sets bit 1 of *err and goes
// on, so every workgroup ends.
// ---------------------------------------------------------------------------
constexpr uint64_t SCAN_AGG = 1ull << 32, SCAN_INCL = 2ull << 32;
constexpr uint32_t SCAN_SPIN_LIMIT = 1u << 20;

__device__ __forceinline__ uint32_t scan_ticket(uint64_t *stat) {
  return (uint32_t)atomicAdd(reinterpret_cast<unsigned long long *>(stat), 1ull);
}
// The sum of the workgroups before `bid` (by one whole wave of it).
__device__ __forceinline__ uint32_t scan_lookback(uint64_t *stat, uint32_t bid, uint32_t total,
                                                  uint32_t lane, uint32_t *err) {
  uint64_t *const st = stat + 1;
  uint32_t off = 0;
  if (lane == 0)
    __hip_atomic_store(&st[bid], (bid == 0 ? SCAN_INCL : SCAN_AGG) | total, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  if (bid == 0) return 0;
  uint32_t spins = 0;
  for (int32_t base = (int32_t)bid - 1;; base -= 64) {
    const int32_t j = base - (int32_t)lane;  // lane 0 the nearest predecessor
    uint64_t s = SCAN_INCL;                  // before workgroup 0: an inclusive zero
    for (;;) {
      if (j >= 0) s = __hip_atomic_load(&st[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (__ballot((s >> 32) == 0) == 0) break;
      if (++spins > SCAN_SPIN_LIMIT) {
        if (lane == 0) atomicOr(err, 2u);
        s = SCAN_INCL | (s & 0xFFFFFFFFull);
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    const uint64_t pm = __ballot((s >> 32) == 2);
    const uint32_t first = pm ? (uint32_t)__builtin_ctzll(pm) : 63u;
    const uint32_t part = (uint32_t)wave_incl_scan(lane <= first ? (int32_t)(uint32_t)s : 0);
    off += (uint32_t)__builtin_amdgcn_readlane((int32_t)part, 63);
    if (pm) break;
  }
  if (lane == 0)
    __hip_atomic_store(&st[bid], SCAN_INCL | (off + total), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  return off;
}

// ---------------------------------------------------------------------------
// Binning: ordered draw lists per band (band_h rows of one surface).
// ---------------------------------------------------------------------------
// One wave per slot: a band and 64 consecutive draws of its surface (every
// band has at least one slot).  The draws whose composite rows meet the band
// are counted, a workgroup's slots (PER for each of its 16 waves) take their
// places by a look-back over the workgroups before, and the wave writes its
// part of the band list (the draws' entry indices, in draw order), the band's
// offset in band_cnt and each listed entry's record (its edge list from
// k_edge_bins).  Bound by latency; as a counting launch, a scan and a writing
// launch it took a small frame 5 us more.  A workgroup's ticket is an add on
// one address (12 ns): past 512 workgroups (PASS_GROUPS) each wave takes
// several slots.  Measured: 1,326 workgroups of the 4K scene take 41 us with a
// slot per wave, 35 with two, 33 with four, 1,024 surfaces 35, 26 and 28, but
// 160 workgroups of 300 surfaces 11 with one and 23 with four.  The strip pass
// below: 8,400 workgroups 185 us with a tile per wave, 136 with two, 116 with four,
// 111 with eight, 126 with 16; 510 workgroups 34 with one and 102 with eight;
// 645 workgroups 20, 18, 17, 25 and 45.
constexpr uint32_t PASS_WAVES = 16, PASS_GROUPS = 512, BAND_PASS_PER = 4, STRIP_PASS_PER = 8;

template <uint32_t PER>
__global__ void __launch_bounds__(64 * PASS_WAVES) k_band_pass(JobView J, uint64_t *stat) {
  __shared__ uint32_t s_cnt[PASS_WAVES * PER], s_bid, s_off;
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (threadIdx.x == 0) s_bid = scan_ticket(stat);
  __syncthreads();
  const uint32_t bid = s_bid;
  if (bid >= gridDim.x) return;  // (uniform) the ticket starts at zero
  bool hit[PER];
  uint32_t idx[PER], dr[PER];
  uint64_t m[PER];
#pragma unroll
  for (uint32_t j = 0; j < PER; j++) {
    const uint32_t slot = (bid * PASS_WAVES + wv) * PER + j;
    hit[j] = false;
    idx[j] = dr[j] = 0;
    if (slot < J.n_slots) {
      const uint2 si = J.slot_info[slot];  // band, surface
      const uint32_t b = si.x, s = si.y;
      const uint32_t lb = b - J.surf_band_off[s];  // band within the surface
      const int32_t y0 = (int32_t)lb * (int32_t)J.band_h, y1 = y0 + (int32_t)J.band_h;
      const uint32_t d = J.surf_draw_off[s] + (slot - J.band_slot_off[b]) * 64 + lane;
      dr[j] = d;
      if (d < J.surf_draw_off[s + 1]) {
        const int2 r = J.draw_rows[d];
        if (r.x < y1 && r.y > y0) {
          // the draw's entry for this band (entries are owned by draws)
          const DevDraw &D = J.draws[d];
          const uint32_t blo = D.band_lo, bhi = D.band_hi;
          if (lb < blo || lb > bhi) {
            atomicOr(&J.counters[2], 1u);  // outside the host's band estimate
          } else {
            hit[j] = true;
            idx[j] = D.entry_base + (lb - blo);
          }
        }
      }
    }
    m[j] = __ballot(hit[j]);
    if (lane == 0) s_cnt[wv * PER + j] = (uint32_t)__popcll(m[j]);
  }
  __syncthreads();
  if (wv == 0) {
    const uint32_t v = lane < PASS_WAVES * PER ? s_cnt[lane] : 0u;
    const uint32_t incl = (uint32_t)wave_incl_scan((int32_t)v);
    const uint32_t total = lane_u32(incl, 63);
    const uint32_t off = scan_lookback(stat, bid, total, lane, J.counters + 2);
    if (lane < PASS_WAVES * PER) s_cnt[lane] = incl - v;
    if (lane == 0) {
      s_off = off;
      if (bid == gridDim.x - 1) J.band_cnt[J.n_bands] = off + total;
    }
  }
  __syncthreads();
#pragma unroll
  for (uint32_t j = 0; j < PER; j++) {
    const uint32_t slot = (bid * PASS_WAVES + wv) * PER + j;
    if (slot >= J.n_slots) break;  // uniform
    const uint2 si = J.slot_info[slot];
    const uint32_t b = si.x;
    const int32_t y0 = (int32_t)(b - J.surf_band_off[si.y]) * (int32_t)J.band_h;
    const uint32_t base = s_off + s_cnt[wv * PER + j];
    if (hit[j]) {
      const uint32_t pos = base + (uint32_t)__popcll(m[j] & ((1ull << lane) - 1ull));
      if (pos < J.max_entries) {
        // only indices below the edge capacity were stored
        const uint32_t off = J.entry_ecnt[idx[j]], cnt = J.entry_ecnt[idx[j] + 1] - off;
        BandEntry e;
        e.draw = dr[j];
        e.edge_off = off;
        e.edge_cnt = off >= J.max_entry_edges ? 0u : min(cnt, J.max_entry_edges - off);
        e.band = b;
        // A tile wholly right of every crossing of the entry's edges, or wholly
        // left of them, sees winding 0 (contours return to their start), so no
        // coverage; with a bounded operator outside SSAA (which composites its
        // whole mask box) nothing changes there.  Sample columns to pixels,
        // rounded outward.
        e.px_lo = INT32_MIN;
        e.px_hi = INT32_MAX;
        const DevDraw &Dd = J.draws[dr[j]];
        if (Dd.mode != MODE_SSAA &&
            !(Dd.flags & (DRAW_UNBOUNDED | DRAW_UNBALANCED | DRAW_ROWPROG | DRAW_SERIAL_PLOT))) {
          const int32_t sc = Dd.mode == MODE_DIRECT ? 1 : 4;
          const int32_t xl = J.entry_xlo[idx[j]], xh = J.entry_xhi[idx[j]];
          if (xl > xh) {  // no edges in the band
            e.px_lo = INT32_MAX;
            e.px_hi = INT32_MIN;
          } else if (xl != INT32_MIN && xh != INT32_MAX) {
            e.px_lo = (int32_t)floor((double)xl / sc);
            e.px_hi = (int32_t)floor((double)xh / sc);
          }
        }
        J.entries[idx[j]] = e;
        // the strip pass's tests for this entry: a tile at column tx0 (>= 0)
        // takes it when it is not wholly beside the entry's crossings (px_lo
        // >= tx0 + TILE_W + 1 or px_hi <= tx0 - 2) and meets the composite
        // region (rx0 < tx0 + TILE_W, tx0 < rx1); a strip when its rows meet
        // [ry0, ry1)
        const int64_t lo_x = max(max((int64_t)Dd.rx0 - TILE_W, (int64_t)e.px_lo - TILE_W - 1),
                                 (int64_t)-1);
        const int64_t hi_x = min(min((int64_t)Dd.rx1, (int64_t)e.px_hi + 2), (int64_t)INT32_MAX);
        uint32_t smask = 0;
        for (uint32_t st = 0; st < J.strips_per_tile; st++) {
          const int32_t sy0 = y0 + (int32_t)st * ROWS_PER_THREAD;
          if (Dd.ry1 > sy0 && Dd.ry0 < sy0 + ROWS_PER_THREAD) smask |= 1u << st;
        }
        const bool slow = !(Dd.flags & DRAW_FAST) || e.edge_cnt > PACKED_EDGE_LIMIT;
        J.band_list[pos] = make_uint4(idx[j], (uint32_t)(int32_t)lo_x,
                                      (uint32_t)(int32_t)max(hi_x, lo_x), smask | (slow ? 256u : 0u));
      } else {
        atomicOr(&J.counters[2], 1u);
      }
    }
    if (lane == 0 && slot == J.band_slot_off[b]) J.band_cnt[b] = base;
  }
}
static_assert(PASS_WAVES * BAND_PASS_PER <= 64, "one lane per slot in the workgroup's scan");

// Exclusive scan of n u32 values in place; a[n] receives the total.  One
// workgroup of 1024 lanes walks the array in chunks of 16 values per lane.
__global__ void __launch_bounds__(1024) k_scan(uint32_t *a, uint32_t n) {
  constexpr uint32_t PER = 16;
  __shared__ uint32_t wsum[16];
  __shared__ uint32_t chunk_total;
  const uint32_t t = threadIdx.x, lane = t & 63, w = t >> 6;
  uint32_t carry = 0;
  for (uint32_t base = 0; base < n; base += 1024 * PER) {
    const uint32_t i0 = base + t * PER;
    uint32_t v[PER];
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t k = 0; k < PER; k++) {
      v[k] = i0 + k < n ? a[i0 + k] : 0u;
      sum += v[k];
    }
    // wave inclusive scan of the lane sums
    const uint32_t x = (uint32_t)wave_incl_scan((int32_t)sum);
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    if (t < 16) {
      const uint32_t s0 = wsum[t];
      uint32_t z = s0;
      for (int off = 1; off < 16; off <<= 1) {
        const uint32_t y = __shfl_up(z, off, 16);
        if (t >= (uint32_t)off) z += y;
      }
      wsum[t] = z - s0;  // exclusive wave offsets
      if (t == 15) chunk_total = z;
    }
    __syncthreads();
    uint32_t run = carry + wsum[w] + x - sum;
#pragma unroll
    for (uint32_t k = 0; k < PER; k++) {
      if (i0 + k < n) a[i0 + k] = run;
      run += v[k];
    }
    carry += chunk_total;
    __syncthreads();
  }
  if (t == 0) a[n] = carry;
}

// Exclusive scan of a[0..n) in place with a[n] = total: SCAN_BLOCK values per
// workgroup, running sums by look-back.
__global__ void __launch_bounds__(256) k_scan_lb(uint32_t *a, uint32_t n, uint64_t *stat,
                                                 uint32_t *err) {
  __shared__ uint32_t ws[4];
  __shared__ uint32_t s_bid, s_off;
  const uint32_t t = threadIdx.x, lane = t & 63, w = t >> 6;
  if (t == 0) s_bid = scan_ticket(stat);
  __syncthreads();
  const uint32_t bid = s_bid;
  if (bid >= gridDim.x) return;  // (uniform) the ticket starts at zero
  const uint32_t i0 = bid * SCAN_BLOCK + t * 16;
  // a lane's 16 values: four 16-byte loads when all lie below n (a is
  // 16-byte aligned and i0 a multiple of 16)
  const bool whole = i0 + 16 <= n;
  uint32_t v[16];
  if (whole) {
#pragma unroll
    for (uint32_t q = 0; q < 4; q++) {
      const uint4 u = reinterpret_cast<const uint4 *>(a + i0)[q];
      v[4 * q] = u.x;
      v[4 * q + 1] = u.y;
      v[4 * q + 2] = u.z;
      v[4 * q + 3] = u.w;
    }
  } else {
#pragma unroll
    for (uint32_t k = 0; k < 16; k++) v[k] = i0 + k < n ? a[i0 + k] : 0u;
  }
  uint32_t sum = 0;
#pragma unroll
  for (uint32_t k = 0; k < 16; k++) sum += v[k];
  const uint32_t x = (uint32_t)wave_incl_scan((int32_t)sum);
  if (lane == 63) ws[w] = x;
  __syncthreads();
  if (w == 0) {
    const uint32_t off = scan_lookback(stat, bid, ws[0] + ws[1] + ws[2] + ws[3], lane, err);
    if (lane == 0) s_off = off;
  }
  __syncthreads();
  uint32_t run = s_off + x - sum;
  for (uint32_t j = 0; j < w; j++) run += ws[j];
  uint32_t o[16];
#pragma unroll
  for (uint32_t k = 0; k < 16; k++) {
    o[k] = run;
    run += v[k];
  }
  if (whole) {
#pragma unroll
    for (uint32_t q = 0; q < 4; q++)
      reinterpret_cast<uint4 *>(a + i0)[q] =
          make_uint4(o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]);
  } else {
#pragma unroll
    for (uint32_t k = 0; k < 16; k++)
      if (i0 + k < n) a[i0 + k] = o[k];
  }
  if (bid == gridDim.x - 1 && t == 255) a[n] = run;
}

// Exclusive scan of a[0..n) in place with a[n] = total; stat holds
// n / SCAN_BLOCK + 2 zeroed words.
static void scan_u32(uint32_t *a, uint32_t n, uint64_t *stat, uint32_t *err, hipStream_t st) {
  const uint32_t nb = n == 0 ? 1u : (n + SCAN_BLOCK - 1) / SCAN_BLOCK;
  hipLaunchKernelGGL(k_scan_lb, dim3(nb), dim3(256), 0, st, a, n, stat, err);
}

// ---------------------------------------------------------------------------
// k_strip_pass: per strip (ROWS_PER_THREAD rows of one tile), the entries of
// its band list whose composite region meets the strip, in draw order.  One
// wave per tile walks the band's entries twice: counting per strip, and, once
// the workgroup's tiles (PER for each of its 16 waves) have their places by
// look-back, writing; the strips that hold a general-renderer entry are
// appended to slow_list.  That list's length is one address and adds to it
// are served one by one, so a workgroup takes its places with one add (one
// add per tile took 304 us for 134,000 tiles, a fifth of them with such
// strips), and as with its ticket, past PASS_GROUPS workgroups each wave takes
// several tiles: 14 us for a 4K page, 6 us for a small frame, whose three launches
// took 14 and 10 and the gaps between them.
// ---------------------------------------------------------------------------
template <uint32_t PER>
__global__ void __launch_bounds__(64 * PASS_WAVES) k_strip_pass(JobView J, uint64_t *stat) {
  constexpr uint32_t TILES = PASS_WAVES * PER;
  constexpr uint32_t LANE_STRIPS = TILES * MAX_STRIPS_PER_TILE / 64;
  // per strip of the workgroup, in strip order: its count, then its offset
  __shared__ uint32_t s_cnt[TILES * MAX_STRIPS_PER_TILE];
  // per tile: its strips with a general-renderer entry, then their place in
  // the slow list (above bit 8)
  __shared__ uint32_t s_slow[TILES];
  __shared__ uint32_t s_slow_base, s_bid, s_off;
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (threadIdx.x == 0) s_bid = scan_ticket(stat);
  __syncthreads();
  const uint32_t bid = s_bid;
  if (bid >= gridDim.x) return;  // (uniform) the ticket starts at zero
  const uint32_t spt = J.strips_per_tile;
  const uint64_t below = (1ull << lane) - 1ull;
  // the band list of tile t, and the strips that its entry e + lane meets
  // (see k_band_pass)
  uint32_t e0 = 0, e1 = 0;
  int32_t tx0 = 0;
  auto tile = [&](uint32_t t) {
    const TileRef T = J.tiles[t];
    const uint32_t b = J.surf_band_off[T.surface] + T.ty;
    e0 = min(J.band_cnt[b], J.max_entries);
    e1 = min(J.band_cnt[b + 1], J.max_entries);
    tx0 = (int32_t)T.tx * TILE_W;
  };
  auto entry = [&](uint32_t e, uint32_t &idx, bool &slow) {
    uint32_t mask = 0;
    idx = 0;
    slow = false;
    if (e + lane < e1) {
      const uint4 it = J.band_list[e + lane];
      idx = it.x;
      slow = (it.w & 256u) != 0;
      if (tx0 > (int32_t)it.y && tx0 < (int32_t)it.z) mask = it.w & 255u;
    }
    return mask;
  };
  for (uint32_t j = 0; j < PER; j++) {
    const uint32_t lt = wv * PER + j, t = bid * TILES + lt;
    uint32_t cnt[MAX_STRIPS_PER_TILE];
#pragma unroll
    for (int s = 0; s < MAX_STRIPS_PER_TILE; s++) cnt[s] = 0;
    uint32_t slow_strips = 0;
    if (t < J.n_tiles) {
      tile(t);
      for (uint32_t e = e0; e < e1; e += 64) {
        uint32_t idx;
        bool slow;
        const uint32_t mask = entry(e, idx, slow);
#pragma unroll
        for (int s = 0; s < MAX_STRIPS_PER_TILE; s++) {
          if ((uint32_t)s >= spt) break;  // uniform
          const bool hit = (mask >> s) & 1u;
          cnt[s] += (uint32_t)__popcll(__ballot(hit));
          if (__ballot(hit && slow)) slow_strips |= 1u << s;
        }
      }
    }
    if (lane == 0) {
#pragma unroll
      for (int s = 0; s < MAX_STRIPS_PER_TILE; s++)
        if ((uint32_t)s < spt) s_cnt[lt * spt + s] = cnt[s];
      s_slow[lt] = slow_strips;
    }
  }
  __syncthreads();
  if (wv == 0) {
    const uint32_t n = TILES * spt, i0 = LANE_STRIPS * lane;
    uint32_t sum = 0;
    for (uint32_t i = i0; i < min(i0 + LANE_STRIPS, n); i++) sum += s_cnt[i];
    const uint32_t incl = (uint32_t)wave_incl_scan((int32_t)sum);
    const uint32_t total = lane_u32(incl, 63);
    const uint32_t off = scan_lookback(stat, bid, total, lane, J.counters + 2);
    uint32_t run = incl - sum;
    for (uint32_t i = i0; i < min(i0 + LANE_STRIPS, n); i++) {
      const uint32_t v = s_cnt[i];
      s_cnt[i] = run;
      run += v;
    }
    uint32_t srun = 0;  // general-renderer strips of the tiles before
    for (uint32_t i = 0; i < TILES; i += 64) {
      const uint32_t sl = i + lane < TILES ? s_slow[i + lane] : 0u;
      const uint32_t ns = (uint32_t)__popc(sl);
      const uint32_t sincl = (uint32_t)wave_incl_scan((int32_t)ns);
      if (i + lane < TILES) s_slow[i + lane] = sl | ((srun + sincl - ns) << 8);
      srun += lane_u32(sincl, 63);
    }
    if (lane == 0) {
      s_off = off;
      if (bid == gridDim.x - 1) J.strip_cnt[J.n_tiles * spt] = off + total;
      if (srun) s_slow_base = atomicAdd(&J.counters[9], srun);
    }
  }
  __syncthreads();
  const uint32_t off = s_off;
  for (uint32_t j = 0; j < PER; j++) {
    const uint32_t lt = wv * PER + j, t = bid * TILES + lt;
    if (t >= J.n_tiles) break;  // uniform
    if (lane < spt) {
      const uint32_t sl = s_slow[lt];
      const bool slow = (sl >> lane) & 1u;
      J.strip_cnt[t * spt + lane] = off + s_cnt[lt * spt + lane];
      J.strip_slow[t * spt + lane] = slow ? 1u : 0u;
      if (slow)
        J.slow_list[s_slow_base + (sl >> 8) + (uint32_t)__popc(sl & ((1u << lane) - 1u))] =
            t * spt + lane;
    }
    uint32_t next[MAX_STRIPS_PER_TILE];
#pragma unroll
    for (int s = 0; s < MAX_STRIPS_PER_TILE; s++)
      next[s] = (uint32_t)s < spt ? off + s_cnt[lt * spt + s] : 0u;
    tile(t);
    for (uint32_t e = e0; e < e1; e += 64) {
      uint32_t idx;
      bool slow;
      const uint32_t mask = entry(e, idx, slow);
#pragma unroll
      for (int s = 0; s < MAX_STRIPS_PER_TILE; s++) {
        if ((uint32_t)s >= spt) break;  // uniform
        const bool hit = (mask >> s) & 1u;
        const uint64_t m = __ballot(hit);
        if (hit) {
          const uint32_t pos = next[s] + (uint32_t)__popcll(m & below);
          if (pos < J.max_strip_entries)
            J.strip_entries[pos] = idx;
          else
            atomicOr(&J.counters[2], 1u);
        }
        next[s] += (uint32_t)__popcll(m);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Longest-first strip order: a counting sort of the strips by list length
// (descending), so that the long strips are dispatched first and the short
// ones fill the tail.  Order within a length class is free.  Its adds to 1,024
// addresses are served one after another on each: 35 to 42 ms for the two million
// strips of 4,096 surfaces, against 8 ms for the rest of their render, so it
// is for batches whose longest strips outweigh that (the autotuner measures).
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t order_bucket(const JobView &J, uint32_t i) {
  const uint32_t n = J.strip_cnt[i + 1] - J.strip_cnt[i];
  return ORDER_BUCKETS - 1u - min(n, ORDER_BUCKETS - 1u);
}
__global__ void k_order_hist(JobView J, uint32_t n_strips) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_strips) atomicAdd(&J.order_hist[order_bucket(J, i)], 1u);
}
// after the scan of order_hist: each strip takes the next slot of its class
__global__ void k_order_scatter(JobView J, uint32_t n_strips) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_strips) return;
  const uint32_t pos = atomicAdd(&J.order_hist[order_bucket(J, i)], 1u);
  if (pos < n_strips) J.strip_order[pos] = i;
}

// ---------------------------------------------------------------------------
// Sample rows of an edge: the smallest y with top < y + 0.5 and the largest
// with y + 0.5 <= bottom (the active-edge test of Polygon.zig:284-285).  The
// floor estimates are corrected with those exact comparisons; values are
// clamped to [-2, 2^29] (rows outside every surface behave alike there).
// ---------------------------------------------------------------------------
constexpr double ROW_CLAMP = 536870912.0;  // 2^29
__device__ __forceinline__ int32_t row_lo(double top) {
  const double f = floor(top - 0.5) + 1.0;
  if (!(f > -2.0)) return -2;
  if (f > ROW_CLAMP) return (int32_t)ROW_CLAMP;
  int32_t y = (int32_t)f;
  if ((double)(y - 1) + 0.5 > top)
    y--;
  else if (!((double)y + 0.5 > top))
    y++;
  return y;
}
__device__ __forceinline__ int32_t row_hi(double bot) {
  const double f = floor(bot - 0.5);
  if (!(f > -2.0)) return -2;
  if (f > ROW_CLAMP) return (int32_t)ROW_CLAMP;
  int32_t y = (int32_t)f;
  if ((double)(y + 1) + 0.5 <= bot)
    y++;
  else if (!((double)y + 0.5 <= bot))
    y--;
  return y;
}
__device__ __forceinline__ REdge make_redge(const z2d_edge &e) {
  const bool down = e.y0 < e.y1;
  const double top = down ? e.y0 : e.y1, bot = down ? e.y1 : e.y0;
  REdge r;
  r.top = top;
  r.x_start = e.x_start;
  r.x_inc = e.x_inc;
  r.ylo = row_lo(top);
  r.yhi2 = row_hi(bot) * 2 + (down ? 1 : 0);
  return r;
}
// The crossing of an edge with sample row y: x_start + x_inc * ((y + 0.5) -
// top), rounded to the nearest integer, ties away from zero (the
// reference's intercept, src/internal/tess/Polygon.zig:302-307; no fused
// multiply-add).
__device__ __forceinline__ double redge_x(double top, double x_start, double x_inc, int32_t y) {
  return x_start + (x_inc * (((double)y + 0.5) - top));
}

// ---------------------------------------------------------------------------
// k_edge_build: the edges of a draw, 64 node slots per wave (slot k: the edge
// that node k adds, if any), their extents, and their number per (draw, band)
// entry.  fill_plotter.plot (src/internal/tess/fill_plotter.zig:21-97) with
// the PointBuffer(1, 3) of src/internal/tess/point_buffer.zig asks of the
// nodes before a line or close only its predecessor's point, and of a close
// what the flattening left in it (FNode), so every slot is on its own; draws
// in which a line follows a close go node by node in their first wave.
// The wave that completes a draw sets it up (draw_setup).
// Bound by latency: one wave per draw before, which took a chunk of 64 nodes
// after the other (57 us for 101 draws of a page of text, 19 us for the 61
// of a small frame, and 13.5 and 5.5 us more in a pass of its own for the
// counting); 20 and 14 us now, of memory latency and of the last wave's set-up.
// ---------------------------------------------------------------------------
// The bands [lo, hi] of `rows` sample rows, among [rb_lo, rb_hi], that an edge
// meets: top < b's last sample row + 0.5 and bot >= its first + 0.5 (the
// active-edge test over the band; lo > hi: none).  Both hold over a range of
// bands; floor estimates, wider by one, are corrected with the exact
// comparisons.  No sample row meets an edge without height (a slot without an
// edge, a caller's horizontal edge) or with a NaN end: no band has it,
// whatever [rb_lo, rb_hi] is, so that k_edge_build, which counts, and
// k_edge_bins, which places, agree on every edge.
__device__ __forceinline__ void edge_bands(double top, double bot, int32_t rows, int32_t rb_lo,
                                           int32_t rb_hi, int32_t &lo, int32_t &hi) {
  lo = INT32_MAX;
  hi = INT32_MIN;
  if (!(top < bot)) return;
  const double flo = fmax(floor(top / (double)rows) - 1.0, (double)rb_lo);
  const double fhi = fmin(floor(bot / (double)rows) + 1.0, (double)rb_hi);
  if (!(flo <= fhi)) return;
  int32_t l = (int32_t)flo, h = (int32_t)fhi;
#pragma unroll
  for (int i = 0; i < 3; i++) {
    if (!(top < (double)((l + 1) * rows - 1) + 0.5)) l++;
    if (!(bot >= (double)(h * rows) + 0.5)) h--;
  }
  if (l > h) return;
  lo = l;
  hi = h;
}
// A wave's edges against the bands [ulo, uhi]: edge by edge, a lane per band,
// where that is fewer steps (a rectangle's two edges down a whole surface)
// than band by band, a lane per edge.
__device__ __forceinline__ bool by_edge(uint64_t edges, int32_t ulo, int32_t uhi) {
  const int32_t n = uhi - ulo + 1;
  return (int32_t)__popcll(edges) * ((n + 63) >> 6) < n;
}

__global__ void __launch_bounds__(256) k_edge_build(JobView J) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t g = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (g >= J.n_egroups) return;
  const uint2 it = J.egroups[g];  // draw, first slot
  const uint32_t d = it.x;
  DevDraw &D = J.draws[d];
  uint32_t flags = D.flags & (DRAW_UNBALANCED | DRAW_ROWPROG | DRAW_SERIAL_PLOT);
  const uint32_t n = D.node_cnt, input = D.input_edges;
  const bool serial = !input && (flags & DRAW_SERIAL_PLOT);
  if (serial && it.y != 0) return;
  // groups that the set-up waits for (given edges come with their extents)
  const uint32_t n_groups = serial || input || n == 0 ? 1u : (n + EDGE_GROUP - 1) / EDGE_GROUP;
  const bool direct = D.mode == MODE_DIRECT;
  const double scale = direct ? 1.0 : 4.0;
  const int32_t band_rows = (int32_t)J.band_h * (direct ? 1 : 4);
  z2d_edge *const out = J.edges + D.node_off;
  DrawAcc &A = J.draw_acc[d];
  // a solid paint's coverage table, for the fast renderer should the draw be
  // one (lane k: entry k)
  if (it.y == 0 && J.fast && lane <= 16) {
    const bool clear = D.op == Z2D_OP_CLEAR;
    if (clear || J.paints[D.paint].kind == Z2D_PATTERN_OPAQUE)
      J.fast[d].srctab[lane] = clear ? 0u : fast_srctab_entry(J.paints[D.paint], lane);
  }

  ExtAcc acc{0, 0.0, 0.0, 0.0, 0.0};
  uint32_t first = it.y, end = min(it.y + EDGE_GROUP, n);  // the slots counted below
  if (serial) {
    // the plotter's state machine node by node (a line may follow a close)
    if (lane == 0) {
      double fx = 0.0, fy = 0.0, lx = 0.0, ly = 0.0;
      int len = 0;
      const FNode *nodes = J.nodes + D.node_off;
      for (uint32_t i = 0; i < n; i++) {
        const FNode nd = nodes[i];
        if (nd.tag == Z2D_NODE_MOVE_TO) {
          if (i == n - 1) break;
          fx = lx = nd.x;
          fy = ly = nd.y;
          len = 1;
        } else if (nd.tag == Z2D_NODE_LINE_TO) {
          if (len == 0) continue;  // InvalidState is rejected on the host
          if (!pt_eq(lx, ly, nd.x, nd.y)) {
            add_edge(out, acc, scale, lx, ly, nd.x, nd.y);
            lx = nd.x;
            ly = nd.y;
            if (len < 3) len++;
          }
        } else if (nd.tag == Z2D_NODE_CLOSE_PATH) {
          if (len >= 3 && !pt_eq(lx, ly, fx, fy)) {
            add_edge(out, acc, scale, lx, ly, fx, fy);
            lx = fx;
            ly = fy;
          }
        }
      }
    }
    __threadfence_block();  // lane 0's edges, read below by the others
    first = 0;
    end = lane_u32(acc.n, 0);
  }
  for (uint32_t k0 = first; k0 < end; k0 += 64) {
    const uint32_t k = k0 + lane;
    const bool slot = k < end;
    z2d_edge ed{0.0, 0.0, 0.0, 0.0};
    if (serial) {
      if (slot) ed = out[k];
    } else if (input) {
      if (slot) ed = J.in_edges[D.in_edge_off + k];
    } else {
      const FNode *nodes = J.nodes + D.node_off;
      FNode nd{0.0, 0.0, 0xFFFFFFFFu, 0u}, pv{0.0, 0.0, 0xFFFFFFFFu, 0u};
      if (slot) nd = nodes[k];
      if (lane == 0 && k0 > 0) pv = nodes[k0 - 1];
      const double px = lane_prev_f64(nd.x, pv.x), py = lane_prev_f64(nd.y, pv.y);
      const uint32_t ptag = lane_prev_u32(nd.tag, pv.tag);
      // (a line or close before the first move is rejected on the host)
      const bool moves = !pt_eq(px, py, nd.x, nd.y);
      const double ax = px * scale, ay = py * scale, bx = nd.x * scale, by = nd.y * scale;
      const bool emit =
          slot && k > 0 && moves && (ay < by || ay > by) &&
          (nd.tag == Z2D_NODE_LINE_TO ||
           (nd.tag == Z2D_NODE_CLOSE_PATH && nd.closes && ptag != Z2D_NODE_CLOSE_PATH));
      double top = 0.0, bot = 0.0, left = 0.0, right = 0.0;
      if (emit) {  // Polygon.addEdge (src/internal/tess/Polygon.zig:61-109)
        ed.y0 = ay;
        ed.y1 = by;
        if (ay < by) {
          ed.x_start = ax;
          ed.x_inc = (bx - ax) / (by - ay);
        } else {
          ed.x_start = bx;
          ed.x_inc = (ax - bx) / (ay - by);
        }
        top = ay < by ? ay : by;
        bot = ay < by ? by : ay;
        left = ax < bx ? ax : bx;
        right = ax < bx ? bx : ax;
      }
      if (slot) out[k] = ed;
      const uint64_t m = __ballot(emit);
      if (m) {
        const double inf = __builtin_huge_val();
        acc.n = (uint32_t)__popcll(m);
        acc.top = wave_fmin_f64(emit ? top : inf);
        acc.bottom = wave_fmax_f64(emit ? bot : -inf);
        acc.left = wave_fmin_f64(emit ? left : inf);
        acc.right = wave_fmax_f64(emit ? right : -inf);
        if (n_groups > 1 && lane < 4) {
          const double v = lane == 0 ? acc.top : lane == 1 ? acc.bottom : lane == 2 ? acc.left : acc.right;
          atomicMax(&A.key[lane], lane & 1u ? f64_key(v) : ~f64_key(v));
        }
      }
    }
    // the edges counted per band of the draw's entries
    const double top = ed.y0 < ed.y1 ? ed.y0 : ed.y1, bot = ed.y0 < ed.y1 ? ed.y1 : ed.y0;
    int32_t lo = INT32_MAX, hi = INT32_MIN;
    edge_bands(top, bot, band_rows, (int32_t)D.band_lo, (int32_t)D.band_hi, lo, hi);
    const int32_t ulo = wave_min_i32(lo), uhi = wave_max_i32(hi);
    const uint64_t em = __ballot(lo <= hi);
    const bool transposed = by_edge(em, ulo, uhi);
    for (int32_t w = ulo; w <= uhi; w += 64) {
      const int32_t bj = w + (int32_t)lane;  // this lane's band
      uint32_t cnt = 0;
      if (transposed) {
        for (uint64_t r = em; r; r &= r - 1) {
          const uint32_t e = (uint32_t)__builtin_ctzll(r);
          const int32_t l = (int32_t)lane_u32((uint32_t)lo, e), h = (int32_t)lane_u32((uint32_t)hi, e);
          cnt += (l <= bj && bj <= h) ? 1u : 0u;
        }
      } else {
        const int32_t wend = min(uhi, w + 63);
        for (int32_t bnd = w; bnd <= wend; bnd++) {
          const uint32_t c = (uint32_t)__popcll(__ballot(lo <= bnd && bnd <= hi));
          if (bj == bnd) cnt = c;
        }
      }
      if (cnt) atomicAdd(&J.entry_ecnt[D.entry_base + ((uint32_t)bj - D.band_lo)], cnt);
    }
  }
  if (n_groups > 1) {
    // the draw's last group sets it up: this wave's maxima have been made
    // (waited for) when it counts itself done, and they and the reads below
    // are atomics at device scope, so the last group reads every group's
    // without a fence (whose write-back of the L2 took 36 ns a group)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    unsigned long long done = 0;
    if (lane == 0) done = atomicAdd(&A.done, (1ull << 32) | acc.n) + ((1ull << 32) | acc.n);
    if (lane != 0 || (uint32_t)(done >> 32) != n_groups) return;
    acc.n = (uint32_t)done;
    double v[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const unsigned long long k =
          __hip_atomic_load(&A.key[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      v[i] = key_f64(i & 1 ? k : ~k);
    }
    if (acc.n) acc = ExtAcc{acc.n, v[0], v[1], v[2], v[3]};
  }
  if (lane != 0 || (input && it.y != 0)) return;
  if (input) acc = ExtAcc{n, D.in_ext[0], D.in_ext[1], D.in_ext[2], D.in_ext[3]};
  D.edge_cnt = serial ? acc.n : n;
  if (J.count_stats && acc.n) atomicAdd(&stat_slot(J, d)[STAT_EDGES], acc.n);
  draw_setup(J, d, flags, acc);
}

// ---------------------------------------------------------------------------
// k_edge_bins: per (draw, band) entry, copies of the draw's edges whose
// y-range meets the band's sample rows (top < last mid && bottom >= first mid,
// the active-edge test of src/internal/raster/multisample.zig and direct.zig
// taken over the band); strips then walk only those edges.  One wave per
// group of EDGE_GROUP edge slots of a draw, after the scan of k_edge_build's
// counts, appending to the entries' lists through the entry_cur cursors (the
// order inside a list is free: the winding deltas of the edges are summed).
// Bound by latency where few edges meet many bands: a band after the other
// was 0.43 us each for a background rectangle's two edges, 58 us of the 61 us
// that a 2160-row page took; with a lane per band instead (by_edge) it takes 20,
// a small frame of 38 bands 9 instead of 17.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_edge_bins(JobView J) {
  __shared__ int32_t s_x[4][2][64];  // per wave: a window's bands' column ranges
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint32_t g = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (g >= J.n_egroups) return;
  const uint2 it = J.egroups[g];  // draw, first edge slot
  const DevDraw &D = J.draws[it.x];
  if (D.mode == MODE_DIRECT && (D.flags & DRAW_UNBOUNDED)) return;  // row records instead
  const int2 rows = J.draw_rows[it.x];
  if (rows.x >= rows.y) return;  // no entries
  const uint32_t ne = D.edge_cnt;
  if (it.y >= ne) return;
  const int32_t bh = (int32_t)J.band_h;
  const int32_t band_rows = bh * (D.mode == MODE_DIRECT ? 1 : 4);
  const int32_t blo = (int32_t)D.band_lo, bhi = (int32_t)D.band_hi;
  const uint32_t ebase = D.entry_base;
  const uint32_t k = it.y + lane;
  z2d_edge ed{0.0, 0.0, 0.0, 0.0};
  double top = 0.0, bot = 0.0;
  int32_t lo = INT32_MAX, hi = INT32_MIN;  // candidate bands among the entries'
  int32_t xlo = INT32_MAX, xhi = INT32_MIN;  // the edge's sample columns
  if (k < min(it.y + EDGE_GROUP, ne)) {
    ed = draw_edges(J, D)[k];
    top = ed.y0 < ed.y1 ? ed.y0 : ed.y1;
    bot = ed.y0 < ed.y1 ? ed.y1 : ed.y0;
    const double xb = ed.x_start + ed.x_inc * (bot - top);
    const double a = fmin(ed.x_start, xb), c = fmax(ed.x_start, xb);
    if (a >= -2.0e9 && c <= 2.0e9) {
      xlo = (int32_t)floor(a);
      xhi = (int32_t)floor(c);
    } else {  // huge or non-finite: the whole row
      xlo = INT32_MIN;
      xhi = INT32_MAX;
    }
    edge_bands(top, bot, band_rows, max(rows.x / bh, blo), min((rows.y - 1) / bh, bhi), lo, hi);
  }
  const REdge red = make_redge(ed);  // the copy every band of the edge receives
  const int32_t ulo = wave_min_i32(lo), uhi = wave_max_i32(hi);
  const uint64_t em = __ballot(lo <= hi);
  const uint64_t below = (1ull << lane) - 1ull;
  const bool transposed = by_edge(em, ulo, uhi);
  // bands in windows of 64: lane j holds the count (then the list position)
  // of band w + j, so each window takes one vector atomic
  for (int32_t w = ulo; w <= uhi; w += 64) {
    const int32_t wend = min(uhi, w + 63);
    const int32_t bj = w + (int32_t)lane;  // this lane's band
    uint32_t cnt = 0;
    if (transposed) {
      int32_t rlo = INT32_MAX, rhi = INT32_MIN;
      for (uint64_t r = em; r; r &= r - 1) {
        const uint32_t e = (uint32_t)__builtin_ctzll(r);
        const int32_t l = (int32_t)lane_u32((uint32_t)lo, e), h = (int32_t)lane_u32((uint32_t)hi, e);
        if (l <= bj && bj <= h) {
          cnt++;
          rlo = min(rlo, (int32_t)lane_u32((uint32_t)xlo, e));
          rhi = max(rhi, (int32_t)lane_u32((uint32_t)xhi, e));
        }
      }
      const uint32_t idx = ebase + (uint32_t)(bj - blo);
      uint32_t pos = 0;
      if (cnt) {
        pos = J.entry_ecnt[idx] + atomicAdd(&J.entry_cur[idx], cnt);
        atomicMin(&J.entry_xlo[idx], rlo);
        atomicMax(&J.entry_xhi[idx], rhi);
      }
      for (uint64_t r = em; r; r &= r - 1) {
        const uint32_t e = (uint32_t)__builtin_ctzll(r);
        const int32_t l = (int32_t)lane_u32((uint32_t)lo, e), h = (int32_t)lane_u32((uint32_t)hi, e);
        const REdge re{lane_f64(red.top, e), lane_f64(red.x_start, e), lane_f64(red.x_inc, e),
                       (int32_t)lane_u32((uint32_t)red.ylo, e),
                       (int32_t)lane_u32((uint32_t)red.yhi2, e)};
        if (l <= bj && bj <= h) {
          if (pos < J.max_entry_edges)
            J.entry_edges[pos] = re;
          else
            atomicOr(&J.counters[2], 1u);
          pos++;
        }
      }
      continue;
    }
    for (int32_t bnd = w; bnd <= wend; bnd++) {
      const uint32_t c = (uint32_t)__popcll(__ballot(lo <= bnd && bnd <= hi));
      if (bj == bnd) cnt = c;
    }
    const uint32_t at = cnt ? J.entry_ecnt[ebase + (uint32_t)(bj - blo)] +
                                  atomicAdd(&J.entry_cur[ebase + (uint32_t)(bj - blo)], cnt)
                            : 0u;
    s_x[wv][0][lane] = INT32_MAX;
    s_x[wv][1][lane] = INT32_MIN;
    wave_lds_sync();
    for (int32_t bnd = w; bnd <= wend; bnd++) {
      const bool hit = lo <= bnd && bnd <= hi;
      const uint64_t m = __ballot(hit);
      if (m == 0) continue;
      const uint32_t base = __builtin_amdgcn_readlane(at, bnd - w);
      if (hit) {
        // the entry's column range, widened by this wave's edges in the band
        atomicMin(&s_x[wv][0][bnd - w], xlo);
        atomicMax(&s_x[wv][1][bnd - w], xhi);
        const uint32_t pos = base + (uint32_t)__popcll(m & below);
        if (pos < J.max_entry_edges)
          J.entry_edges[pos] = red;
        else
          atomicOr(&J.counters[2], 1u);
      }
    }
    wave_lds_sync();
    if (cnt) {
      atomicMin(&J.entry_xlo[ebase + (uint32_t)(bj - blo)], s_x[wv][0][lane]);
      atomicMax(&J.entry_xhi[ebase + (uint32_t)(bj - blo)], s_x[wv][1][lane]);
    }
    wave_lds_sync();
  }
}

// ---------------------------------------------------------------------------
// k_render: tile renderer.
// ---------------------------------------------------------------------------
// Gradients with up to this many stops are read from LDS while a draw is
// composited.
constexpr uint32_t STAGED_STOPS = 64;

// LDS of one strip worker (one wave).
struct StripShared {
  // Winding deltas per sample row and sample column of the strip, two int16
  // columns per word (column 2i in the low half).  Zero between entries:
  // the coverage phase clears what it reads.
  uint32_t acc[STRIP_SUBROWS][ACC_WORDS];
  int32_t clo[64];     // first active sample row in the strip
  uint32_t coff[64];   // exclusive offsets of active-row counts
  float soff[STAGED_STOPS];   // the draw's gradient stops, staged
  float4 spre[STAGED_STOPS];
  union {
    struct {                               // coverage (phase A)
      REdge cedge[64];                     // staged band edges
      uint8_t own[64 * STRIP_SUBROWS];     // owning edge of each work item
    } a;
    struct {                               // composite
      uint32_t ppaint[ROWS_PER_THREAD][64];  // paint samples (RGBA8)
      uint8_t plist[ROWS_PER_THREAD * 64];   // covered (row, lane) pairs
    } c;
  } u;
  uint32_t srctab[17];  // solid paint masked by each coverage count (RGBA8)
  DevPaint paint;      // the draw's paint and gradient, staged
  DevGradient grad;
};

// Loads a value every lane of the wave reads at the same address through the
// scalar data cache (constant address space: read-only for the kernel).
template <typename T>
__device__ __forceinline__ T load_uniform(const T *p) {
#if __HIP_DEVICE_COMPILE__
  return *((const __attribute__((address_space(4))) T *)p);
#else
  return *p;  // host pass only parses device code
#endif
}

// Lane `src`'s value of v (every lane of the wave active).
__device__ __forceinline__ uint32_t lane_read_u32(uint32_t v, uint32_t src) {
  return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(src << 2), (int)v);
}
__device__ __forceinline__ double lane_read_f64(double v, uint32_t src) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = lane_read_u32((uint32_t)u, src), hi = lane_read_u32((uint32_t)(u >> 32), src);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Splits a word of two int16 deltas accumulated with 32-bit adds (the low
// half's borrows land in the high half and are undone here).
__device__ __forceinline__ void unpack_pair(uint32_t w, int32_t &lo, int32_t &hi) {
  lo = (int32_t)(int16_t)(w & 0xFFFFu);
  hi = (int32_t)(w - (uint32_t)lo) >> 16;
}

// Paint samples of a linear or radial (TYPE) gradient pattern interpolated in
// linear RGB
// (Gradient.getOffset, Stop.List.search, interpolateEncodeVec of
// src/gradient.zig) for the pixels listed in sh.u.c.plist; G is wave-uniform
// and its stops are staged in sh.soff / sh.spre.
template <uint32_t TYPE>
__device__ __forceinline__ void dense_gradient(const DevGradient &G, StripShared &sh,
                                               uint32_t tot_p, uint32_t lane, int32_t tx0,
                                               int32_t ty0) {
#pragma unroll 1
  for (uint32_t it = lane; it < tot_p; it += 64) {
    const uint32_t v = sh.u.c.plist[it];
    const uint32_t pl = v & 63u, pi = v >> 6;
    const int32_t x = tx0 + (int32_t)pl, y = ty0 + (int32_t)pi;
    float off;
    if constexpr (TYPE == Z2D_GRADIENT_LINEAR)
      off = linear_offset(G, x, y);
    else
      off = radial_offset(G, x, y);
    int i0, i1;
    float t;
    bool transparent;
    stops_search(sh.soff, G.n_stops, off, i0, i1, t, transparent);
    const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float4 A = transparent ? z : sh.spre[i0];
    const float4 B = transparent ? z : sh.spre[i1];
    const uint32_t r = f2u8(255.0f * lerpf_(A.x, B.x, t));
    const uint32_t g = f2u8(255.0f * lerpf_(A.y, B.y, t));
    const uint32_t b = f2u8(255.0f * lerpf_(A.z, B.z, t));
    const uint32_t a = f2u8(255.0f * lerpf_(A.w, B.w, t));
    sh.u.c.ppaint[pi][pl] = r | (g << 8) | (b << 16) | (a << 24);
  }
}

// The rows of the src_over fast composite.  full_raw: the packed source that
// full coverage stores when the draw takes the solid fast path.
__device__ __forceinline__ void src_over_rows(uint32_t (&pix)[ROWS_PER_THREAD],
                                              const int (&kk)[ROWS_PER_THREAD], uint32_t need,
                                              bool solid, bool fast_full, int kfull,
                                              uint32_t full_raw, const StripShared &sh,
                                              uint32_t lane, uint32_t fmt, uint32_t &n_cov) {
#pragma unroll
  for (int i = 0; i < ROWS_PER_THREAD; i++) {
    if (!((need >> i) & 1u)) continue;
    n_cov++;
    const int k = kk[i];
    if (fast_full && k >= kfull) {
      pix[i] = full_raw;
      continue;
    }
    const uint32_t pv = solid ? sh.srctab[k] : sh.u.c.ppaint[i][lane];
    I4 src{pv & 0xFFu, (pv >> 8) & 0xFFu, (pv >> 16) & 0xFFu, pv >> 24};
    if (!solid && k < kfull) src = mask_coverage(src, k);
    pix[i] = composite_src_over(pix[i], fmt, src);
  }
}

__device__ __forceinline__ bool msaa_preclear(const DevDraw &D, int W, int x, int y) {
  if (y < D.sy) return true;
  if (y > D.ey) return y < W;
  if (D.sx > 0 && x < D.sx) return true;
  if (D.ex < W && x < W - D.ex) return true;
  return false;
}

__device__ __forceinline__ bool wind_in(int32_t w, bool eo) { return eo ? (w & 1) != 0 : w != 0; }

// Covered samples (of 4 x 4) per pixel of the lane's column for the strip's
// rows: each sample row's winding is the prefix sum of the deltas up to the
// sample column (lane-local over the pixel's 4 columns, a wave scan across
// lanes, two sample rows packed into one scan).  Reads and clears the deltas.
// CUT: the row records' cutoff columns apply (unbalanced contours).
template <bool EO, bool CUT>
__device__ __forceinline__ void coverage_msaa(uint32_t (&acc)[STRIP_SUBROWS][ACC_WORDS],
                                              uint32_t lane, int32_t xs_base, int32_t ys_base,
                                              const RowRec *R, int32_t row_y0, int32_t row_n,
                                              int *kk) {
  const int c_lo = (int)lane * 4;
#pragma unroll
  for (int i = 0; i < ROWS_PER_THREAD; i++) {
    int k = 0;
#pragma unroll
    for (int pr = 0; pr < 2; pr++) {
      int32_t d[2][4], tot[2];
#pragma unroll
      for (int q = 0; q < 2; q++) {
        uint2 *slot = reinterpret_cast<uint2 *>(&acc[i * 4 + pr * 2 + q][lane * 2]);
        const uint2 v = *slot;
        *slot = make_uint2(0u, 0u);
        unpack_pair(v.x, d[q][0], d[q][1]);
        unpack_pair(v.y, d[q][2], d[q][3]);
        tot[q] = d[q][0] + d[q][1] + d[q][2] + d[q][3];
      }
      const uint32_t pk = (uint32_t)tot[0] + ((uint32_t)tot[1] << 16);
      const uint32_t exc = (uint32_t)wave_incl_scan((int32_t)pk) - pk;
      int32_t base[2];
      unpack_pair(exc, base[0], base[1]);
#pragma unroll
      for (int q = 0; q < 2; q++) {
        int32_t cutoff = INT32_MAX;
        if (CUT) {
          const int32_t rr = ys_base + i * 4 + pr * 2 + q - row_y0;
          if (rr >= 0 && rr < row_n) cutoff = load_uniform(&R[rr]).cutoff;
        }
        int32_t w = base[q];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          w += d[q][j];
          const bool in = EO ? (w & 1) != 0 : w != 0;
          if (CUT)
            k += (in && xs_base + c_lo + j < cutoff) ? 1 : 0;
          else
            k += in ? 1 : 0;
        }
      }
    }
    kk[i] = k;
  }
}

// Inclusive exclusive-or scan over the lanes of a wave (the steps of
// wave_incl_scan with an xor).  Every lane of the wave must be active.
__device__ __forceinline__ uint32_t wave_xor_scan(uint32_t x) {
  asm("s_nop 1\n\t"
      "v_xor_b32_dpp %0, %0, %0 row_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "s_nop 1\n\t"
      "v_xor_b32_dpp %0, %0, %0 row_shr:2 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "s_nop 1\n\t"
      "v_xor_b32_dpp %0, %0, %0 row_shr:4 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "s_nop 1\n\t"
      "v_xor_b32_dpp %0, %0, %0 row_shr:8 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "s_nop 1\n\t"
      "v_xor_b32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_xor_b32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf"
      : "+v"(x));
  return x;
}

// The fast strip worker's crossings, FAST_ACC_ROWS words per sample column of
// the strip.  A sample is inside by the parity of the crossings at columns up
// to its own (even-odd) or by their winding (non-zero), so what a column has
// to hold depends on the rule:
//   WIND_EO    one bit per sample row (16 of them) in row 0, crossings
//              flipping their bit: exact for any number of edges
//   WIND_NZ    four sample rows (a pixel row) per word, row b as w_b * 256^b
//              summed in 32-bit arithmetic.  The sums are taken modulo 2^32,
//              where they stay exact whatever carries between the bytes, so
//              a word decodes if the four windings at its column lie in
//              [-127, 127]: adding 0x80808080 then leaves each byte
//              w_b + 128.
//   WIND_NZ16  two sample rows per word as lo + hi * 65536, windings in
//              [-32767, 32767]: half a strip (8 sample rows) at a time, for
//              the entries whose windings may not fit a byte
// Words of the earlier layout, two rows to a word for both rules, took 8 reads
// and wave scans per entry; these take 1 (even-odd) and 4, and the block's
// LDS goes from 10.0 KB to 5.9 KB.
constexpr int FAST_ACC_ROWS = ROWS_PER_THREAD, FAST_ACC_COLS = TILE_W * 4;
enum WindMode { WIND_EO = 0, WIND_NZ = 1, WIND_NZ16 = 2 };
typedef uint32_t FastAcc[FAST_ACC_ROWS][FAST_ACC_COLS];

// 1 in each 16-bit half of v that is nonzero, 0 in each that is zero (a
// packed unsigned min with 1; written out because the compiler otherwise
// expands the packed min into per-half compares).
__device__ __forceinline__ uint32_t pk_nonzero_u16(uint32_t v) {
  uint32_t r;
  asm("v_pk_min_u16 %0, %1, %2" : "=v"(r) : "v"(v), "s"(0x00010001u));
  return r;
}

// Covered samples per pixel of the lane's column (kk, a strip's rows; rows
// row0 and row0 + 1 for WIND_NZ16), by prefix sums of the crossings up to
// each sample column (lane-local over the pixel's 4 columns, a wave scan
// across lanes).  Reads and clears the words.  left (WIND_EO): the sample
// rows with an odd number of crossings left of the strip.
__device__ __forceinline__ void coverage_eo(FastAcc &acc, uint32_t lane, uint32_t left, int *kk) {
  uint4 *slot = reinterpret_cast<uint4 *>(&acc[0][lane * 4]);
  const uint4 p = *slot;
  *slot = make_uint4(0u, 0u, 0u, 0u);
  const uint32_t tot = p.x ^ p.y ^ p.z ^ p.w;
  const uint32_t u0 = wave_xor_scan(tot) ^ tot ^ left ^ p.x;
  const uint32_t u1 = u0 ^ p.y, u2 = u1 ^ p.z, u3 = u2 ^ p.w;
  // two columns to a word: the 4 sample rows of pixel row i are bits 4i.. of
  // each half
  const uint32_t v0 = u0 | (u1 << 16), v1 = u2 | (u3 << 16);
#pragma unroll
  for (int i = 0; i < ROWS_PER_THREAD; i++) {
    const uint32_t m = 0x000F000Fu << (4 * i);
    kk[i] = __popc(v0 & m) + __popc(v1 & m);
  }
}
__device__ __forceinline__ void coverage_nz(FastAcc &acc, uint32_t lane, int *kk) {
#pragma unroll
  for (int i = 0; i < ROWS_PER_THREAD; i++) {
    uint4 *slot = reinterpret_cast<uint4 *>(&acc[i][lane * 4]);
    const uint4 p = *slot;
    *slot = make_uint4(0u, 0u, 0u, 0u);
    const uint32_t tot = p.x + p.y + p.z + p.w;
    uint32_t u = (uint32_t)wave_incl_scan((int32_t)tot) - tot + 0x80808080u;
    const uint32_t col[4] = {p.x, p.y, p.z, p.w};
    uint32_t k = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      u += col[j];
      // a byte's mean with 255, rounded down, is below 128 for 0 alone
      const uint32_t nz = __builtin_amdgcn_lerp(u ^ 0x80808080u, 0xFFFFFFFFu, 0u);
      k += (uint32_t)__popc(nz & 0x80808080u);
    }
    kk[i] = (int)k;
  }
}
__device__ __forceinline__ void coverage_nz16(FastAcc &acc, uint32_t lane, int *kk) {
#pragma unroll
  for (int i = 0; i < ROWS_PER_THREAD / 2; i++) {
    uint32_t k = 0;
#pragma unroll
    for (int pr = 0; pr < 2; pr++) {
      uint4 *slot = reinterpret_cast<uint4 *>(&acc[i * 2 + pr][lane * 4]);
      const uint4 p = *slot;
      *slot = make_uint4(0u, 0u, 0u, 0u);
      const uint32_t tot = p.x + p.y + p.z + p.w;
      uint32_t u = (uint32_t)wave_incl_scan((int32_t)tot) - tot + 0x8000u;
      const uint32_t col[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
      for (int j = 0; j < 4; j++) {
        u += col[j];
        k += (uint32_t)__popc(pk_nonzero_u16(u ^ 0x8000u));
      }
    }
    kk[i] = (int)k;
  }
}

// A strip's work counts (stat_pix per lane, the others wave-uniform) added
// to its workgroup's copy of the counters.
__device__ __forceinline__ void strip_stats(const JobView &J, uint32_t stat_pix,
                                            uint32_t stat_entries, uint32_t stat_unpacked,
                                            uint32_t lane) {
  const uint32_t pix = (uint32_t)wave_incl_scan((int32_t)stat_pix);  // < 2^32: 256 px x entries
  if (lane != 63) return;
  uint32_t *const c = stat_slot(J, blockIdx.x);
  if (pix) atomicAdd(reinterpret_cast<unsigned long long *>(&c[STAT_PIX]), (unsigned long long)pix);
  if (stat_entries) atomicAdd(&c[STAT_ENTRIES], stat_entries);
  if (stat_unpacked) atomicAdd(&c[STAT_UNPACKED], stat_unpacked);
}

// The strip worker of the general renderer: one-wave workgroups, each of
// which renders every draw of a strip's list over its ROWS_PER_THREAD x
// TILE_W pixels; they stay in registers from the first draw to the last.
// The hardware's dispatcher hands out the strips (a workgroup for each, or
// for every fourth where there are many, see z2d_launch_render).  (Persistent
// waves took them from a counter before; adds to one address are served one
// after another, about 12 ns each, so the 537,000 strips of a batch of 1,024
// uneven surfaces took 6.5 ms in each renderer whatever was on them: 6.39 +
// 6.58 ms, with the dispatcher 2.06 + 1.16; a page of text, 32,400 strips, 428
// us, then 110.)  Three waves per SIMD (168 VGPRs, 12 spilled): two and four
// take 1.1 times as long on a scene of every operator.  Half of the time the
// chip waits for the strips with the most draws.
//   STRIPS_SLOW     a launch over all tiles: item i is slow_list[i]
//   STRIPS_ORDERED  a launch over all tiles in J.strip_order
//   STRIPS_TILES    tiles [tile_base, tile_base + tile_count)
// the last two pass by the strips of k_render_fast.
enum : uint32_t { STRIPS_SLOW = 0, STRIPS_ORDERED = 1, STRIPS_TILES = 2 };

__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3)))
k_render(JobView J, uint32_t tile_base, uint32_t tile_count, uint32_t take) {
  __shared__ StripShared sh;
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t spt = J.strips_per_tile;
  const uint32_t n_items =
      take == STRIPS_SLOW ? load_uniform(&J.counters[9]) : tile_count * spt;
  if (blockIdx.x >= n_items) return;

  // The accumulator starts at zero and every entry leaves it at zero.
  for (uint32_t i = lane; i < (uint32_t)(STRIP_SUBROWS * ACC_WORDS); i += 64)
    (&sh.acc[0][0])[i] = 0u;
  wave_lds_sync();

  uint32_t stat_pix = 0;  // work counters (count_stats), per lane
  uint32_t stat_entries = 0, stat_unpacked = 0;
  for (uint32_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const uint32_t sidx = take == STRIPS_SLOW      ? load_uniform(&J.slow_list[item])
                          : take == STRIPS_ORDERED ? load_uniform(&J.strip_order[item])
                                                   : tile_base * spt + item;
    if (!load_uniform(&J.strip_slow[sidx])) continue;  // k_render_fast's strip
    const TileRef T = load_uniform(&J.tiles[sidx / spt]);
    const uint32_t strip = sidx % spt;
    const DevSurface S = load_uniform(&J.surfaces[T.surface]);
    const int32_t W = S.w, H = S.h;
    const int32_t tx0 = (int32_t)T.tx * TILE_W;
    const int32_t ty0 = (int32_t)T.ty * (int32_t)J.band_h + (int32_t)strip * ROWS_PER_THREAD;
    if (ty0 >= H) continue;
    const uint32_t e0 = min(load_uniform(&J.strip_cnt[sidx]), J.max_strip_entries);
    const uint32_t e1 = min(load_uniform(&J.strip_cnt[sidx + 1]), J.max_strip_entries);
    if (e0 == e1 && !S.clip) continue;
    const int32_t px = tx0 + (int32_t)lane;
    const bool col_ok = px < W;

    uint32_t pix[ROWS_PER_THREAD];
#pragma unroll
    for (int i = 0; i < ROWS_PER_THREAD; i++) {
      const int32_t py = ty0 + i;
      pix[i] = (col_ok && py < H) ? load_raw(S, (int64_t)py * W + px) : 0u;
    }
    uint32_t orig[ROWS_PER_THREAD];
#pragma unroll
    for (int i = 0; i < ROWS_PER_THREAD; i++) orig[i] = pix[i];

    for (uint32_t c = e0; c < e1; c += 64) {
      // this chunk's entries, one per lane, and which of their draws' regions
      // meet the strip (a load chain of five for each entry becomes one for 64
      // of them and two each: 1917x1080 with every operator, precision and
      // mode, 600 paths, 0.541 -> 0.527 ms)
      uint32_t g_draw = 0, g_off = 0, g_cnt = 0, g_paint = 0;
      const DevGradient *g_grad = nullptr;
      bool meets = false;
      if (c + lane < e1) {
        const BandEntry E = J.entries[J.strip_entries[c + lane]];
        const DevDraw &Dl = J.draws[E.draw];
        g_draw = E.draw;
        g_off = E.edge_off;
        g_cnt = E.edge_cnt;
        g_paint = Dl.paint;
        g_grad = J.paints[g_paint].gradient;
        meets = Dl.rx1 > tx0 && Dl.rx0 < tx0 + TILE_W && Dl.ry1 > ty0 &&
                Dl.ry0 < ty0 + ROWS_PER_THREAD;
      }
      for (uint64_t todo = __ballot(meets); todo != 0; todo &= todo - 1) {
        const uint32_t j = (uint32_t)__ffsll((unsigned long long)todo) - 1;
        const uint32_t e_off = __builtin_amdgcn_readlane(g_off, j);
        const uint32_t e_cnt = __builtin_amdgcn_readlane(g_cnt, j);
        const DevDraw D = load_uniform(&J.draws[__builtin_amdgcn_readlane(g_draw, j)]);
        const DevPaint &P = J.paints[__builtin_amdgcn_readlane(g_paint, j)];
        const DevGradient *const p_grad = reinterpret_cast<const DevGradient *>(
            (uint64_t)(uint32_t)__builtin_amdgcn_readlane((uint32_t)(uint64_t)g_grad, j) |
            ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((uint32_t)((uint64_t)g_grad >> 32), j)
             << 32));
        const uint32_t p_kind = load_uniform(&P.kind);
        const I4 p_px = load_uniform(&P.px);
        // a linear or radial gradient pattern interpolated in linear RGB with
        // its stops staged: sampled by dense_gradient, without the paint in LDS
        // (conic gradients go through paint_int: atan2 inlined here would
        // spill)
        uint32_t g_type = Z2D_GRADIENT_CONIC, g_method = 0, g_nstops = 0;
        if (p_grad) {
          g_type = load_uniform(&p_grad->type);
          g_method = load_uniform(&p_grad->method);
          g_nstops = load_uniform(&p_grad->n_stops);
        }
        const bool grad_dense = p_kind == Z2D_PATTERN_GRADIENT && g_type != Z2D_GRADIENT_CONIC &&
                                g_method == Z2D_INTERP_LINEAR_RGB && g_nstops <= STAGED_STOPS;
        StopView sv{nullptr, nullptr};
        if (p_kind != Z2D_PATTERN_OPAQUE && !grad_dense) {
          // the paint and its gradient in LDS for the samplers
          wave_lds_sync();
          constexpr uint32_t PW = sizeof(DevPaint) / 4, GW = sizeof(DevGradient) / 4;
          static_assert(PW <= 64 && GW <= 128, "staging sizes");
          if (lane < PW) reinterpret_cast<uint32_t *>(&sh.paint)[lane] =
              reinterpret_cast<const uint32_t *>(&J.paints[D.paint])[lane];
          if (p_grad) {
            const uint32_t *gs = reinterpret_cast<const uint32_t *>(p_grad);
            uint32_t *gd = reinterpret_cast<uint32_t *>(&sh.grad);
            if (lane < GW) gd[lane] = gs[lane];
            if (lane + 64 < GW) gd[lane + 64] = gs[lane + 64];
            if (lane == 0) sh.paint.gradient = &sh.grad;
          }
          wave_lds_sync();
        }
        if (p_grad) {
          const DevGradient G = load_uniform(p_grad);
          if (G.n_stops <= STAGED_STOPS) {
            wave_lds_sync();
            if (lane < G.n_stops) {
              sh.soff[lane] = G.offs[lane];
              sh.spre[lane] = G.pre[lane];
            }
            wave_lds_sync();
            sv = StopView{sh.soff, sh.spre};
          } else {
            sv = StopView{G.offs, G.pre};
          }
        }
        const int SC = D.mode == MODE_DIRECT ? 1 : 4;
        const int SR = ROWS_PER_THREAD * SC;  // sample rows in this strip
        const int32_t ys_base = ty0 * SC;
        const int32_t xs_base = tx0 * SC;
        const int32_t cols = TILE_W * SC;
        const bool direct_unb = D.mode == MODE_DIRECT && (D.flags & DRAW_UNBOUNDED);

        if (J.count_stats) stat_entries++;
        int kk[ROWS_PER_THREAD];
        if (direct_unb) {
          // Row records give the whole result of the reference's quirky
          // per-pair clears (src/internal/raster/direct.zig:88-124): cleared
          // pixels become transparent, the rest composite at full coverage
          // onto themselves or onto a cleared pixel.
          const RowRec *R = J.rows + D.row_off;
#pragma unroll
          for (int i = 0; i < ROWS_PER_THREAD; i++) {
            const int32_t py = ty0 + i;
            kk[i] = 0;
            if (!col_ok || py >= H) continue;
            const RowRec rr = load_uniform(&R[py - D.row_y0]);
            if (rr.kind == 1) continue;
            if (rr.kind == 0 || px < rr.s || px >= rr.e) {
              pix[i] = pack(I4{0, 0, 0, 0}, S.fmt);
              continue;
            }
            if (rr.kind != 2) pix[i] = pack(I4{0, 0, 0, 0}, S.fmt);
            kk[i] = 1;
          }
        } else {
          const REdge *edges = J.entry_edges + e_off;
          const uint32_t ne = e_off >= J.max_entry_edges
                                  ? 0u
                                  : min(e_cnt, J.max_entry_edges - e_off);
          const bool eo = D.rule == Z2D_FILL_EVEN_ODD;
          const bool packed = ne <= PACKED_EDGE_LIMIT;  // uniform

          // ---- phase A: winding deltas of this draw's band edges.  Each
          // crossing adds its direction at its sample column (crossings left of
          // the strip at column 0, right of it nowhere); work items are the
          // (edge, active sample row) pairs, compacted by a wave scan.
          uint32_t inner = 0;  // a crossing at a column past 0 (per lane)
          if (packed) {
            for (uint32_t c0 = 0; c0 < ne; c0 += 64) {
              const uint32_t k = c0 + lane;
              int32_t n_sr = 0, lo = 0;
              REdge ed{0.0, 0.0, 0.0, 0, 0};
              if (k < ne) {
                ed = edges[k];
                const int32_t a = max(ed.ylo, ys_base), b = min(ed.yhi2 >> 1, ys_base + SR - 1);
                if (a <= b) {
                  n_sr = b - a + 1;
                  lo = a - ys_base;
                  // every crossing right of the strip: no effect here (the
                  // crossings are monotone in the row, so the extremes are at
                  // the first and last active rows)
                  const double xa = redge_x(ed.top, ed.x_start, ed.x_inc, a);
                  const double xb = redge_x(ed.top, ed.x_start, ed.x_inc, b);
                  if (fmin(xa, xb) > (double)(xs_base + cols) + 1.0) n_sr = 0;
                }
              }
              const int32_t incl = wave_incl_scan(n_sr);
              const uint32_t total = (uint32_t)__builtin_amdgcn_readlane(incl, 63);
              if (total == 0) continue;  // uniform
              sh.u.a.cedge[lane] = ed;
              sh.clo[lane] = lo;
              const uint32_t my_off = (uint32_t)(incl - n_sr);
              sh.coff[lane] = my_off;
              // each edge marks its own items (at most SR per edge)
              for (int t = 0; t < n_sr; t++) sh.u.a.own[my_off + (uint32_t)t] = (uint8_t)lane;
              wave_lds_sync();
              for (uint32_t it = lane; it < total; it += 64) {
                const uint32_t lj = sh.u.a.own[it];
                const REdge ce = sh.u.a.cedge[lj];
                const int sr = sh.clo[lj] + (int)(it - sh.coff[lj]);
                const int32_t x = round_i32(redge_x(ce.top, ce.x_start, ce.x_inc, ys_base + sr));
                const int32_t xr = x - xs_base;
                if (xr >= cols) continue;
                const int32_t col = xr < 0 ? 0 : xr;
                inner |= (uint32_t)col;
                const int32_t dv = eo ? 1 : ((ce.yhi2 & 1) ? -1 : 1);
                atomicAdd(&sh.acc[sr][col >> 1], (col & 1) ? ((uint32_t)dv << 16) : (uint32_t)dv);
              }
              wave_lds_sync();
            }
          }

          // ---- phase B: coverage per pixel (samples covered of SC x SC), then
          // the composite in draw order.
          const RowRec *R = (D.flags & DRAW_ROWPROG) ? J.rows + D.row_off : nullptr;
          const int c_lo = (int)lane * SC;
          // every delta at column 0: each sample row's winding is the same
          // across the strip, so a pixel row's coverage is 4 samples per
          // sample row inside (no prefix sums)
          const bool uniform = packed && SC == 4 && !R && __ballot(inner != 0) == 0;
          if (uniform) {
            uint32_t w0 = 0;  // lane < 16: sample row `lane`'s column-0 word
            if (lane < (uint32_t)SR) {
              w0 = sh.acc[lane][0];
              sh.acc[lane][0] = 0u;
            }
            int32_t lo, hi;
            unpack_pair(w0, lo, hi);
            const uint64_t in_rows = __ballot(lane < (uint32_t)SR && wind_in(lo, eo));
#pragma unroll
            for (int i = 0; i < ROWS_PER_THREAD; i++)
              kk[i] = 4 * __popcll((in_rows >> (4 * i)) & 0xFull);
          } else if (packed && SC == 4) {
            if (eo) {
              if (R)
                coverage_msaa<true, true>(sh.acc, lane, xs_base, ys_base, R, D.row_y0, D.row_n, kk);
              else coverage_msaa<true, false>(sh.acc, lane, xs_base, ys_base, R, 0, 0, kk);
            } else {
              if (R)
                coverage_msaa<false, true>(sh.acc, lane, xs_base, ys_base, R, D.row_y0, D.row_n, kk);
              else coverage_msaa<false, false>(sh.acc, lane, xs_base, ys_base, R, 0, 0, kk);
            }
          } else if (packed) {
            // one sample per pixel: rows paired into one scan
    #pragma unroll
            for (int pr = 0; pr < ROWS_PER_THREAD / 2; pr++) {
              int32_t d[2];
    #pragma unroll
              for (int q = 0; q < 2; q++) {
                uint32_t *slot = &sh.acc[pr * 2 + q][lane >> 1];
                const uint32_t v = *slot;
                if ((lane & 1) == 0) *slot = 0u;
                int32_t lo, hi;
                unpack_pair(v, lo, hi);
                d[q] = (lane & 1) ? hi : lo;
              }
              const uint32_t pk = (uint32_t)d[0] + ((uint32_t)d[1] << 16);
              const uint32_t inc = (uint32_t)wave_incl_scan((int32_t)pk);
              int32_t w[2];
              unpack_pair(inc, w[0], w[1]);
    #pragma unroll
              for (int q = 0; q < 2; q++) {
                int32_t cutoff = INT32_MAX;
                if (R) {
                  const int32_t rr = ys_base + pr * 2 + q - D.row_y0;
                  if (rr >= 0 && rr < D.row_n) cutoff = load_uniform(&R[rr]).cutoff;
                }
                kk[pr * 2 + q] = (wind_in(w[q], eo) && xs_base + c_lo < cutoff) ? 1 : 0;
              }
            }
          } else {
            // more band edges than the packed deltas can hold: each lane
            // evaluates the crossings of its own sample rows
            if (J.count_stats) stat_unpacked++;
    #pragma unroll
            for (int i = 0; i < ROWS_PER_THREAD; i++) {
              int k = 0;
              for (int o = 0; o < SC; o++) {
                const int32_t ys = ys_base + i * SC + o;
                const double mid = (double)ys + 0.5;
                int32_t w[4] = {0, 0, 0, 0};
                for (uint32_t q = 0; q < ne; q++) {
                  const REdge ed = edges[q];
                  if (ys < ed.ylo || ys > (ed.yhi2 >> 1)) continue;
                  const int32_t x = round_i32(ed.x_start + (ed.x_inc * (mid - ed.top)));
                  const int32_t dv = eo ? 1 : ((ed.yhi2 & 1) ? -1 : 1);
                  const int32_t xr = x - xs_base;
    #pragma unroll
                  for (int j = 0; j < 4; j++)
                    if (j < SC && xr <= c_lo + j) w[j] += dv;
                }
                int32_t cutoff = INT32_MAX;
                if (R) {
                  const int32_t rr = ys - D.row_y0;
                  if (rr >= 0 && rr < D.row_n) cutoff = load_uniform(&R[rr]).cutoff;
                }
    #pragma unroll
                for (int j = 0; j < 4; j++)
                  if (j < SC && wind_in(w[j], eo) && xs_base + c_lo + j < cutoff) k++;
              }
              kk[i] = k;
            }
          }
          wave_lds_sync();
        }

        uint32_t n_cov = 0;
        if (D.op == Z2D_OP_SRC_OVER && D.precision == Z2D_PRECISION_INTEGER &&
            D.mode != MODE_SSAA) {
          uint32_t need = 0;  // covered pixels inside the composite region
#pragma unroll
          for (int i = 0; i < ROWS_PER_THREAD; i++) {
            const int32_t py = ty0 + i;
            if (col_ok && py < H && px >= D.rx0 && px < D.rx1 && py >= D.ry0 && py < D.ry1 &&
                kk[i] > 0)
              need |= 1u << i;
          }
          const bool solid = p_kind == Z2D_PATTERN_OPAQUE;
          const int kfull = SC * SC;
          if (__ballot(need != 0) == 0) continue;  // nothing covered in this strip (uniform)
          if (solid) {
            // the 17 possible masked sources of a solid paint
            if (lane <= 16) {
              const I4 m = (int)lane >= kfull ? p_px : mask_coverage(p_px, (int)lane);
              sh.srctab[lane] = m.r | (m.g << 8) | (m.b << 16) | (m.a << 24);
            }
            wave_lds_sync();
          } else {
            // paint samples of the covered pixels, evaluated densely: the
            // (row, lane) pairs are listed with a wave scan and taken 64 at a
            // time by one evaluation site; results go to LDS by pixel
            const int32_t np = __popc(need);
            const int32_t incl_p = wave_incl_scan(np);
            const uint32_t tot_p = (uint32_t)__builtin_amdgcn_readlane(incl_p, 63);
            uint32_t o = (uint32_t)(incl_p - np);
#pragma unroll
            for (int i = 0; i < ROWS_PER_THREAD; i++)
              if ((need >> i) & 1u) sh.u.c.plist[o++] = (uint8_t)((i << 6) | lane);
            wave_lds_sync();
            if (grad_dense) {
              const DevGradient G = load_uniform(p_grad);
              if (G.type == Z2D_GRADIENT_LINEAR)
                dense_gradient<Z2D_GRADIENT_LINEAR>(G, sh, tot_p, lane, tx0, ty0);
              else
                dense_gradient<Z2D_GRADIENT_RADIAL>(G, sh, tot_p, lane, tx0, ty0);
            } else {
#pragma unroll 1
              for (uint32_t it = lane; it < tot_p; it += 64) {
                const uint32_t v = sh.u.c.plist[it];
                const uint32_t pl = v & 63u, pi = v >> 6;
                const I4 c = paint_int(sh.paint, sv, J.blue_noise, tx0 + (int32_t)pl,
                                       ty0 + (int32_t)pi);
                sh.u.c.ppaint[pi][pl] = c.r | (c.g << 8) | (c.b << 16) | (c.a << 24);
              }
            }
            wave_lds_sync();
          }
          const bool fast_full = (D.flags & DRAW_FAST_SRC) != 0;
          // the solid fast path stores the source where coverage is full
          const uint32_t full_raw = fast_full ? pack(p_px, S.fmt) : 0u;
          src_over_rows(pix, kk, need, solid, fast_full, kfull, full_raw, sh, lane, S.fmt, n_cov);
        } else {
          // every other operator / precision / mode: one composite instance,
          // rows in a rolled loop over a copy of the strip's pixels
          uint32_t tp[ROWS_PER_THREAD];
#pragma unroll
          for (int i = 0; i < ROWS_PER_THREAD; i++) tp[i] = pix[i];
#pragma unroll 1
          for (int i = 0; i < ROWS_PER_THREAD; i++) {
            const int32_t py = ty0 + i;
            if (!col_ok || py >= H) continue;
            const bool in_region = px >= D.rx0 && px < D.rx1 && py >= D.ry0 && py < D.ry1;
            if (!in_region) continue;
            uint32_t v = tp[i];
            if (D.mode == MODE_MSAA && (D.flags & DRAW_UNBOUNDED) && msaa_preclear(D, W, px, py))
              v = pack(I4{0, 0, 0, 0}, S.fmt);
            const int k = kk[i];
            n_cov += k > 0;
            tp[i] = composite_cov(v, S.fmt, k, SC * SC, D, P, sv, J.blue_noise, px, py);
          }
#pragma unroll
          for (int i = 0; i < ROWS_PER_THREAD; i++) pix[i] = tp[i];
        }
        if (J.count_stats) stat_pix += n_cov;  // per lane
      }
    }

    if (S.clip) {
      // Clip stage: Surface.composite(dst, mask, .dst_in) after the draws.
#pragma unroll
      for (int i = 0; i < ROWS_PER_THREAD; i++) {
        const int32_t py = ty0 + i;
        if (!col_ok || py >= H) continue;
        const I4 m{0, 0, 0, S.clip[(int64_t)py * W + px]};
        pix[i] = pack(op_int(Z2D_OP_DST_IN, unpack(pix[i], S.fmt), m), S.fmt);
      }
    }
#pragma unroll
    for (int i = 0; i < ROWS_PER_THREAD; i++) {
      const int32_t py = ty0 + i;
      if (col_ok && py < H && pix[i] != orig[i]) store_raw(S, (int64_t)py * W + px, pix[i]);
    }
  }
  if (J.count_stats) strip_stats(J, stat_pix, stat_entries, stat_unpacked, lane);
}

// ---------------------------------------------------------------------------
// k_render_fast: the strip worker for the common draws (DRAW_FAST: multisample,
// src_over in integer precision of a solid paint or a linear-RGB gradient of
// at most FAST_STOPS stops, src of a solid paint, clear), over the
// strips whose every entry is such a draw (k_render skips them).  The
// coverage and composite arithmetic is k_render's; the difference is how the
// work reaches the wave: one wave per workgroup, the entries of a strip
// gathered 64 at a time into registers, and each draw's constants (its
// FastDraw block, with the gradient's stops inline) loaded one entry ahead
// of their use, so the dependent chain strip list -> entry -> draw -> paint
// -> gradient no longer stalls every entry.
// ---------------------------------------------------------------------------
struct FastShared {
  FastAcc acc;  // the entry's crossings (WindMode; zero between entries)
  union {
    struct {                             // coverage (phase A)
      // owning lane of the work items, at an owner's first item (its edge's
      // terms are read from its registers by ds_bpermute)
      uint8_t own[64 * STRIP_SUBROWS];
    } a;
    struct {                             // composite
      uint32_t ppaint[ROWS_PER_THREAD][64];  // paint samples (RGBA8)
      uint8_t plist[ROWS_PER_THREAD * 64];   // covered (row, lane) pairs
    } c;
  } u;
  FastDraw blk;  // the current entry's draw constants
  // non-zero rule: winding of the edges wholly left of the strip, as a
  // difference array over its sample rows (zero between entries)
  int32_t ldiff[STRIP_SUBROWS + 1];
  uint32_t stat_pix;  // pixel-draws of the strip (count_stats)
};

// Phase A: the crossings of a draw's band edges with SR sample rows from ys0
// on, added to acc.  An edge wholly right of the strip does nothing, one
// wholly left of it counts in every sample row it is active on (its bits of
// `left` for even-odd, per lane, to be combined over the wave; two entries of
// a row difference array for non-zero); the other edges' (edge, sample row)
// items are compacted by a wave scan and spread over the lanes.
// inner: nonzero in some lane if a crossing lies past column 0.  count
// (WIND_NZ): the difference array's high halves get the rows' items.
template <int MODE, int SR>
__device__ __forceinline__ void fast_edges(const REdge *edges, uint32_t ne, FastShared &sh,
                                           uint32_t lane, int32_t ys0, int32_t xs_base,
                                           bool count, uint32_t &inner, uint32_t &left) {
  constexpr int32_t COLS = TILE_W * 4;
  inner = 0;
  left = 0;
  for (uint32_t c0 = 0; c0 < ne; c0 += 64) {
    const uint32_t k = c0 + lane;
    int32_t n_sr = 0, lo = 0;
    REdge ed{0.0, 0.0, 0.0, 0, 0};
    if (k < ne) {
      ed = edges[k];
      const int32_t a = max(ed.ylo, ys0), b = min(ed.yhi2 >> 1, ys0 + SR - 1);
      if (a <= b) {
        n_sr = b - a + 1;
        lo = a - ys0;
        // the crossings are monotone in the row, so their extremes are at
        // the first and last active rows
        const double xa = redge_x(ed.top, ed.x_start, ed.x_inc, a);
        const double xb = redge_x(ed.top, ed.x_start, ed.x_inc, b);
        const double xr = (double)(xs_base + COLS) + 1.0, xl = (double)xs_base - 1.0;
        if (xa > xr && xb > xr) {
          n_sr = 0;
        } else if (xa < xl && xb < xl) {  // (rounded below the first sample column)
          if (MODE == WIND_EO) {
            left ^= ((1u << n_sr) - 1u) << lo;
          } else {
            const int32_t dv = (ed.yhi2 & 1) ? -1 : 1;
            atomicAdd(&sh.ldiff[lo], dv);
            atomicAdd(&sh.ldiff[lo + n_sr], -dv);
            left = 1;
          }
          n_sr = 0;
        }
      }
    }
    const int32_t incl = wave_incl_scan(n_sr);
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane(incl, 63);
    if (total == 0) continue;  // uniform
    if (MODE == WIND_NZ && count && n_sr > 0) {
      atomicAdd(&sh.ldiff[lo], 1 << 16);
      atomicAdd(&sh.ldiff[lo + n_sr], -(1 << 16));
    }
    const uint32_t my_off = (uint32_t)(incl - n_sr);
    // an owner's first item, first row and direction
    const uint32_t info = ((ed.yhi2 & 1) ? 0x80000000u : 0u) | ((uint32_t)lo << 16) | my_off;
    // owners in lane order have items in order: each marks its first item,
    // and an item's owner is the largest mark up to it
    reinterpret_cast<uint4 *>(sh.u.a.own)[lane] = make_uint4(0u, 0u, 0u, 0u);
    wave_lds_sync();
    if (n_sr > 0) sh.u.a.own[my_off] = (uint8_t)lane;
    wave_lds_sync();
    uint32_t before = 0;  // the owner of the last item of the round before
    // every lane takes part in each round's scan and register reads (the
    // owner of an item may be a lane with no item of its own this round)
    for (uint32_t it0 = 0; it0 < total; it0 += 64) {
      const uint32_t it = it0 + lane;
      const uint32_t lj = max(
          (uint32_t)wave_max_scan((int32_t)sh.u.a.own[it & (64u * STRIP_SUBROWS - 1u)]), before);
      before = (uint32_t)__builtin_amdgcn_readlane((int32_t)lj, 63);
      const uint32_t q = lane_read_u32(info, lj);
      const double etop = lane_read_f64(ed.top, lj), exs = lane_read_f64(ed.x_start, lj),
                   exi = lane_read_f64(ed.x_inc, lj);
      if (it >= total) continue;
      const uint32_t sr = ((q >> 16) & 0x7FFFu) + (it - (q & 0xFFFFu));
      const int32_t x = round_i32(redge_x(etop, exs, exi, ys0 + (int32_t)sr));
      const int32_t xr = x - xs_base;
      if (xr >= COLS) continue;
      const int32_t col = xr < 0 ? 0 : xr;
      inner |= (uint32_t)col;
      if (MODE == WIND_EO) {
        atomicXor(&sh.acc[0][col], 1u << sr);
      } else {
        const uint32_t dv = (q >> 31) ? 0xFFFFFFFFu : 1u;
        if (MODE == WIND_NZ)
          atomicAdd(&sh.acc[sr >> 2][col], dv << (8u * (sr & 3u)));
        else
          atomicAdd(&sh.acc[sr >> 1][col], dv << (16u * (sr & 1u)));
      }
    }
    wave_lds_sync();
  }
}

// The non-zero rule's left edges: each sample row's winding (and the row's
// items, where they were counted, in the high half) from the difference array
// (cleared), in lane `row`, 0 in the others.
__device__ __forceinline__ int32_t left_windings(FastShared &sh, uint32_t lane) {
  wave_lds_sync();
  int32_t dl = 0;
  if (lane <= (uint32_t)STRIP_SUBROWS) {
    dl = lane < (uint32_t)STRIP_SUBROWS ? sh.ldiff[lane] : 0;
    sh.ldiff[lane] = 0;
  }
  const int32_t wl = wave_incl_scan(dl);
  return lane < (uint32_t)STRIP_SUBROWS ? wl : 0;
}

// The non-zero rule's coverage of a strip whose windings may not fit a byte:
// its two halves one after the other, two sample rows to a word.
__device__ __forceinline__ void coverage_halves(const REdge *edges, uint32_t ne, FastShared &sh,
                                             uint32_t lane, int32_t ys_base, int32_t xs_base,
                                             int *kk) {
#pragma unroll 1
  for (int h = 0; h < 2; h++) {
    uint32_t inner, left;
    fast_edges<WIND_NZ16, STRIP_SUBROWS / 2>(edges, ne, sh, lane,
                                             ys_base + h * (STRIP_SUBROWS / 2), xs_base, false,
                                             inner, left);
    const int32_t wl = left_windings(sh, lane);
    if (wl != 0 && lane < (uint32_t)STRIP_SUBROWS / 2)
      atomicAdd(&sh.acc[lane >> 1][0], (uint32_t)wl << (16u * (lane & 1u)));
    wave_lds_sync();
    int k2[ROWS_PER_THREAD / 2];
    coverage_nz16(sh.acc, lane, k2);
    if (h == 0) {
      kk[0] = k2[0];
      kk[1] = k2[1];
    } else {
      kk[2] = k2[0];
      kk[3] = k2[1];
    }
    wave_lds_sync();
  }
}

// Gradient.getOffset (src/gradient.zig:349-375, :605-652, :731-742) on a
// fast draw's block: the arithmetic of linear_offset / radial_offset /
// conic_offset, term for term.
__device__ __forceinline__ float fast_linear_offset(const FastDraw &g, int x, int y) {
  double px = (double)x + 0.5, py = (double)y + 0.5;
  if (!g.identity) user_to_device(g.m, px, py);
  if (g.p[3] != 0.0) return -1.0f;
  double spx = px - g.gx, spy = py - g.gy;
  double dt = 0.0;
  dt += g.p[0] * spx;
  dt += g.p[1] * spy;
  return (float)dclamp01(dt * g.p[2]);
}
__device__ __forceinline__ float fast_radial_offset(const FastDraw &g, int x, int y) {
  double px = (double)x + 0.5, py = (double)y + 0.5;
  const double r1 = g.p[0], r2 = g.p[1], cdx = g.p[2], cdy = g.p[3], dr = g.p[4],
               min_dr = g.p[5], a = g.p[6], inv_a = g.p[7];
  if (r1 == 0.0 && r2 == 0.0) return -1.0f;
  if (!g.identity) user_to_device(g.m, px, py);
  double pdx = px - g.gx, pdy = py - g.gy;
  double b = 0.0;
  b += pdx * cdx;
  b += pdy * cdy;
  b += r1 * dr;
  double c = 0.0;
  c += pdx * pdx;
  c += pdy * pdy;
  c += (-r1) * r1;
  if (a == 0.0) {
    if (b == 0.0) return -1.0f;
    double t = 0.5 * c / b;
    if (t * dr >= min_dr) return (float)dclamp01(t);
    return -1.0f;
  }
  double discr = 0.0;
  discr += b * b;
  discr += a * (-c);
  if (discr >= 0.0) {
    double sq = sqrt(discr);
    double t0 = (b + sq) * inv_a;
    double t1 = (b - sq) * inv_a;
    if (t0 * dr >= min_dr) return (float)dclamp01(t0);
    if (t1 * dr >= min_dr) return (float)dclamp01(t1);
  }
  return -1.0f;
}
__device__ __forceinline__ float fast_conic_offset(const FastDraw &g, int x, int y) {
  double px = (double)x + 0.5, py = (double)y + 0.5;
  const double two_pi = 3.14159265358979323846 * 2.0;
  if (!g.identity) user_to_device(g.m, px, py);
  double ang = zmodd(zatan2<true>(py - g.gy, px - g.gx) - g.p[0], two_pi);
  return (float)(ang / two_pi);
}

// f2u8 of a value below 65536.
__device__ __forceinline__ uint32_t f2u8_sat(float v) { return cvt_u32_sat(v + 0x1.fffffep-2f); }

// Paint samples of the covered pixels listed in plist (as dense_gradient).
template <uint32_t PF>
__device__ __forceinline__ void fast_gradient(const FastDraw &B, FastShared &sh, uint32_t tot_p,
                                              uint32_t lane, int32_t tx0, int32_t ty0) {
  const uint32_t n_stops = min(__builtin_amdgcn_readfirstlane(B.n_stops), FAST_STOPS);
#pragma unroll 1
  for (uint32_t it = lane; it < tot_p; it += 64) {
    // the gradient's constants are read from the block in LDS on each pass
    // instead of being held in registers across the loop
    asm volatile("" ::: "memory");
    const uint32_t v = sh.u.c.plist[it];
    const uint32_t pl = v & 63u, pi = v >> 6;
    const int32_t x = tx0 + (int32_t)pl, y = ty0 + (int32_t)pi;
    float off;
    if constexpr (PF == FAST_PAINT_LINEAR)
      off = fast_linear_offset(B, x, y);
    else if constexpr (PF == FAST_PAINT_RADIAL)
      off = fast_radial_offset(B, x, y);
    else
      off = fast_conic_offset(B, x, y);
    int i0, i1;
    float t;
    bool transparent;
    stops_find8(B.offs, n_stops, off, i0, i1, t, transparent);
    // both stop colors read whole (i0, i1 are valid indices either way); a
    // transparent sample is all zeros.  The colors are premultiplied and in
    // [0, 1], the interpolation of two of them at most a rounding above.
    const float4 A = B.pre[i0], C2 = B.pre[i1];
    const uint32_t r = f2u8_sat(255.0f * lerpf_(A.x, C2.x, t));
    const uint32_t g = f2u8_sat(255.0f * lerpf_(A.y, C2.y, t));
    const uint32_t b = f2u8_sat(255.0f * lerpf_(A.z, C2.z, t));
    const uint32_t a = f2u8_sat(255.0f * lerpf_(A.w, C2.w, t));
    sh.u.c.ppaint[pi][pl] = transparent ? 0u : (r | (g << 8) | (b << 16) | (a << 24));
  }
}

// Bound by VALU issue and, at few waves, by latency: six waves per SIMD (79
// VGPRs and 5.9 KB of LDS) take 0.78 ms for the 4K scene of 10,000 paths, five
// 0.81, four 0.89.  No register is spilled: what lives from entry to entry
// leaves the registers while a gradient is evaluated, and the formats other
// than RGBA8 are read and written in a loop over LDS (9 spilled before, a
// third more code; a page of text 0.087 -> 0.082 ms).  A src or a clear takes
// one more branch here; its strips were k_render's before (1,024 surfaces of
// every format, one op in ten of them: 2.97 -> 1.94 ms for both kernels).
// Strips are handed out as in k_render (take is never STRIPS_SLOW here).
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(6)))
k_render_fast(JobView J, uint32_t tile_base, uint32_t tile_count, uint32_t first,
              uint32_t take) {
  __shared__ FastShared sh;
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t spt = J.strips_per_tile;
  const uint32_t item = first + blockIdx.x;
  if (item >= tile_count * spt) return;
  const uint32_t sidx =
      take == STRIPS_ORDERED ? load_uniform(&J.strip_order[item]) : tile_base * spt + item;
  if (load_uniform(&J.strip_slow[sidx])) return;  // k_render's strip

  uint32_t stat_entries = 0;  // work counter (count_stats; the pixels' in LDS)
  {
    const TileRef T = load_uniform(&J.tiles[sidx / spt]);
    const uint32_t strip = sidx % spt;
    const DevSurface S = load_uniform(&J.surfaces[T.surface]);
    const int32_t W = S.w, H = S.h;
    const int32_t tx0 = (int32_t)T.tx * TILE_W;
    const int32_t ty0 = (int32_t)T.ty * (int32_t)J.band_h + (int32_t)strip * ROWS_PER_THREAD;
    if (ty0 >= H) return;
    const uint32_t e0 = min(load_uniform(&J.strip_cnt[sidx]), J.max_strip_entries);
    const uint32_t e1 = min(load_uniform(&J.strip_cnt[sidx + 1]), J.max_strip_entries);
    if (e0 == e1 && !S.clip) return;
    // the winding deltas start at zero and every entry leaves them at zero
    for (uint32_t i = lane; i < (uint32_t)(FAST_ACC_ROWS * FAST_ACC_COLS / 4); i += 64)
      reinterpret_cast<uint4 *>(&sh.acc[0][0])[i] = make_uint4(0u, 0u, 0u, 0u);
    if (lane <= (uint32_t)STRIP_SUBROWS) sh.ldiff[lane] = 0;
    if (lane == 0) sh.stat_pix = 0u;
    wave_lds_sync();
    const int32_t px = tx0 + (int32_t)lane;
    const bool col_ok = px < W;
    // the strip's pixels, from here to the store below as channel pairs
    Px2 pix[ROWS_PER_THREAD];
    uint32_t dirty = 0;  // byte i nonzero: a draw composited on row i
    const bool rgba8 = S.fmt == Z2D_FORMAT_RGBA;  // uniform: no format switch per row
    if (rgba8) {
#pragma unroll
      for (int i = 0; i < ROWS_PER_THREAD; i++) {
        const int32_t py = ty0 + i;
        pix[i] = px2_rgba8((col_ok && py < H)
                               ? reinterpret_cast<const uint32_t *>(S.data)[(int64_t)py * W + px]
                               : 0u);
      }
    } else {
      // (a loop through LDS: the format switches once in the code, not per row)
#pragma unroll 1
      for (int i = 0; i < ROWS_PER_THREAD; i++) {
        const int32_t py = ty0 + i;
        sh.u.c.ppaint[i][lane] = px2_to_rgba8(
            px2_unpack((col_ok && py < H) ? load_raw(S, (int64_t)py * W + px) : 0u, S.fmt));
      }
#pragma unroll
      for (int i = 0; i < ROWS_PER_THREAD; i++) pix[i] = px2_rgba8(sh.u.c.ppaint[i][lane]);
    }
    // packed alpha surfaces hold fewer bits than a lane between draws
    const int a_bits = S.fmt >= Z2D_FORMAT_ALPHA4 ? fmt_bits(S.fmt) : 8;
    const int32_t ys_base = ty0 * 4, xs_base = tx0 * 4;

    for (uint32_t c = e0; c < e1; c += 64) {
      // this chunk's entries, one per lane
      const uint32_t nc = min(64u, e1 - c);
      uint32_t g_draw = 0, g_off = 0, g_cnt = 0;
      if (lane < nc) {
        const BandEntry E = J.entries[J.strip_entries[c + lane]];
        g_draw = E.draw;
        g_off = E.edge_off;
        g_cnt = E.edge_off >= J.max_entry_edges ? 0u
                                                : min(E.edge_cnt, J.max_entry_edges - E.edge_off);
      }
      uint4 nb = make_uint4(0u, 0u, 0u, 0u);  // the next entry's block, 16 B per lane
      {
        const uint32_t d0 = __builtin_amdgcn_readlane(g_draw, 0);
        if (lane < FAST_DRAW_CHUNKS) nb = reinterpret_cast<const uint4 *>(J.fast + d0)[lane];
      }
      for (uint32_t j = 0; j < nc; j++) {
        // entry j's block to LDS, entry j+1's in flight
        wave_lds_sync();
        if (lane < FAST_DRAW_CHUNKS) reinterpret_cast<uint4 *>(&sh.blk)[lane] = nb;
        wave_lds_sync();
        // its region, rule and paint kind straight from the lanes holding them
        const int32_t rx0 = __builtin_amdgcn_readlane(nb.x, 0),
                      rx1 = __builtin_amdgcn_readlane(nb.y, 0),
                      ry0 = __builtin_amdgcn_readlane(nb.z, 0),
                      ry1 = __builtin_amdgcn_readlane(nb.w, 0);
        const bool eo = __builtin_amdgcn_readlane(nb.x, 1) == Z2D_FILL_EVEN_ODD;
        const uint32_t pf = __builtin_amdgcn_readlane(nb.y, 1);
        if (j + 1 < nc) {
          const uint32_t dn = __builtin_amdgcn_readlane(g_draw, j + 1);
          if (lane < FAST_DRAW_CHUNKS) nb = reinterpret_cast<const uint4 *>(J.fast + dn)[lane];
        }
        const FastDraw &B = sh.blk;
        // uniform: the draw's composite region misses this strip
        if (rx1 <= tx0 || rx0 >= tx0 + TILE_W) continue;
        if (ry1 <= ty0 || ry0 >= ty0 + ROWS_PER_THREAD) continue;
        const uint32_t ne = __builtin_amdgcn_readlane(g_cnt, j);
        const REdge *edges = J.entry_edges + __builtin_amdgcn_readlane(g_off, j);
        if (J.count_stats) stat_entries++;

        // ---- phases A and B: covered samples per pixel
        int kk[ROWS_PER_THREAD];
        uint32_t inner, left;
        if (eo) {
          fast_edges<WIND_EO, STRIP_SUBROWS>(edges, ne, sh, lane, ys_base, xs_base, false, inner,
                                             left);
          if (__ballot(left != 0))  // parity of the left edges over the wave
            left = (uint32_t)__builtin_amdgcn_readlane((int32_t)wave_xor_scan(left), 63);
          coverage_eo(sh.acc, lane, left, kk);
        } else {
          // |winding| <= half the edges (contours return to their start), and
          // in a sample row <= that left of the strip plus the row's
          // crossings in it.  (By the strip's edges instead of its rows'
          // crossings the strips of a stroke's many short edges were taken
          // three times: 47 served requests of 91 px, 223 us of this kernel,
          // 186 now; 64 surfaces of 128 px one by one, 158 us each and 133.)
          const bool many = ne > 254u;
          fast_edges<WIND_NZ, STRIP_SUBROWS>(edges, ne, sh, lane, ys_base, xs_base, many, inner,
                                             left);
          int32_t most = 0;
          if (many || __ballot(left != 0)) {
            int32_t wl, cross;
            unpack_pair((uint32_t)left_windings(sh, lane), wl, cross);
            most = abs(wl) + cross;
            if (wl != 0) atomicAdd(&sh.acc[lane >> 2][0], (uint32_t)wl << (8u * (lane & 3u)));
          }
          wave_lds_sync();
          if (many && wave_max_i32(most) > 127) {
#pragma unroll
            for (int i = 0; i < FAST_ACC_ROWS; i++)
              *reinterpret_cast<uint4 *>(&sh.acc[i][lane * 4]) = make_uint4(0u, 0u, 0u, 0u);
            wave_lds_sync();
            coverage_halves(edges, ne, sh, lane, ys_base, xs_base, kk);
          } else if (__ballot(inner != 0) == 0) {
            // every crossing at column 0: uniform winding across each sample
            // row (lane = sample row; every fourth lane clears the word)
            uint32_t w0 = 0;
            if (lane < (uint32_t)STRIP_SUBROWS) w0 = sh.acc[lane >> 2][0];
            wave_lds_sync();
            if (lane < (uint32_t)STRIP_SUBROWS && !(lane & 3u)) sh.acc[lane >> 2][0] = 0u;
            const bool in = (((w0 + 0x80808080u) >> (8u * (lane & 3u))) & 0xFFu) != 0x80u;
            const uint64_t in_rows = __ballot(lane < (uint32_t)STRIP_SUBROWS && in);
#pragma unroll
            for (int i = 0; i < ROWS_PER_THREAD; i++)
              kk[i] = 4 * __popcll((in_rows >> (4 * i)) & 0xFull);
          } else {
            coverage_nz(sh.acc, lane, kk);
          }
        }
        wave_lds_sync();

        // ---- composite: src_over of the masked paint.  A draw's region lies
        // on the surface; outside it (columns [rx0, rx1), rows [r_lo, r_hi)
        // of the strip) the coverage is taken as 0, whose source is 0 and
        // leaves the pixel as it is, so every row is composited without a
        // branch.
        const int32_t r_lo = max(ry0, ty0) - ty0, r_hi = min(ry1, ty0 + ROWS_PER_THREAD) - ty0;
        const bool in_col = px >= rx0 && px < rx1;
        uint32_t cov = 0;  // row i's coverage in byte i
#pragma unroll
        for (int i = 0; i < ROWS_PER_THREAD; i++) {
          if (!(in_col && i >= r_lo && i < r_hi)) kk[i] = 0;
          cov |= (uint32_t)kk[i] << (8 * i);
        }
        if (__ballot(cov != 0) == 0) continue;  // nothing covered in this strip (uniform)
        dirty |= cov;
        const bool solid = pf == FAST_PAINT_SOLID || pf == FAST_PAINT_REPLACE;
        if (!solid || J.count_stats) {
          uint32_t need = 0;
#pragma unroll
          for (int i = 0; i < ROWS_PER_THREAD; i++) need |= (kk[i] > 0 ? 1u : 0u) << i;
          if (J.count_stats) {
            // one lane's add (the compiler takes 64 lanes' adds to one address
            // one after another: 8 served requests of 256 px, 208 us of this
            // kernel, 165 now)
            uint32_t n_cov = 0;
#pragma unroll
            for (int i = 0; i < ROWS_PER_THREAD; i++)
              n_cov += (uint32_t)__popcll(__ballot(kk[i] > 0));
            if (lane == 0) atomicAdd(&sh.stat_pix, n_cov);
          }
          if (!solid) {
            const int32_t np = __popc(need);
            const int32_t incl_p = wave_incl_scan(np);
            const uint32_t tot_p = (uint32_t)__builtin_amdgcn_readlane(incl_p, 63);
            uint32_t o = (uint32_t)(incl_p - np);
#pragma unroll
            for (int i = 0; i < ROWS_PER_THREAD; i++)
              if ((need >> i) & 1u) sh.u.c.plist[o++] = (uint8_t)((i << 6) | lane);
            wave_lds_sync();
            // the gradients' 64-bit arithmetic needs the registers of the
            // strip's pixels: they wait in a row of acc, zero again after
            uint4 &kept = *reinterpret_cast<uint4 *>(&sh.acc[0][lane * 4]);
            kept = make_uint4(px2_to_rgba8(pix[0]), px2_to_rgba8(pix[1]), px2_to_rgba8(pix[2]),
                              px2_to_rgba8(pix[3]));
            if (pf == FAST_PAINT_LINEAR)
              fast_gradient<FAST_PAINT_LINEAR>(B, sh, tot_p, lane, tx0, ty0);
            else if (pf == FAST_PAINT_RADIAL)
              fast_gradient<FAST_PAINT_RADIAL>(B, sh, tot_p, lane, tx0, ty0);
            else
              fast_gradient<FAST_PAINT_CONIC>(B, sh, tot_p, lane, tx0, ty0);
            wave_lds_sync();
            const uint4 back = kept;
            pix[0] = px2_rgba8(back.x);
            pix[1] = px2_rgba8(back.y);
            pix[2] = px2_rgba8(back.z);
            pix[3] = px2_rgba8(back.w);
            kept = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
            for (int i = 0; i < ROWS_PER_THREAD; i++) kk[i] = (int)((cov >> (8 * i)) & 0xFFu);
          }
        }
        if (pf == FAST_PAINT_REPLACE) {
          // over a transparent pixel src_over gives the source, whatever it
          // is; a format without alpha reads back as opaque
          const uint32_t under =
              S.fmt == Z2D_FORMAT_RGB || S.fmt == Z2D_FORMAT_XRGB ? 0x00FF0000u : 0u;
#pragma unroll
          for (int i = 0; i < ROWS_PER_THREAD; i++) {
            pix[i].rb = kk[i] > 0 ? 0u : pix[i].rb;
            pix[i].ga = kk[i] > 0 ? under : pix[i].ga;
          }
        }
        if (solid) {
#pragma unroll
          for (int i = 0; i < ROWS_PER_THREAD; i++)
            pix[i] = px2_src_over(pix[i], B.srctab[kk[i]]);
        } else {
          // (a pixel without coverage reads a stale sample, masked to 0)
#pragma unroll
          for (int i = 0; i < ROWS_PER_THREAD; i++)
            pix[i] = px2_src_over(pix[i], mask_coverage_rgba8(sh.u.c.ppaint[i][lane], kk[i]));
        }
        if (a_bits < 8) {  // uniform
#pragma unroll
          for (int i = 0; i < ROWS_PER_THREAD; i++)
            pix[i].ga = alpha_up8(alpha_down(pix[i].ga >> 16, a_bits), a_bits) << 16;
        }
      }
    }

    if (rgba8 && !S.clip) {
#pragma unroll
      for (int i = 0; i < ROWS_PER_THREAD; i++) {
        const int32_t py = ty0 + i;
        if (col_ok && py < H && ((dirty >> (8 * i)) & 0xFFu))
          reinterpret_cast<uint32_t *>(S.data)[(int64_t)py * W + px] = px2_to_rgba8(pix[i]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < ROWS_PER_THREAD; i++) sh.u.c.ppaint[i][lane] = px2_to_rgba8(pix[i]);
#pragma unroll 1
      for (int i = 0; i < ROWS_PER_THREAD; i++) {
        const int32_t py = ty0 + i;
        if (!col_ok || py >= H) continue;
        uint32_t raw = px2_pack(px2_rgba8(sh.u.c.ppaint[i][lane]), S.fmt);
        bool changed = ((dirty >> (8 * i)) & 0xFFu) != 0;
        if (S.clip) {
          // Clip stage: Surface.composite(dst, mask, .dst_in) after the draws.
          const I4 m{0, 0, 0, S.clip[(int64_t)py * W + px]};
          const uint32_t before = raw;
          raw = pack(op_int(Z2D_OP_DST_IN, unpack(raw, S.fmt), m), S.fmt);
          changed |= raw != before;
        }
        if (changed) store_raw(S, (int64_t)py * W + px, raw);
      }
    }
  }
  if (J.count_stats) {
    wave_lds_sync();
    strip_stats(J, lane == 0 ? sh.stat_pix : 0u, stat_entries, 0u, lane);
  }
}

// ---------------------------------------------------------------------------
// k_grad_setup: per-stop interpolation colors of every gradient of a job.
// ---------------------------------------------------------------------------
__global__ void k_grad_setup(DevGradient *grads, uint32_t n_grads) {
  const uint32_t gi = blockIdx.x * blockDim.x + threadIdx.x;
  if (gi >= n_grads) return;
  const DevGradient &g = grads[gi];
  float4 *pre = const_cast<float4 *>(g.pre);
  for (uint32_t i = 0; i < g.n_stops; i++) pre[i] = stop_interp_color(g, g.stops[i]);
}

// ---------------------------------------------------------------------------
// k_composite: SurfaceCompositor.run batches.
// ---------------------------------------------------------------------------
__device__ __forceinline__ I4 comp_param_int(const DevCompParam &p, const CompJob &J, int64_t row_off,
                                             int32_t j, int x, int y) {
  switch (p.kind) {
    case Z2D_PARAM_PIXEL: return p.px;
    case Z2D_PARAM_SURFACE: {
      int64_t idx = p.base + row_off + j;
      if (idx < 0 || idx >= (int64_t)p.surf.w * p.surf.h) return I4{0, 0, 0, 0};
      return unpack(load_raw(p.surf, idx), p.surf.fmt);
    }
    default: return paint_int(*p.paint, paint_stops(*p.paint), J.blue_noise, x, y);
  }
}
__device__ __forceinline__ F4 comp_param_float(const DevCompParam &p, const CompJob &J,
                                               int64_t row_off, int32_t j, int x, int y) {
  switch (p.kind) {
    case Z2D_PARAM_PIXEL: return decode_raw(p.px);
    case Z2D_PARAM_SURFACE: {
      int64_t idx = p.base + row_off + j;
      if (idx < 0 || idx >= (int64_t)p.surf.w * p.surf.h) return F4{0, 0, 0, 0};
      return decode_raw(unpack(load_raw(p.surf, idx), p.surf.fmt));
    }
    default: return paint_float(*p.paint, paint_stops(*p.paint), J.blue_noise, x, y);
  }
}

__device__ __forceinline__ uint32_t comp_pixel(const CompJob &J, int32_t r, int32_t j,
                                               uint32_t dst_raw) {
  const int x = J.x0 + j, y = J.y0 + r;
  if (J.precision == Z2D_PRECISION_INTEGER) {
    I4 cur{0, 0, 0, 0};
    for (uint32_t k = 0; k < J.n_ops; k++) {
      const DevCompOp &o = J.ops[k];
      I4 s = o.src.kind == Z2D_PARAM_NONE
                 ? cur
                 : comp_param_int(o.src, J, (int64_t)r * o.src.surf.w, j, x, y);
      I4 d = o.dst.kind == Z2D_PARAM_NONE
                 ? unpack(dst_raw, J.dst.fmt)
                 : comp_param_int(o.dst, J, (int64_t)r * o.dst.surf.w, j, x, y);
      cur = op_int(o.op, d, s);
    }
    return pack(cur, J.out.fmt);
  }
  F4 cur{0, 0, 0, 0};
  for (uint32_t k = 0; k < J.n_ops; k++) {
    const DevCompOp &o = J.ops[k];
    F4 s = o.src.kind == Z2D_PARAM_NONE
               ? cur
               : comp_param_float(o.src, J, (int64_t)r * o.src.surf.w, j, x, y);
    F4 d = o.dst.kind == Z2D_PARAM_NONE
               ? decode_raw(unpack(dst_raw, J.dst.fmt))
               : comp_param_float(o.dst, J, (int64_t)r * o.dst.surf.w, j, x, y);
    cur = op_float(o.op, d, s);
  }
  return pack(encode_raw(cur), J.out.fmt);
}

// Generic path: one pixel per lane, rows on blockIdx.y (strided).
__global__ void k_composite(const CompJob *__restrict__ Jp) {
  const CompJob &J = *Jp;
  for (int32_t r = blockIdx.y; r < J.height; r += gridDim.y) {
    for (int32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < J.width;
         j += gridDim.x * blockDim.x) {
      const int64_t didx = (int64_t)(J.y0 + r) * J.dst.w + (J.x0 + j);
      const uint32_t v = comp_pixel(J, r, j, load_raw(J.dst, didx));
      if (J.out.fmt >= Z2D_FORMAT_ALPHA4 && J.out.fmt <= Z2D_FORMAT_ALPHA1)
        store_raw(J.out, didx, v);
      else if (J.out.fmt == Z2D_FORMAT_ALPHA8)
        J.out.data[didx] = (uint8_t)v;
      else
        reinterpret_cast<uint32_t *>(J.out.data)[didx] = v;
    }
  }
}

// Streaming path for whole-surface 4-byte-format batches whose surface
// sources start at the same pixel as the destination: 4 pixels per lane via
// 16-byte loads/stores, grid-stride over the flat pixel range.
__global__ void __launch_bounds__(256) k_composite_stream(const CompJob *__restrict__ Jp,
                                                          uint64_t n_quads) {
  const CompJob &J = *Jp;
  const uint32_t *dst = reinterpret_cast<const uint32_t *>(J.dst.data);
  uint32_t *out = reinterpret_cast<uint32_t *>(J.out.data);
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n_quads; q += stride) {
    const uint64_t p0 = q * 4;
    const uint4 dv = *reinterpret_cast<const uint4 *>(dst + p0);
    uint32_t dvals[4] = {dv.x, dv.y, dv.z, dv.w};
    uint32_t res[4];
    const int32_t W = J.dst.w;
    const int32_t r = (int32_t)(p0 / (uint64_t)W);
    const int32_t j = (int32_t)(p0 - (uint64_t)r * W);
#pragma unroll
    for (int l = 0; l < 4; l++) {
      // the flat index maps to (r, j + l) with j + l < W because W % 4 == 0
      res[l] = comp_pixel(J, r, j + l, dvals[l]);
    }
    *reinterpret_cast<uint4 *>(out + p0) = make_uint4(res[0], res[1], res[2], res[3]);
  }
}

// ---------------------------------------------------------------------------
// k_composite_quad: the compositor of one operator, specialised per operator.
// The operator is a template parameter (one instance per operator and
// precision, chosen once per launch), 4-byte formats unpack through a byte
// permute whose selector is in a scalar register, and every source is one
// 16-byte (or 4-byte for alpha8) load per four pixels.  Per pixel it computes what comp_pixel
// computes for the same batch.  Bound by HBM for the integer operators.  The
// loads take any pixel's address (the hardware asks for 4-byte alignment at
// most), so a region at an offset and surfaces of any width come here too:
// overlay through an alpha8 mask at 3837x2159, one pixel per lane in
// k_composite before, 142.7 us a pass then and 48.5 now (start and end of the
// call included).  WHOLE: a flat run of whole quads on 16-byte addresses, with
// no last quad to look at.  The one loop for both cost such surfaces up to 40%
// (clear at 4096x4096 2.98 TB/s, 4.88 with the loop of its own; overlay 3.64
// and 3.90, darken 4.35 and 4.62, exclusion 3.93 and 4.21).
// ---------------------------------------------------------------------------
// A format's byte order as the selectors of a byte permute, to and from RGBA8
// (0x0C selects a zero byte, 0x0D one of 255).
struct Fmt32 {
  uint32_t to, from;
};
__device__ __forceinline__ Fmt32 fmt32(uint32_t fmt) {
  switch (fmt) {
    case Z2D_FORMAT_ARGB: return Fmt32{0x03000102u, 0x03000102u};
    case Z2D_FORMAT_XRGB: return Fmt32{0x0D000102u, 0x0C000102u};
    case Z2D_FORMAT_RGB: return Fmt32{0x0D020100u, 0x0C020100u};
    default: return Fmt32{0x03020100u, 0x03020100u};
  }
}
// unpack / pack of the four 4-byte formats
__device__ __forceinline__ I4 unpack32(uint32_t raw, Fmt32 f) {
  const uint32_t w = __builtin_amdgcn_perm(raw, raw, f.to);
  return I4{w & 0xFFu, (w >> 8) & 0xFFu, (w >> 16) & 0xFFu, w >> 24};
}
__device__ __forceinline__ uint32_t pack32(I4 v, Fmt32 f) {
  const uint32_t w =
      (v.r & 0xFFu) | ((v.g & 0xFFu) << 8) | ((v.b & 0xFFu) << 16) | ((v.a & 0xFFu) << 24);
  return __builtin_amdgcn_perm(w, w, f.from);
}
// Four consecutive pixels (n of them in the last quad of a row, the others
// read as 0): 16 and 4 bytes at any pixel's address, one load each.  WHOLE:
// always four, on addresses of 16 (4) bytes.
struct __attribute__((packed, aligned(4))) Quad32 {
  uint32_t v[4];
};
template <bool WHOLE>
__device__ __forceinline__ Quad32 quad_words(const uint32_t *p, uint32_t n) {
  if (WHOLE) {
    const uint4 v = *reinterpret_cast<const uint4 *>(p);
    return Quad32{{v.x, v.y, v.z, v.w}};
  }
  if (n >= 4) return *reinterpret_cast<const Quad32 *>(p);
  Quad32 o{};
#pragma unroll
  for (uint32_t l = 0; l < 3; l++)
    if (l < n) o.v[l] = p[l];
  return o;
}
template <bool WHOLE>
__device__ __forceinline__ uint32_t quad_bytes(const uint8_t *p, uint32_t n) {
  if (WHOLE) return *reinterpret_cast<const uint32_t *>(p);
  uint32_t v = 0;
  if (n >= 4) {
    __builtin_memcpy(&v, p, 4);
    return v;
  }
#pragma unroll
  for (uint32_t l = 0; l < 3; l++)
    if (l < n) v |= (uint32_t)p[l] << (8 * l);
  return v;
}
template <bool WHOLE>
__device__ __forceinline__ void quad_load(const QuadSrc &s, Fmt32 f, uint32_t row, uint64_t i,
                                          uint32_t n, I4 (&o)[4]) {
  if (s.kind == QUAD_SURF32) {
    const Quad32 v =
        quad_words<WHOLE>(reinterpret_cast<const uint32_t *>(s.data) + row * s.pitch + i, n);
#pragma unroll
    for (int l = 0; l < 4; l++) o[l] = unpack32(v.v[l], f);
  } else if (s.kind == QUAD_ALPHA8) {
    const uint32_t v = quad_bytes<WHOLE>(s.data + row * s.pitch + i, n);
#pragma unroll
    for (int l = 0; l < 4; l++) o[l] = I4{0u, 0u, 0u, (v >> (8 * l)) & 0xFFu};
  } else {
#pragma unroll
    for (int l = 0; l < 4; l++) o[l] = s.px;
  }
}

template <uint32_t OP, bool FLOAT, bool WHOLE>
__device__ __attribute__((always_inline, flatten)) void quad_run(const QuadJob &J) {
  const Fmt32 fd = fmt32(J.dst_fmt), fo = fmt32(J.out_fmt), fs = fmt32(J.src.fmt),
              fm = fmt32(J.mask.fmt);
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x * 4;
  const uint32_t rows = WHOLE ? 1u : J.rows;
  for (uint32_t row = WHOLE ? 0u : blockIdx.y * blockDim.y + threadIdx.y; row < rows;
       row += gridDim.y * blockDim.y)
    for (uint64_t i = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4; i < J.row_px;
         i += stride) {
      const uint32_t n = WHOLE ? 4u : (uint32_t)min((uint64_t)4, J.row_px - i);
      const uint64_t at = (uint64_t)row * J.pitch + i;
      const Quad32 draw = quad_words<WHOLE>(J.dst + at, n);
      I4 s[4];
      quad_load<WHOLE>(J.src, fs, row, i, n, s);
      I4 m[4];
      if (J.masked) quad_load<WHOLE>(J.mask, fm, row, i, n, m);
      Quad32 res;
#pragma unroll
      for (int l = 0; l < 4; l++) {
        const I4 d = unpack32(draw.v[l], fd);
        if (FLOAT) {
          F4 sv = decode_raw(s[l]);
          if (J.masked) sv = op_float(Z2D_OP_DST_IN, sv, decode_raw(m[l]));
          res.v[l] = pack32(encode_raw(op_float(OP, decode_raw(d), sv)), fo);
        } else {
          I4 sv = s[l];
          if (J.masked) sv = op_int(Z2D_OP_DST_IN, sv, m[l]);
          res.v[l] = pack32(op_int(OP, d, sv), fo);
        }
      }
      if (WHOLE) {
        *reinterpret_cast<uint4 *>(J.out + at) =
            make_uint4(res.v[0], res.v[1], res.v[2], res.v[3]);
      } else if (n >= 4) {
        *reinterpret_cast<Quad32 *>(J.out + at) = res;
      } else {
#pragma unroll
        for (uint32_t l = 0; l < 3; l++)
          if (l < n) J.out[at + l] = res.v[l];
      }
    }
}

template <bool WHOLE>
__global__ void __launch_bounds__(256) k_composite_quad(QuadJob J) {
  const bool flt = J.precision != Z2D_PRECISION_INTEGER;
  switch (J.op) {
#define Z2D_QUAD_CASE(n)            \
  case n:                          \
    if (flt)                       \
      quad_run<n, true, WHOLE>(J); \
    else                           \
      quad_run<n, false, WHOLE>(J); \
    break;
    Z2D_QUAD_CASE(0) Z2D_QUAD_CASE(1) Z2D_QUAD_CASE(2) Z2D_QUAD_CASE(3) Z2D_QUAD_CASE(4)
    Z2D_QUAD_CASE(5) Z2D_QUAD_CASE(6) Z2D_QUAD_CASE(7) Z2D_QUAD_CASE(8) Z2D_QUAD_CASE(9)
    Z2D_QUAD_CASE(10) Z2D_QUAD_CASE(11) Z2D_QUAD_CASE(12) Z2D_QUAD_CASE(13) Z2D_QUAD_CASE(14)
    Z2D_QUAD_CASE(15) Z2D_QUAD_CASE(16) Z2D_QUAD_CASE(17) Z2D_QUAD_CASE(18) Z2D_QUAD_CASE(19)
    Z2D_QUAD_CASE(20) Z2D_QUAD_CASE(21) Z2D_QUAD_CASE(22) Z2D_QUAD_CASE(23) Z2D_QUAD_CASE(24)
    Z2D_QUAD_CASE(25) Z2D_QUAD_CASE(26) Z2D_QUAD_CASE(27)
#undef Z2D_QUAD_CASE
    default: break;
  }
}

// ---------------------------------------------------------------------------
// k_composite_paint: a whole surface painted with a gradient or a dither, PX
// (four or one) pixels of a row per lane, per pixel what comp_pixel computes
// for the same
// batch.  Bound by VALU work (the f64 offset, the stop search, the divisions):
// the gradient's constants and stops are in LDS once per workgroup, the
// source kind is a template parameter, and the dither thresholds, which
// repeat every 64 columns, are read once per row and lane.  A 3840x2160
// surface, radial gradient under blue noise: 153 us a launch in the general
// kernel before, 48 now; 164 and 73 us a call.
// ---------------------------------------------------------------------------
constexpr uint32_t PAINT_COLOR = 3;  // KIND: a gradient type, or a color's dither

template <uint32_t KIND, bool DITHER, uint32_t PX>
__global__ void __launch_bounds__(256) k_composite_paint(PaintJob J) {
  __shared__ FastDraw B;
  const DevPaint &P = *J.paint;
  if constexpr (KIND != PAINT_COLOR) {
    if (threadIdx.x == 0 && threadIdx.y == 0)
      write_fast_gradient(B, *P.gradient, FAST_PAINT_LINEAR + KIND);
    __syncthreads();
  }
  const uint32_t n_stops =
      KIND == PAINT_COLOR ? 0u : min(__builtin_amdgcn_readfirstlane(B.n_stops), FAST_STOPS);
  const Fmt32 fd = fmt32(J.dst_fmt), fo = fmt32(J.out_fmt);
  const uint32_t d_type = DITHER ? load_uniform(&P.dither_type) : 0u;
  const F4 color = load_uniform(&P.dither_color);
  const float sc = DITHER ? 1.0f / (float)((1 << load_uniform(&P.dither_scale)) - 1) : 0.0f;
  const int32_t x0 = (int32_t)((blockIdx.x * 64u + threadIdx.x) * PX);
  const int32_t step = (int32_t)(gridDim.x * 64u * PX);  // a multiple of 64
  for (int32_t y = (int32_t)(blockIdx.y * blockDim.y + threadIdx.y); y < J.h;
       y += (int32_t)(gridDim.y * blockDim.y)) {
    float th[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // the columns' thresholds, scaled
    if (DITHER && d_type != Z2D_DITHER_NONE) {
#pragma unroll
      for (int l = 0; l < (int)PX; l++) {
        const int x = x0 + l;
        const float m = d_type == Z2D_DITHER_BAYER
                            ? bayer8(x, y)
                            : (float)J.blue_noise[((x & 63) << 6) | (y & 63)] * (2.0f / 8192.0f) -
                                  (4095.0f / 8192.0f);
        th[l] = m * sc;
      }
    }
    for (int32_t x = x0; x < J.w; x += step) {
      const uint32_t n = (uint32_t)min((int32_t)PX, J.w - x);
      const uint64_t at = (uint64_t)y * (uint32_t)J.w + (uint32_t)x;
      Quad32 dst{};
      if (J.op != Z2D_OP_SRC) dst = quad_words<false>(J.dst + at, n);
      Quad32 res;
#pragma unroll 1
      for (uint32_t l = 0; l < PX; l++) {
        I4 s;
        F4 c = color;
        if constexpr (KIND != PAINT_COLOR) {
          float off;
          if constexpr (KIND == Z2D_GRADIENT_LINEAR)
            off = fast_linear_offset(B, x + (int)l, y);
          else if constexpr (KIND == Z2D_GRADIENT_RADIAL)
            off = fast_radial_offset(B, x + (int)l, y);
          else
            off = fast_conic_offset(B, x + (int)l, y);
          int i0, i1;
          float t;
          bool transparent;
          stops_find8(B.offs, n_stops, off, i0, i1, t, transparent);
          const float4 p = B.pre[i0], q = B.pre[i1];
          c = F4{lerpf_(p.x, q.x, t), lerpf_(p.y, q.y, t), lerpf_(p.z, q.z, t),
                 lerpf_(p.w, q.w, t)};
          if (transparent) c = F4{0.0f, 0.0f, 0.0f, 0.0f};
          if (DITHER) {  // straight alpha
            const Divisor a = divisor(c.a);
            const bool none = c.a == 0.0f;
            c.r = none ? 0.0f : div_by(c.r, a);
            c.g = none ? 0.0f : div_by(c.g, a);
            c.b = none ? 0.0f : div_by(c.b, a);
          }
        }
        if (DITHER) {
          if (d_type != Z2D_DITHER_NONE) {
            const float m = l == 0 ? th[0] : l == 1 ? th[1] : l == 2 ? th[2] : th[3];
            c = F4{clampz(c.r + m, 0.0f, 1.0f), clampz(c.g + m, 0.0f, 1.0f),
                   clampz(c.b + m, 0.0f, 1.0f), clampz(c.a + m, 0.0f, 1.0f)};
          }
          const float v[4] = {c.r, c.g, c.b, c.a};
          s = encode_premul(v);
        } else {
          s = I4{f2u8(255.0f * c.r), f2u8(255.0f * c.g), f2u8(255.0f * c.b), f2u8(255.0f * c.a)};
        }
        const uint32_t d = l == 0 ? dst.v[0] : l == 1 ? dst.v[1] : l == 2 ? dst.v[2] : dst.v[3];
        const uint32_t o = J.op == Z2D_OP_SRC ? pack32(s, fo)
                                              : pack32(op_int(J.op, unpack32(d, fd), s), fo);
        if (l == 0) res.v[0] = o;
        if (l == 1) res.v[1] = o;
        if (l == 2) res.v[2] = o;
        if (l == 3) res.v[3] = o;
      }
      if (n >= 4) {
        *reinterpret_cast<Quad32 *>(J.out + at) = res;
      } else {
        for (uint32_t l = 0; l < n; l++)
          J.out[at + l] = l == 0 ? res.v[0] : l == 1 ? res.v[1] : res.v[2];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// launchers (called from host.cpp)
// ---------------------------------------------------------------------------
}  // namespace z2d

using namespace z2d;

// Reference streams for the achievable HBM rate: a copy (1 read : 1 write)
// and, the compositor's mix, two reads and one write (dst = a ^ b).  The
// same shape as the whole-surface compositor's loop (16 B per buffer per
// lane per iteration, at most 8192 blocks of 256 threads striding over the
// buffers), so the two are compared on equal terms; also the known-size
// kernel that calibrates the HBM byte counters.
template <bool READ2>
__global__ void __launch_bounds__(256) k_stream(const uint4 *__restrict__ a,
                                                const uint4 *__restrict__ b,
                                                uint4 *__restrict__ dst, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    uint4 v = a[i];
    if (READ2) {
      const uint4 w = b[i];
      v.x ^= w.x; v.y ^= w.y; v.z ^= w.z; v.w ^= w.w;
    }
    dst[i] = v;
  }
}

static uint32_t stream_blocks(uint64_t n) {
  const uint64_t blocks = (n + 255) / 256;
  return (uint32_t)(blocks > 8192 ? 8192 : blocks);
}

hipError_t z2d_launch_stream_copy(const void *src, void *dst, uint64_t bytes, hipStream_t st) {
  const uint64_t n = bytes / 16;
  hipLaunchKernelGGL(k_stream<false>, dim3(stream_blocks(n)), dim3(256), 0, st,
                     reinterpret_cast<const uint4 *>(src), nullptr, reinterpret_cast<uint4 *>(dst),
                     n);
  return hipGetLastError();
}

hipError_t z2d_launch_stream_read2(const void *a, const void *b, void *dst, uint64_t bytes,
                                   hipStream_t st) {
  const uint64_t n = bytes / 16;
  hipLaunchKernelGGL(k_stream<true>, dim3(stream_blocks(n)), dim3(256), 0, st,
                     reinterpret_cast<const uint4 *>(a), reinterpret_cast<const uint4 *>(b),
                     reinterpret_cast<uint4 *>(dst), n);
  return hipGetLastError();
}

__global__ void k_fill_u32(uint32_t *p, uint64_t n, uint32_t v) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Command y of the list, strided over the x blocks: 16-byte moves where the
// addresses and the size allow, bytes otherwise; fills write whole words.
__global__ void __launch_bounds__(256) k_multi_copy(const CopyCmd *__restrict__ cmds) {
  const CopyCmd c = cmds[blockIdx.y];
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint64_t t0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (!c.src) {
    uint32_t *d = reinterpret_cast<uint32_t *>(c.dst);
    const uint64_t n = c.bytes / 4;
    for (uint64_t i = t0; i < n; i += stride) d[i] = c.value;
    return;
  }
  const bool v16 = ((reinterpret_cast<uintptr_t>(c.src) | reinterpret_cast<uintptr_t>(c.dst)) &
                    15u) == 0;
  uint64_t done = 0;
  if (v16) {
    const uint64_t n = c.bytes / 16;
    const uint4 *s4 = reinterpret_cast<const uint4 *>(c.src);
    uint4 *d4 = reinterpret_cast<uint4 *>(c.dst);
    for (uint64_t i = t0; i < n; i += stride) d4[i] = s4[i];
    done = n * 16;
  }
  for (uint64_t i = done + t0; i < c.bytes; i += stride) c.dst[i] = c.src[i];
}

hipError_t z2d_launch_multi_copy(const CopyCmd *cmds, uint32_t n, hipStream_t st) {
  for (uint32_t c0 = 0; c0 < n; c0 += 65535u) {  // grid y is at most 65535
    hipLaunchKernelGGL(k_multi_copy, dim3(64, min(65535u, n - c0)), dim3(256), 0, st, cmds + c0);
  }
  return hipGetLastError();
}

hipError_t z2d_launch_grad_setup(DevGradient *grads, uint32_t n_grads, hipStream_t st) {
  if (n_grads == 0) return hipSuccess;
  hipLaunchKernelGGL(k_grad_setup, dim3((n_grads + 63) / 64), dim3(64), 0, st, grads, n_grads);
  return hipGetLastError();
}

__global__ void __launch_bounds__(256) k_fill_set(FillSet F) {
  const uint32_t f = blockIdx.y;
  uint32_t *const p = F.p[f];
  const uint64_t n = F.n[f];
  const uint32_t v = F.v[f];
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

hipError_t z2d_launch_fill_set(const FillSet &F, hipStream_t st) {
  if (F.count == 0) return hipSuccess;
  uint64_t most = 0;
  for (uint32_t f = 0; f < F.count; f++) most = F.n[f] > most ? F.n[f] : most;
  const uint64_t blocks = (most + 255) / 256;
  hipLaunchKernelGGL(k_fill_set, dim3((uint32_t)(blocks < 1 ? 1 : (blocks > 1024 ? 1024 : blocks)), F.count),
                     dim3(256), 0, st, F);
  return hipGetLastError();
}

hipError_t z2d_launch_fill_u32(uint32_t *p, uint64_t n, uint32_t v, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_u32, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, st, p, n, v);
  return hipGetLastError();
}

hipError_t z2d_launch_edge_build(const JobView &J, hipStream_t st) {
  if (J.n_draws == 0) return hipSuccess;
  const dim3 grid((J.n_egroups + 3) / 4);
  hipLaunchKernelGGL(k_edge_build, grid, dim3(256), 0, st, J);
  return hipGetLastError();
}

hipError_t z2d_launch_rowprog(const JobView &J, const uint32_t *list, uint32_t n,
                              z2d_edge *sedges, int32_t *sx, const uint32_t *soff,
                              hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_rowprog, dim3((n + 63) / 64), dim3(64), 0, st, J, list, n, sedges, sx,
                     soff);
  return hipGetLastError();
}

hipError_t z2d_launch_binning(const JobView &J, hipStream_t st) {
  if (J.n_bands == 0) return hipSuccess;
  // entry edge lists: offsets from k_edge_build's counts, then the copies
  // (entry_ecnt, entry_cur and the entry column ranges were reset by the
  // pipeline's first fill, z2d_launch_fill_set)
  dim3 ggrid((J.n_egroups + 3) / 4);
  scan_u32(J.entry_ecnt, J.max_entries, J.scan_tmp, J.counters + 2, st);
  if (J.n_egroups) hipLaunchKernelGGL(k_edge_bins, ggrid, dim3(256), 0, st, J);
  // band lists and entry records
  const dim3 pblock(64 * PASS_WAVES);
  uint64_t *const bstat = J.scan_tmp + J.scan_words, *const sstat = bstat + J.scan_words;
  auto groups = [](uint32_t n, uint32_t per) {
    return dim3((n + PASS_WAVES * per - 1) / (PASS_WAVES * per));
  };
  if (groups(J.n_slots, 1).x <= PASS_GROUPS)
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_band_pass<1>), groups(J.n_slots, 1), pblock, 0, st, J, bstat);
  else
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_band_pass<BAND_PASS_PER>),
                       groups(J.n_slots, BAND_PASS_PER), pblock, 0, st, J, bstat);
  if (J.n_tiles) {
    if (groups(J.n_tiles, 1).x <= PASS_GROUPS)
      hipLaunchKernelGGL(HIP_KERNEL_NAME(k_strip_pass<1>), groups(J.n_tiles, 1), pblock, 0, st, J, sstat);
    else
      hipLaunchKernelGGL(HIP_KERNEL_NAME(k_strip_pass<STRIP_PASS_PER>),
                         groups(J.n_tiles, STRIP_PASS_PER), pblock, 0, st, J, sstat);
    if (J.strip_order) {
      const uint32_t ns = J.n_tiles * J.strips_per_tile;
      const dim3 og((ns + 255) / 256);
      hipLaunchKernelGGL(k_fill_u32, dim3((ORDER_BUCKETS + 1 + 255) / 256), dim3(256), 0, st,
                         J.order_hist, (uint64_t)ORDER_BUCKETS + 1, 0u);
      hipLaunchKernelGGL(k_order_hist, og, dim3(256), 0, st, J, ns);
      hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, st, J.order_hist, ORDER_BUCKETS);
      hipLaunchKernelGGL(k_order_scatter, og, dim3(256), 0, st, J, ns);
    }
  }
  return hipGetLastError();
}

// Count pass (emit = false): the curve pieces, their combination per curve,
// the per-node pass for every draw, then the per-draw walk for the draws it
// marked FLAT_NONSIMPLE.  Emit pass: each draw by the form its
// FlatJob.serial names (the per-draw walk launched only when any_serial),
// curves by pieces, and the fills of *fill (when given) done by the per-node
// kernel's workgroups before their draws.
hipError_t z2d_launch_flatten(const z2d_path_node *raw, const FlatJob *jobs, uint32_t n_jobs,
                              FNode *out, FlatResult *res, uint32_t *rel, const uint2 *curves,
                              uint32_t n_curves, FlatTask *tasks, uint32_t *toff, FlatCurve *cv,
                              const uint2 *groups, uint32_t n_groups, uint32_t *mvi, bool emit,
                              hipStream_t st, const FillSet *fill, bool any_serial) {
  if (n_jobs == 0) return hipSuccess;
  const FillSet no_fill{};
  const dim3 wgrid((n_jobs + 3) / 4), sgrid((n_jobs + 63) / 64);
  const dim3 tgrid((uint32_t)(((uint64_t)n_curves * FLAT_TASKS + 255) / 256)),
      cgrid((n_curves + 255) / 256);
  if (emit) {
    hipLaunchKernelGGL(k_flatten_nodes, dim3((n_groups + 3) / 4), dim3(256), 0, st, raw, jobs,
                       groups, n_groups, out, rel, mvi, fill ? *fill : no_fill);
    if (n_curves)
      hipLaunchKernelGGL(k_curve_tasks<true>, tgrid, dim3(256), 0, st, raw, jobs, curves, n_curves,
                         tasks, toff, rel, out);
    if (any_serial)
      hipLaunchKernelGGL(k_flatten_serial<true>, sgrid, dim3(64), 0, st, raw, jobs, n_jobs, out,
                         res);
  } else {
    if (n_curves) {
      hipLaunchKernelGGL(k_curve_tasks<false>, tgrid, dim3(256), 0, st, raw, jobs, curves,
                         n_curves, tasks, toff, rel, out);
      hipLaunchKernelGGL(k_curve_combine, cgrid, dim3(256), 0, st, raw, jobs, curves, n_curves,
                         tasks, toff, cv);
    }
    hipLaunchKernelGGL(k_flatten_wave, wgrid, dim3(256), 0, st, raw, jobs, n_jobs, res, rel, mvi,
                       cv);
    hipLaunchKernelGGL(k_flatten_serial<false>, sgrid, dim3(64), 0, st, raw, jobs, n_jobs, out,
                       res);
  }
  return hipGetLastError();
}

// The tile render of tiles [tile_base, tile_base + tile_count): k_render_fast
// over the strips of fast draws, a workgroup per strip, then k_render over
// the others.  How many those are is known on the device only: beyond 8,192
// strips k_render gets a workgroup for every fourth, which costs a render
// without any of them 3 us instead of 9 (32,400 strips) and leaves 8 waves a
// SIMD to hand out where all are.
hipError_t z2d_launch_render(const JobView &J, uint32_t tile_base, uint32_t tile_count,
                             hipStream_t st) {
  if (tile_count == 0) return hipSuccess;
  const bool all = tile_base == 0 && tile_count == J.n_tiles;
  const uint32_t take = all && J.strip_order ? STRIPS_ORDERED : all ? STRIPS_SLOW : STRIPS_TILES;
  // a launch has fewer than 2^32 lanes
  const uint32_t n = tile_count * J.strips_per_tile, most = 1u << 25;
  for (uint32_t i = 0; i < n; i += most)
    hipLaunchKernelGGL(k_render_fast, dim3(min(most, n - i)), dim3(64), 0, st, J, tile_base,
                       tile_count, i, take == STRIPS_SLOW ? (uint32_t)STRIPS_TILES : take);
  hipLaunchKernelGGL(k_render, dim3(min(most, n <= 8192 ? n : max(8192u, n / 4))), dim3(64), 0, st,
                     J, tile_base, tile_count, take);
  return hipGetLastError();
}

// One row (whole surfaces): 256 lanes along it.  A region of several: four
// rows of 64 lanes, so that a region narrower than 1,024 pixels fills the
// workgroup.
hipError_t z2d_launch_composite_quad(const QuadJob &job, hipStream_t st) {
  if (job.row_px == 0 || job.rows == 0) return hipSuccess;
  const dim3 block = job.rows == 1 ? dim3(256) : dim3(64, 4);
  const uint64_t bx = ((job.row_px + 3) / 4 + block.x - 1) / block.x;
  const uint32_t by = (job.rows + block.y - 1) / block.y;
  // whole quads on their own addresses: one row of them, nothing shifted
  uintptr_t low = reinterpret_cast<uintptr_t>(job.dst) | reinterpret_cast<uintptr_t>(job.out);
  for (const QuadSrc *q : {&job.src, &job.mask})
    if (q == &job.src || job.masked) {
      const uintptr_t a = reinterpret_cast<uintptr_t>(q->data);
      if (q->kind == QUAD_SURF32) low |= a;
      if (q->kind == QUAD_ALPHA8) low |= (a & 3u) << 2;
    }
  const bool whole = job.rows == 1 && job.row_px % 4 == 0 && (low & 15u) == 0;
  hipLaunchKernelGGL(whole ? k_composite_quad<true> : k_composite_quad<false>,
                     dim3((uint32_t)min(bx, (uint64_t)8192), min(by, 16384u)), block, 0, st, job);
  return hipGetLastError();
}

// Up to this many pixels a lane paints one: such a surface leaves most of the
// chip idle, and a lane's four pixels are one chain after the other.  A call
// on 640x480 (linear to conic, dithered or not) takes 25.3 to 28.3 us with one
// and 26.2 to 34.3 with four, on 150x150 24.7 to 26.5 and 25.9 to 33.5 (the
// general kernel, which gives every pixel a lane where the width is no
// multiple of four: 26.8 to 28.8); on 701x601 linear takes 27.2 and 26.4,
// conic 29.8 and 31.6, on 1024x768 radial 31.0 and 27.8.
constexpr uint64_t PAINT_SINGLE = 5u << 16;

template <uint32_t KIND, bool DITHER>
static void launch_paint(const PaintJob &J, hipStream_t st) {
  const bool single = (uint64_t)J.w * (uint32_t)J.h <= PAINT_SINGLE;
  const uint32_t cols = single ? 64u : 256u;  // of a workgroup
  const dim3 block(64, 4);
  const uint32_t bx = ((uint32_t)J.w + cols - 1) / cols, by = (uint32_t)((J.h + 3) / 4);
  // some 4,096 workgroups: enough for eight waves a SIMD twice over
  const dim3 grid(min(bx, 16u), min(by, 4096u / min(bx, 16u)));
  if (single)
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_composite_paint<KIND, DITHER, 1>), grid, block, 0, st, J);
  else
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_composite_paint<KIND, DITHER, 4>), grid, block, 0, st, J);
}

// kind: a gradient type or PAINT_COLOR.
hipError_t z2d_launch_composite_paint(const PaintJob &J, uint32_t kind, bool dither,
                                      hipStream_t st) {
  switch (kind * 2 + (dither ? 1 : 0)) {
    case 0: launch_paint<0, false>(J, st); break;
    case 1: launch_paint<0, true>(J, st); break;
    case 2: launch_paint<1, false>(J, st); break;
    case 3: launch_paint<1, true>(J, st); break;
    case 4: launch_paint<2, false>(J, st); break;
    case 5: launch_paint<2, true>(J, st); break;
    default: launch_paint<PAINT_COLOR, true>(J, st);
  }
  return hipGetLastError();
}

hipError_t z2d_launch_composite(const CompJob *dev_job, const CompJob &host_job, bool stream,
                                hipStream_t st) {
  if (host_job.width <= 0 || host_job.height <= 0) return hipSuccess;
  if (stream) {
    uint64_t quads = (uint64_t)host_job.width * (uint64_t)host_job.height / 4;
    uint64_t blocks = (quads + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(k_composite_stream, dim3((uint32_t)blocks), dim3(256), 0, st, dev_job,
                       quads);
  } else {
    uint32_t bx = (uint32_t)((host_job.width + 255) / 256);
    uint32_t by = (uint32_t)(host_job.height < 65535 ? host_job.height : 65535);
    hipLaunchKernelGGL(k_composite, dim3(bx, by), dim3(256), 0, st, dev_job);
  }
  return hipGetLastError();
}
