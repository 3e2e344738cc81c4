// Device-side bodies of the 2D distance-driven kernels, shared by the
// one-call kernels (dd2d.hip) and the persistent batched kernels
// (ddbatch.hip), so both paths execute the same arithmetic.
//
// Behaviour followed: deeprecon/cpu/dis2d/FanArcDisCPU2d.cpp (fan arc),
// FanFlatDisCPU2d.cpp (fan flat), ParaDisCPU2d.cpp (parallel).
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "dd.h"
#include "dd_common.h"

namespace dd {
namespace body2d {


constexpr int kThreads = 256;
constexpr int kTile = 16;  // pixel tile edge of k_pixels (16 x 16 = 256)

enum WMode { W_FP = 0, W_BP = 1, W_BPW = 2 };

struct Geo2 {
  int W, H, D, V, B, Bp, BT, Lmax, scan;
  float dx, dy, det, sid, sdd, shx, shy, bin;
};

// Output epilogue of an op (fused update steps): out = alpha * s * result
// + beta * c, s = *scale (a device scalar) or 1, c a device array shaped
// like the output or null.  The default leaves the result untouched, bit for
// bit.
struct Epi {
  const float* c = nullptr;
  const float* scale = nullptr;
  float alpha = 1.0f, beta = 0.0f;
};

__device__ __forceinline__ float epi_value(const Epi& e, float v, size_t at) {
  if (e.scale) v *= e.alpha * *e.scale;
  else if (e.alpha != 1.0f) v *= e.alpha;
  if (e.c) v = fmaf(e.beta, e.c[at], v);
  return v;
}

// ---------------------------------------------------------------------------
// 1. per-view setup (FP64 boundary mapping)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void setup2d_view(
    const Geo2& g, const float* __restrict__ angles, ViewGeo* __restrict__ views,
    double* __restrict__ edges, float* __restrict__ wfp,
    LineGeo* __restrict__ lines, float* __restrict__ pint, int v) {
  const float thf = angles[v];
  const double th = static_cast<double>(thf);
  int xaxis, flip;
  choose_axis(thf, &xaxis, &flip);
  const double s = sin(th), c = cos(th);
  const double sid = g.sid, sdd = g.sdd, det = g.det, bin = g.bin;
  const double dx = g.dx, dy = g.dy, shx = g.shx, shy = g.shy;
  const double sx = -s * sid, sy = c * sid;
  const int D = g.D;
  if (threadIdx.x == 0) {
    ViewGeo vg;
    vg.sx = sx;
    vg.sy = sy;
    vg.s = s;
    vg.c = c;
    vg.theta_ref = th + bin;
    vg.xaxis = xaxis;
    vg.flip = flip;
    vg.sxf = static_cast<float>(sx);
    vg.syf = static_cast<float>(sy);
    vg.cref = static_cast<float>(cos(th + bin));
    vg.sref = static_cast<float>(sin(th + bin));
    views[v] = vg;
  }
  // Bin edges, walk-ordered (FanArcDisCPU2d.cpp:77-86; FanFlatDisCPU2d.cpp:
  // 72-84; ParaDisCPU2d.cpp:51-55).
  double* ev = edges + static_cast<size_t>(v) * (D + 1);
  for (int k = threadIdx.x; k <= D; k += blockDim.x) {
    const double off = flip ? (D / 2.0 - k) : (k - D / 2.0);
    double e;
    if (g.scan == DD_FAN_ARC) {
      const double t = tan(off * det + bin + th);
      e = xaxis ? sx + sy * t : sy + sx / t;
    } else if (g.scan == DD_FAN_FLAT) {
      const double u = off * (sid / sdd * det) + sid / sdd * bin;
      const double px = u * c, py = u * s;
      e = xaxis ? (sx * py - sy * px) / (py - sy)
                : (sy * px - sx * py) / (px - sx);
    } else {
      e = (off * det + bin) / (xaxis ? c : s);
    }
    ev[k] = e;
  }
  __syncthreads();
  // FP weight: perpendicular pixel size / (bin width on the axis * cosine of
  // the bin-centre ray to the axis normal) (FanArcDisCPU2d.cpp:87-93);
  // parallel beam dy/det or dx/det (ParaDisCPU2d.cpp:60,113).
  const double perp = xaxis ? dy : dx;
  for (int k = threadIdx.x; k < D; k += blockDim.x) {
    double w;
    if (g.scan == DD_PARA) {
      w = perp / det;
    } else {
      const double e0 = ev[k], e1 = ev[k + 1];
      const double mid = 0.5 * (e0 + e1);
      const double cs = xaxis ? fabs(sy) / sqrt((mid - sx) * (mid - sx) + sy * sy)
                              : fabs(sx) / sqrt((mid - sy) * (mid - sy) + sx * sx);
      w = perp / ((e1 - e0) * cs);
    }
    wfp[static_cast<size_t>(v) * D + k] = static_cast<float>(w);
  }
  // Pixel edges of each line on the axis (FanArcDisCPU2d.cpp:95-101,165-171;
  // ParaDisCPU2d.cpp:57-64,110-117).
  const int L = xaxis ? g.H : g.W;
  for (int l = threadIdx.x; l < L; l += blockDim.x) {
    double a0, p;
    if (xaxis) {
      const double yl = (g.H / 2.0 - l - 0.5) * dy + shy;
      const double x0 = -g.W / 2.0 * dx + shx, x1 = g.W / 2.0 * dx + shx;
      if (g.scan == DD_PARA) {
        a0 = x0 + yl * s / c;
        p = dx;
      } else {
        a0 = (sx * yl - sy * x0) / (yl - sy);
        const double a1 = (sx * yl - sy * x1) / (yl - sy);
        p = (a1 - a0) / g.W;
      }
    } else {
      const double xl = (l - g.W / 2.0 + 0.5) * dx + shx;
      const double y0 = -g.H / 2.0 * dy + shy, y1 = g.H / 2.0 * dy + shy;
      if (g.scan == DD_PARA) {
        a0 = y0 + xl * c / s;
        p = dy;
      } else {
        a0 = (sy * xl - sx * y0) / (xl - sx);
        const double a1 = (sy * xl - sx * y1) / (xl - sx);
        p = (a1 - a0) / g.H;
      }
    }
    LineGeo lg;
    lg.a0 = a0;
    lg.inv_p = 1.0 / p;
    lines[static_cast<size_t>(v) * g.Lmax + l] = lg;
    pint[static_cast<size_t>(v) * g.Lmax + l] = static_cast<float>(p);
  }
}

// ---------------------------------------------------------------------------
// 2. layout prologues
// ---------------------------------------------------------------------------
// x [B][H][W] -> xrow [H][W][Bp] (lines = rows) and
//               xcol [W][H][Bp] with xcol[l][i] = x[H-1-i][l] (lines = columns,
//               pixel index from the bottom, FanArcDisCPU2d.cpp:194).
// Instance-interleaved image copies for tiles of 8+ instances are quad-major,
// [Bp / 4][line][pixel][4]: the 4 float4 loads a lane makes for one pixel of
// a 16-instance tile then each read consecutive pixels across the wavefront
// (one 16-byte slice per pixel, the wave's pixels contiguous), instead of
// every load touching every pixel record's cache line.  Tiles of 1-4 keep
// [line][pixel][Bp].
template <int BT>
constexpr bool image_quad_major() {
  return BT >= 8;
}

// The sinogram copy of the sinogram -> image gathers likewise:
// [Bp / 4][view][bin][4] for tiles of 8+ instances, [view][bin][Bp] below.
template <int BT>
constexpr bool sino_quad_major() {
  return BT >= 8;
}

// View v of the sinogram copy for the tile starting at instance b0.
template <int BT>
__device__ __forceinline__ const float* sino_view(const Geo2& g, const float* sino, int v,
                                                  int b0) {
  if constexpr (sino_quad_major<BT>())
    return sino + (static_cast<size_t>(b0 / 4) * g.V * g.D + static_cast<size_t>(v) * g.D) * 4;
  else
    return sino + static_cast<size_t>(v) * g.D * g.Bp + b0;
}

// The BT values of bin k of a view returned by sino_view.
template <int BT>
__device__ __forceinline__ void load_sino(const Geo2& g, const float* __restrict__ sv, int k,
                                          float (&q)[BT]) {
  if constexpr (sino_quad_major<BT>()) {
    const size_t plane4 = static_cast<size_t>(g.V) * g.D * 4;
#pragma unroll
    for (int j = 0; j < BT / 4; ++j) {
      const float4 t =
          *reinterpret_cast<const float4*>(sv + j * plane4 + static_cast<size_t>(k) * 4);
      q[4 * j] = t.x;
      q[4 * j + 1] = t.y;
      q[4 * j + 2] = t.z;
      q[4 * j + 3] = t.w;
    }
  } else {
    load_tile<BT>(sv + static_cast<size_t>(k) * g.Bp, q);
  }
}

template <int BT>
__device__ __forceinline__ void load_image_px(const Geo2& g, const float* __restrict__ x, int h,
                                              int w, int b0, float (&v)[BT]) {
#pragma unroll
  for (int b = 0; b < BT; ++b)
    v[b] = (b0 + b < g.B)
               ? x[(static_cast<size_t>(b0 + b) * g.H + h) * g.W + w]
               : 0.0f;
}

// Pixel (h, w)'s BT values into the row copy (COL false) or the column copy
// (COL true, lines read bottom-up).
template <int BT, bool COL>
__device__ __forceinline__ void store_image_px(const Geo2& g, float* __restrict__ xc, int h,
                                               int w, int b0, const float (&v)[BT]) {
  const size_t px = COL ? static_cast<size_t>(w) * g.H + (g.H - 1 - h)
                        : static_cast<size_t>(h) * g.W + w;
  if constexpr (image_quad_major<BT>()) {
    const size_t plane = static_cast<size_t>(g.W) * g.H;  // pixels per quad plane
#pragma unroll
    for (int q = 0; q < BT / 4; ++q)
      *reinterpret_cast<float4*>(xc + (static_cast<size_t>(b0 / 4 + q) * plane + px) * 4) =
          make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
  } else {
    store_tile<BT>(xc + px * g.Bp + b0, v);
  }
}

template <int BT>
__device__ __forceinline__ void interleave_image_px(
    const Geo2& g, const float* __restrict__ x, float* __restrict__ xrow,
    float* __restrict__ xcol, int h, int w, int b0) {
  float v[BT];
  load_image_px<BT>(g, x, h, w, b0, v);
  store_image_px<BT, false>(g, xrow, h, w, b0, v);
  store_image_px<BT, true>(g, xcol, h, w, b0, v);
}

// p [B][V][D] -> s [V][D][Bp] in walk order, optionally scaled by the FP
// weight of the bin (the adjoint's left factor).
template <int BT, bool FOLD_W>
__device__ __forceinline__ void interleave_sino_bin(
    const Geo2& g, const ViewGeo* __restrict__ views, const float* __restrict__ wfp,
    const float* __restrict__ p, float* __restrict__ s, int v, int k, int b0) {
  const int kk = views[v].flip ? g.D - 1 - k : k;
  const float wk = FOLD_W ? wfp[static_cast<size_t>(v) * g.D + k] : 1.0f;
  float val[BT];
#pragma unroll
  for (int b = 0; b < BT; ++b)
    val[b] = (b0 + b < g.B)
                 ? p[(static_cast<size_t>(b0 + b) * g.V + v) * g.D + kk] * wk
                 : 0.0f;
  if constexpr (sino_quad_major<BT>()) {
#pragma unroll
    for (int j = 0; j < BT / 4; ++j)
      *reinterpret_cast<float4*>(
          s + ((static_cast<size_t>(b0 / 4 + j) * g.V + v) * g.D + k) * 4) =
          make_float4(val[4 * j], val[4 * j + 1], val[4 * j + 2], val[4 * j + 3]);
  } else {
    store_tile<BT>(s + (static_cast<size_t>(v) * g.D + k) * g.Bp + b0, val);
  }
}

// ---------------------------------------------------------------------------
// weights shared by both gather kernels
// ---------------------------------------------------------------------------
// BackProj constant: arc SID*dgamma (FanArcDisCPU2d.cpp:451), flat virtual
// pitch (FanFlatDisCPU2d.cpp:478), parallel det (ParaDisCPU2d.cpp:202); the
// reference divides it by the pixel interval and multiplies by the overlap on
// the axis, which is this constant times the overlap in pixel units.
__host__ __device__ __forceinline__ float bp_const(const Geo2& g) {
  if (g.scan == DD_FAN_ARC) return g.sid * g.det;
  if (g.scan == DD_FAN_FLAT) return g.sid / g.sdd * g.det;
  return g.det;
}

// FBP distance weight of a pixel centre: arc 1/|S-P|^2
// (FanArcDisCPU2d.cpp:27-29,507), flat (r/(r-d))^2 (FanFlatDisCPU2d.cpp:19-22).
// Every product that feeds a sum here and in pixel_centre is an explicit
// fmaf: left to contraction, which product the compiler fuses depends on
// the code around the inlined call, and every kernel must get the same bits.
__device__ __forceinline__ float fbp_weight(const Geo2& g, const ViewGeo& vg,
                                            float xc, float yc) {
  if (g.scan == DD_FAN_ARC) {
    const float ddx = vg.sxf - xc, ddy = vg.syf - yc;
    const float dy2 = ddy * ddy;
    return 1.0f / fmaf(ddx, ddx, dy2);
  }
  const float r = g.sid;
  const float syy = vg.syf * yc;
  const float d = fmaf(vg.sxf, xc, syy) / r;
  return (r * r) / ((r - d) * (r - d));
}

// Pixel centre of (line, pixel) in world coordinates.  The offsets
// (i - W/2 + 1/2 etc.) are exact in FP32, only the scaling rounds.
__device__ __forceinline__ void pixel_centre(const Geo2& g, int xaxis, int l,
                                             int i, float* xc, float* yc) {
  const int cx = xaxis ? i : l, ry = xaxis ? l : i;
  *xc = fmaf(static_cast<float>(cx) - g.W * 0.5f + 0.5f, g.dx, g.shx);
  *yc = xaxis ? fmaf(g.H * 0.5f - static_cast<float>(ry) - 0.5f, g.dy, g.shy)
              : fmaf(static_cast<float>(ry) - g.H * 0.5f + 0.5f, g.dy, g.shy);
}

// ---------------------------------------------------------------------------
// 3a. image -> sinogram: one thread per (view, bin), BT instances
// ---------------------------------------------------------------------------
// Image -> sinogram gathers split each bin's line loop into kSplit chunks
// (one per XCD) and add the chunk sums in chunk order in a second pass.
constexpr int kSplit = 8;

// Forward gathers run 63 bins per wavefront: consecutive lanes hold
// consecutive bins, every lane evaluates the position of its lower edge on
// each line and takes its upper edge's from the next lane (a DPP wave shift,
// the same bits), and lane 63 only serves lane 62's upper edge.  Each edge is
// evaluated once per line instead of twice.
constexpr int kBinsPerWave = 63;
// Tiles from this size up share pixels between forward lanes (below).
constexpr int kSharedPixelMinBT = 2;

__device__ __forceinline__ EdgePos edge_from_next_lane(EdgePos p) {
  constexpr int kWaveShl1 = 0x130;  // DPP wave_shl:1: lane i reads lane i + 1
  EdgePos q;
  q.c = __builtin_amdgcn_update_dpp(0, p.c, kWaveShl1, 0xf, 0xf, false);
  q.f = __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, p.f), kWaveShl1, 0xf, 0xf,
                                         false));
  return q;
}

// Sum over lines [l0, l1) of one bin's overlaps with the image (no bin
// weight); e1 is the bin's lower edge.  The whole wavefront calls this
// together (every lane active: the DPP reads the next lane); `edge_lane`
// marks lane 63.
template <int BT, int WM>
__device__ __forceinline__ void bins_accumulate(
    const Geo2& g, const ViewGeo& vg, double e1, const LineGeo* __restrict__ lv,
    const float* __restrict__ pv, const float* __restrict__ src, float kbp, int l0, int l1,
    int N, float (&acc)[BT], bool edge_lane) {
  const int xaxis = vg.xaxis;
  if (l0 >= l1) return;
  // the next line's geometry is loaded while this line is worked on
  LineGeo lg_next = const_load(lv + l0);
  float lw_next = (WM == W_FP) ? const_load(pv + l0) : kbp;
  for (int l = l0; l < l1; ++l) {
    const LineGeo lg = lg_next;
    const float lw = lw_next;
    lg_next = const_load(lv + min(l + 1, l1 - 1));
    if constexpr (WM == W_FP) lw_next = const_load(pv + min(l + 1, l1 - 1));
    const EdgePos p1 = edge_pos(e1, lg.a0, lg.inv_p, N);
    const EdgePos p2 = edge_from_next_lane(p1);
    const float* __restrict__ line = src + static_cast<size_t>(l) * N *
                                               (image_quad_major<BT>() ? 4 : g.Bp);
    auto load_px = [&](int c, float (&xv)[BT]) {
      if constexpr (image_quad_major<BT>()) {
        const size_t plane4 = static_cast<size_t>(g.W) * g.H * 4;
#pragma unroll
        for (int q = 0; q < BT / 4; ++q) {
          const float4 t = *reinterpret_cast<const float4*>(line + q * plane4 +
                                                            static_cast<size_t>(c) * 4);
          xv[4 * q] = t.x;
          xv[4 * q + 1] = t.y;
          xv[4 * q + 2] = t.z;
          xv[4 * q + 3] = t.w;
        }
      } else {
        load_tile<BT>(line + static_cast<size_t>(c) * g.Bp, xv);
      }
    };
    auto weight = [&](int c) {
      float w = overlap_in_pixel(p1, p2, c) * lw;
      if constexpr (WM == W_BPW) {
        float xc, yc;
        pixel_centre(g, xaxis, l, c, &xc, &yc);
        w *= fbp_weight(g, vg, xc, yc);
      }
      return w;
    };
    const int cs = max(p1.c, 0);
    if constexpr (BT >= kSharedPixelMinBT) {
      // A bin's last pixel is the pixel of its upper edge, which is the next
      // bin's first pixel: every lane (lane 63 too) loads its first pixel and
      // takes its last one from the next lane, so each pixel of the line is
      // loaded once per wavefront instead of once per bin that reaches it.
      float x0[BT];
      if (p1.c <= N - 1) {
        load_px(cs, x0);
      } else {
#pragma unroll
        for (int b = 0; b < BT; ++b) x0[b] = 0.0f;
      }
      float xn[BT];
#pragma unroll
      for (int b = 0; b < BT; ++b)
        xn[b] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                                              0, __builtin_bit_cast(int, x0[b]), 0x130, 0xf,
                                              0xf, false));
      if (edge_lane) continue;
      const int ce = min(p2.c, N - 1);
      if (cs > ce) continue;
      {
        const float w = weight(cs);
#pragma unroll
        for (int b = 0; b < BT; ++b) acc[b] = fmaf(w, x0[b], acc[b]);
      }
      if (ce > cs) {
        for (int c = cs + 1; c < ce; ++c) {  // footprints wider than two pixels
          float xv[BT];
          load_px(c, xv);
          const float w = weight(c);
#pragma unroll
          for (int b = 0; b < BT; ++b) acc[b] = fmaf(w, xv[b], acc[b]);
        }
        // the next lane's first pixel is this bin's last whenever the upper
        // edge lies inside the image (p2.c == ce); past the image, load it
        if (p2.c != ce) load_px(ce, xn);
        const float w = weight(ce);
#pragma unroll
        for (int b = 0; b < BT; ++b) acc[b] = fmaf(w, xn[b], acc[b]);
      }
    } else {
      if (edge_lane) continue;
      const int ce = min(p2.c, N - 1);
      if (cs > ce) continue;
      for (int c = cs; c <= ce; ++c) {
        const float w = weight(c);
        float xv[BT];
        load_px(c, xv);
#pragma unroll
        for (int b = 0; b < BT; ++b) acc[b] = fmaf(w, xv[b], acc[b]);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// 3a'. image -> sinogram through running sums along the lines (one instance
// per geometry, no per-pixel weight)
// ---------------------------------------------------------------------------
// A bin's integral over a line is F(t2) - F(t1), F the running sum of the
// line's pixels, linear inside each pixel: F(t) = C_c + x_c (t - c),
// C_c = x_0 + ... + x_{c-1}, t in pixel units clamped to [0, n].  Each
// (bin, line) is then one lookup instead of a walk over the 1-3 pixels the
// bin covers.  C is accumulated in FP64 and stored as two floats, hi = fl(C)
// and lo = fl(C - hi), beside the pixel itself, {hi_c, lo_c, x_c, 0} (one
// aligned 16-byte load), so differences of nearby sums lose nothing to
// cancellation: F(t2) - F(t1) = (hi2 - hi1) + (m2 - m1) with m = lo + x f,
// where hi2 - hi1 rounds once, relative to the result.  A line of n pixels
// holds n + 1 entries (entry n: the total, x = 0).
__host__ __device__ constexpr int prefix_entries(int n) { return n + 1; }

// Running sums of one line of n pixels x[0], x[stride], ... into
// out[0 .. n], by one workgroup of blockDim.x threads (a power of two
// <= 1024), each owning a contiguous segment.
__device__ __forceinline__ void prefix_line(const float* __restrict__ x, long long stride,
                                            int n, float4* __restrict__ out,
                                            double* __restrict__ lds) {
  const int t = static_cast<int>(threadIdx.x), nt = static_cast<int>(blockDim.x);
  const int seg = (n + nt - 1) / nt;
  const int p0 = min(t * seg, n), p1 = min(p0 + seg, n);
  double s = 0.0;
  for (int p = p0; p < p1; ++p) s += static_cast<double>(x[p * stride]);
  lds[t] = s;
  __syncthreads();
  // inclusive scan of the segment sums (Hillis-Steele)
  for (int d = 1; d < nt; d *= 2) {
    const double add = (t >= d) ? lds[t - d] : 0.0;
    __syncthreads();
    lds[t] += add;
    __syncthreads();
  }
  double c = lds[t] - s;  // sum of the segments before this one
  auto entry = [](double v, float xv) {
    const float hi = static_cast<float>(v);
    return make_float4(hi, static_cast<float>(v - static_cast<double>(hi)), xv, 0.0f);
  };
  for (int p = p0; p < p1; ++p) {
    const float xv = x[p * stride];
    out[p] = entry(c, xv);
    c += static_cast<double>(xv);
  }
  if (t == nt - 1) out[n] = entry(lds[nt - 1], 0.0f);
  __syncthreads();  // lds is reused by the next line
}

// Sum over lines [l0, l1) of one bin's integrals over the lines (no bin
// weight), from the lines' running-sum tables tab[line][n + 1]; e1 is the
// bin's lower edge, the upper edge's sum comes from the next lane.  The whole
// wavefront calls this together (the DPP reads the next lane); lane 63's sum
// is meaningless and not written.
template <int WM>
__device__ __forceinline__ float bins_accumulate_prefix(
    double e1, const LineGeo* __restrict__ lv, const float* __restrict__ pv,
    const float4* __restrict__ tab, float kbp, int l0, int l1, int n) {
  float acc = 0.0f;
  if (l0 >= l1) return acc;
  LineGeo lg_next = const_load(lv + l0);
  float lw_next = (WM == W_FP) ? const_load(pv + l0) : kbp;
  const float4* __restrict__ row = tab + static_cast<size_t>(l0) * prefix_entries(n);
  for (int l = l0; l < l1; ++l, row += prefix_entries(n)) {
    const LineGeo lg = lg_next;
    const float lw = lw_next;
    lg_next = const_load(lv + min(l + 1, l1 - 1));
    if constexpr (WM == W_FP) lw_next = const_load(pv + min(l + 1, l1 - 1));
    const double t = fmin(fmax((e1 - lg.a0) * lg.inv_p, 0.0), static_cast<double>(n));
    const double fl = floor(t);
    const float f = static_cast<float>(t - fl);
    const float4 e = row[static_cast<int>(fl)];
    const float m = fmaf(f, e.z, e.y);
    constexpr int kWaveShl1 = 0x130;  // DPP wave_shl:1: lane i reads lane i + 1
    const float hn = __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, e.x), kWaveShl1, 0xf, 0xf,
                                           false));
    const float mn = __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, m), kWaveShl1, 0xf, 0xf,
                                           false));
    acc = fmaf((hn - e.x) + (mn - m), lw, acc);
  }
  return acc;
}

// ---------------------------------------------------------------------------
// 3b. sinogram -> image: one thread per pixel, BT instances, all views
// ---------------------------------------------------------------------------
// First walk-ordered bin worth testing for an axis point a: the inverse of
// the edge map, closed form per geometry, in FP32 with hardware reciprocals
// (v_rcp_f32) instead of IEEE divisions.  Only a starting guess; the exact
// bin is then fixed against the edge table with edge_pos().
__device__ __forceinline__ float guess_bin_real(const Geo2& g, const ViewGeo& vg, double a) {
  float kf;
  if (g.scan == DD_FAN_ARC) {
    // Fan angle of the ray through a relative to the detector centre,
    // d = gamma - theta_ref (mod pi): tan d = (Y cos - X sin) / (X cos + Y sin)
    // with (X, Y) the ray direction; atan by the odd polynomial of degree 13
    // with the least maximal error on [-1, 1] (3.2e-7 in FP32).  The staged
    // walk's windows start 1/16 bin early and a tile whose guess is later goes
    // the long way (walk_views_again): at 1e-5, the error of degree 9, a sixth
    // of the tiles and views of 4096 x 4096 pixels with 8e-5 rad a bin did.
    const float Y = vg.xaxis ? static_cast<float>(a - vg.sx) : vg.sxf;
    const float X = vg.xaxis ? vg.syf : static_cast<float>(a - vg.sy);
    const float num = Y * vg.cref - X * vg.sref;
    const float den = X * vg.cref + Y * vg.sref;
    const float t = fminf(fmaxf(num * __builtin_amdgcn_rcpf(den), -1.0f), 1.0f);
    const float t2 = t * t;
    const float d =
        t * (0.999996126f +
             t2 * (-0.333173692f +
                   t2 * (0.198078156f +
                         t2 * (-0.132333398f +
                               t2 * (0.0796236396f + t2 * (-0.0336041935f + t2 * 0.00681178458f))))));
    kf = g.D * 0.5f + (vg.flip ? -d : d) * __builtin_amdgcn_rcpf(g.det);
  } else if (g.scan == DD_FAN_FLAT) {
    const float R = g.sid, af = static_cast<float>(a);
    const float sf = static_cast<float>(vg.s), cf = static_cast<float>(vg.c);
    const float u = vg.xaxis ? R * af * cf * __builtin_amdgcn_rcpf(R + sf * af)
                             : R * af * sf * __builtin_amdgcn_rcpf(R - cf * af);
    const float vdet = g.sid / g.sdd * g.det, vbin = g.sid / g.sdd * g.bin;
    kf = g.D * 0.5f + (vg.flip ? -(u - vbin) : (u - vbin)) * __builtin_amdgcn_rcpf(vdet);
  } else {
    const float u = static_cast<float>(vg.xaxis ? a * vg.c : a * vg.s);
    kf = g.D * 0.5f + (vg.flip ? -(u - g.bin) : (u - g.bin)) * __builtin_amdgcn_rcpf(g.det);
  }
  return kf;
}

__device__ __forceinline__ int guess_bin_fast(const Geo2& g, const ViewGeo& vg, double a) {
  const float kf = fminf(fmaxf(guess_bin_real(g, vg, a), -4.0f), g.D + 4.0f);
  return static_cast<int>(floorf(kf));
}

// Adds the bins from k on that reach the pixel, given the search's state
// (u1, u2: bin k's edges; k the last bin whose lower edge lies before the
// pixel, or 0): overlap * weight * sinogram, bins ascending.
template <int BT>
__device__ __forceinline__ void pixel_walk(const Geo2& g, const double* __restrict__ ev,
                                           const PixelFrame& fr, double u1, double u2, int k,
                                           float gw, const float* __restrict__ sv,
                                           float (&acc)[BT]) {
  float p1 = pixel_fraction(u1);
  while (u1 < 1.0) {
    const float p2 = pixel_fraction(u2);
    const float w = (p2 - p1) * gw;
    float q[BT];
    load_sino<BT>(g, sv, k, q);
#pragma unroll
    for (int b = 0; b < BT; ++b) acc[b] = fmaf(w, q[b], acc[b]);
    if (++k >= g.D) break;
    u1 = u2;
    p1 = p2;
    if (u1 >= 1.0) break;
    u2 = fr.at(ev[k + 1]);
  }
}

// Contribution of view v to pixel (r, c): find the bins whose edges bracket
// the pixel in its line (closed-form guess, fixed exactly against the edge
// table), then accumulate overlap * weight * sinogram.
template <int BT, int WM>
__device__ __forceinline__ void pixel_one_view(
    const Geo2& g, const ViewGeo& vg, int v, const double* __restrict__ edges,
    const LineGeo* __restrict__ lines, const float* __restrict__ pint,
    const float* __restrict__ sino, int r, int c, int b0, float xcw, float ycw,
    float (&acc)[BT]) {
  // line geometry loaded in the branch, so a caller whose row r is
  // wave-uniform gets scalar loads on row-axis views
  int i;
  LineGeo lg;
  float pl;
  if (vg.xaxis) {
    i = c;
    lg = lines[static_cast<size_t>(v) * g.Lmax + r];
    pl = pint[static_cast<size_t>(v) * g.Lmax + r];
  } else {
    i = g.H - 1 - r;
    lg = lines[static_cast<size_t>(v) * g.Lmax + c];
    pl = pint[static_cast<size_t>(v) * g.Lmax + c];
  }
  const double* __restrict__ ev = edges + static_cast<size_t>(v) * (g.D + 1);
  const PixelFrame fr(lg.a0, lg.inv_p, i);
  // k = the last bin whose lower edge lies before pixel i (or 0): unique,
  // whatever the guess
  int k = min(max(guess_bin_fast(g, vg, lg.a0 + (i + 0.5) * static_cast<double>(pl)), 0),
              g.D - 1);
  double u1 = fr.at(ev[k]);
  while (k > 0 && u1 >= 0.0) u1 = fr.at(ev[--k]);
  double u2 = fr.at(ev[k + 1]);
  while (u2 < 0.0) {
    if (++k >= g.D) return;
    u1 = u2;
    u2 = fr.at(ev[k + 1]);
  }
  float gw = (WM == W_FP) ? pl : bp_const(g);
  if constexpr (WM == W_BPW) gw *= fbp_weight(g, vg, xcw, ycw);
  pixel_walk<BT>(g, ev, fr, u1, u2, k, gw, sino_view<BT>(g, sino, v, b0), acc);
}

// First-bin guess for the pixel centred at (xc, yc) from the view alone: the
// axis coordinate of the ray from the source through the centre (the line's
// pixel-edge map evaluated at the centre), in FP32.  It needs no per-line
// table, so a view's search can be started before the previous view's walk.
// Only a guess: the search below it is exact whatever it returns.
__device__ __forceinline__ int guess_bin_centre(const Geo2& g, const ViewGeo& vg, float xc,
                                                float yc) {
  float a;
  if (g.scan == DD_PARA) {
    const float s = static_cast<float>(vg.s), c = static_cast<float>(vg.c);
    a = vg.xaxis ? xc + yc * s * __builtin_amdgcn_rcpf(c) : yc + xc * c * __builtin_amdgcn_rcpf(s);
  } else {
    a = vg.xaxis ? (vg.sxf * yc - vg.syf * xc) * __builtin_amdgcn_rcpf(yc - vg.syf)
                 : (vg.syf * xc - vg.sxf * yc) * __builtin_amdgcn_rcpf(xc - vg.sxf);
  }
  return min(max(guess_bin_fast(g, vg, static_cast<double>(a)), 0), g.D - 1);
}

// What a pixel's search in one view starts from: the line's pixel-edge map,
// the guessed bin and that bin's two edges, all loaded ahead.
struct PixViewStart {
  LineGeo lg;
  float pl;
  int k0;
  double ea, eb;  // edges k0 and k0 + 1
};

__device__ __forceinline__ PixViewStart pixel_view_start(
    const Geo2& g, const ViewGeo& vg, int v, const double* __restrict__ edges,
    const LineGeo* __restrict__ lines, const float* __restrict__ pint, int r, int c, float xc,
    float yc) {
  PixViewStart s;
  // a branch per axis, so a caller whose row r is wave-uniform gets scalar
  // loads on row-axis views
  if (vg.xaxis) {
    s.lg = lines[static_cast<size_t>(v) * g.Lmax + r];
    s.pl = pint[static_cast<size_t>(v) * g.Lmax + r];
  } else {
    s.lg = lines[static_cast<size_t>(v) * g.Lmax + c];
    s.pl = pint[static_cast<size_t>(v) * g.Lmax + c];
  }
  s.k0 = guess_bin_centre(g, vg, xc, yc);
  const double* __restrict__ ev = edges + static_cast<size_t>(v) * (g.D + 1);
  s.ea = ev[s.k0];
  s.eb = ev[s.k0 + 1];
  return s;
}

// pixel_one_view from a start loaded ahead: the same search (going down, the
// old lower edge becomes the upper one), the same walk.  Same bins, same
// order, same values: equal bit for bit.
template <int BT, int WM>
__device__ __forceinline__ void pixel_view_from(
    const Geo2& g, const ViewGeo& vg, int v, const double* __restrict__ edges,
    const PixViewStart& s, const float* __restrict__ sino, int r, int c, int b0, float xcw,
    float ycw, float (&acc)[BT]) {
  const int i = vg.xaxis ? c : g.H - 1 - r;
  const double* __restrict__ ev = edges + static_cast<size_t>(v) * (g.D + 1);
  const PixelFrame fr(s.lg.a0, s.lg.inv_p, i);
  int k = s.k0;
  double u1 = fr.at(s.ea), u2 = fr.at(s.eb);
  while (k > 0 && u1 >= 0.0) {
    u2 = u1;
    u1 = fr.at(ev[--k]);
  }
  while (u2 < 0.0) {
    if (++k >= g.D) return;
    u1 = u2;
    u2 = fr.at(ev[k + 1]);
  }
  float gw = (WM == W_FP) ? s.pl : bp_const(g);
  if constexpr (WM == W_BPW) gw *= fbp_weight(g, vg, xcw, ycw);
  pixel_walk<BT>(g, ev, fr, u1, u2, k, gw, sino_view<BT>(g, sino, v, b0), acc);
}

// ---------------------------------------------------------------------------
// 3b'. sinogram -> image through running sums over the bins (one instance
// per geometry, no per-pixel weight)
// ---------------------------------------------------------------------------
// A pixel's value from one view is (G(i + 1) - G(i)) / P, G the running
// integral of the walk-ordered sinogram s (FP weight folded in) along the
// common axis, piecewise linear between the knots (e_k, R_k), R_k =
// sum_{j<k} s_j (e_{j+1} - e_j), k = 0 .. D.  The knots are FP64 (the running
// sum is kept as it is accumulated) and a view's table is {e_k, R_k}: one
// aligned 16-byte load per bin the walk visits, and no per-(bin, pixel)
// overlap terms at all.

// Knots of view v of one instance's sinogram p [V][D] (detector order) into
// that view's table tab[0 .. D] (walk order, s scaled by the FP weight when
// FOLD_W), by one workgroup of blockDim.x threads (a power of two <= 1024).
template <bool FOLD_W>
__device__ __forceinline__ void prefix_sino_view(
    const Geo2& g, const ViewGeo* __restrict__ views, const double* __restrict__ edges,
    const float* __restrict__ wfp, const float* __restrict__ p, int v, double2* __restrict__ tab,
    double* __restrict__ lds) {
  const int t = static_cast<int>(threadIdx.x), nt = static_cast<int>(blockDim.x);
  const int D = g.D;
  const int flip = views[v].flip;
  const double* __restrict__ ev = edges + static_cast<size_t>(v) * (D + 1);
  const float* __restrict__ pv = p + static_cast<size_t>(v) * D;
  auto term = [&](int k) {
    const float wk = FOLD_W ? wfp[static_cast<size_t>(v) * D + k] : 1.0f;
    return static_cast<double>(pv[flip ? D - 1 - k : k] * wk) * (ev[k + 1] - ev[k]);
  };
  const int seg = (D + nt - 1) / nt;
  const int k0 = min(t * seg, D), k1 = min(k0 + seg, D);
  double s = 0.0;
  for (int k = k0; k < k1; ++k) s += term(k);
  lds[t] = s;
  __syncthreads();
  for (int d = 1; d < nt; d *= 2) {
    const double add = (t >= d) ? lds[t - d] : 0.0;
    __syncthreads();
    lds[t] += add;
    __syncthreads();
  }
  double c = lds[t] - s;
  for (int k = k0; k < k1; ++k) {
    tab[k] = make_double2(ev[k], c);
    c += term(k);
  }
  if (t == nt - 1) tab[D] = make_double2(ev[D], lds[nt - 1]);
  __syncthreads();
}

// Adds view v's values of the pixels ib + pf .. ib + plst of one line to
// acc[pf .. plst] (times gw, the line's weight): one first-bin search, then
// the run's pixel edges and the bin edges merged in one monotone walk, G at
// each pixel edge interpolated between the two knots around it.  Knot k is
// kn[k - kmin]; the walk stays within bins kmin .. kmax - 1, which must hold
// every bin the run's pixel edges fall in (then the result does not depend
// on the range).  KP is a global or an LDS pointer to the knots as pairs of
// doubles {e, R}.
template <typename KP>
__device__ __forceinline__ double2 knot_at(KP kn, int i) {
  return make_double2(kn[2 * i], kn[2 * i + 1]);
}

template <int NP, typename KP>
__device__ __forceinline__ void pixel_run_view_prefix(
    const Geo2& g, const ViewGeo& vg, const LineGeo& lg, float pl, float gw, KP kn, int kmin,
    int kmax, int ib, int pf, int plst, float (&acc)[NP]) {
  // Positions relative to the run's edge ib (tau = e / P - a0 / P - ib) and
  // running sums relative to the first knot read (rho = R - rbase) are
  // formed in FP64 once per knot and kept in FP32: over a run of NP pixels
  // both stay of the size of a few pixels and bins, so FP32 holds them to
  // its precision relative to the values the pixels receive.
  const double bb = fma(lg.a0, lg.inv_p, static_cast<double>(ib));
  auto tau = [&](double e) { return static_cast<float>(fma(e, lg.inv_p, -bb)); };
  // the bin whose lower knot lies at or before the run's first pixel edge
  // (guessed at that edge)
  int k = min(max(guess_bin_fast(g, vg, lg.a0 + (ib + pf) * static_cast<double>(pl)), kmin),
              kmax - 1);
  double2 q = knot_at(kn, k - kmin);
  const double rbase = q.y;
  float t1 = tau(q.x), r1 = 0.0f;
  const float fpf = static_cast<float>(pf);
  while (k > kmin && t1 > fpf) {
    --k;
    q = knot_at(kn, k - kmin);
    t1 = tau(q.x);
    r1 = static_cast<float>(q.y - rbase);
  }
  q = knot_at(kn, k + 1 - kmin);
  float t2 = tau(q.x), r2 = static_cast<float>(q.y - rbase);
  float rw = __builtin_amdgcn_rcpf(t2 - t1);
  const float scale = static_cast<float>(lg.inv_p) * gw;
  float gprev = 0.0f;
#pragma unroll
  for (int j = 0; j <= NP; ++j) {
    if (j < pf || j > plst + 1) continue;
    const float dj = static_cast<float>(j);
    while (k < kmax - 1 && t2 <= dj) {
      ++k;
      t1 = t2;
      r1 = r2;
      q = knot_at(kn, k + 1 - kmin);
      t2 = tau(q.x);
      r2 = static_cast<float>(q.y - rbase);
      rw = __builtin_amdgcn_rcpf(t2 - t1);
    }
    // fraction of bin k below the edge, clamped: 0 below the first knot,
    // 1 past the last
    const float fr = __builtin_amdgcn_fmed3f((dj - t1) * rw, 0.0f, 1.0f);
    const float gv = fmaf(r2 - r1, fr, r1);
    if (j > pf) acc[j - 1] = fmaf(gv - gprev, scale, acc[j - 1]);
    gprev = gv;
  }
}

// One view's contribution to the Q x Q pixel block at (r0, c0) (nr x nc of
// it inside the image) through the view's knots (pixel_run_view_prefix).
// WM is W_FP or W_BP.
template <int WM, int Q, typename KP>
__device__ __forceinline__ void block_view_prefix(
    const Geo2& g, const ViewGeo& vg, const LineGeo* __restrict__ lv,
    const float* __restrict__ pv, KP kn, int kmin, int kmax, int r0, int c0, int nr, int nc,
    float (&acc)[Q][Q]) {
  static_assert(WM != W_BPW, "per-pixel weights need the bin walk");
  const float kbp = bp_const(g);
  if (vg.xaxis) {
#pragma unroll
    for (int dr = 0; dr < Q; ++dr) {
      if (dr >= nr) break;
      const int l = r0 + dr;
      const float pl = const_load(pv + l);
      pixel_run_view_prefix<Q>(g, vg, lv[l], pl, (WM == W_FP) ? pl : kbp, kn, kmin, kmax, c0,
                               0, nc - 1, acc[dr]);
    }
  } else {
    // lines = image columns c0 + dc, pixels read bottom-up: run position p
    // (pixel H - r0 - Q + p) is row r0 + Q - 1 - p, real when p >= Q - nr
#pragma unroll
    for (int dc = 0; dc < Q; ++dc) {
      if (dc >= nc) break;
      const int l = c0 + dc;
      const float pl = const_load(pv + l);
      float run[Q];
#pragma unroll
      for (int p = 0; p < Q; ++p) run[p] = acc[Q - 1 - p][dc];
      pixel_run_view_prefix<Q>(g, vg, lv[l], pl, (WM == W_FP) ? pl : kbp, kn, kmin, kmax,
                               g.H - r0 - Q, Q - nr, Q - 1, run);
#pragma unroll
      for (int p = 0; p < Q; ++p) acc[Q - 1 - p][dc] = run[p];
    }
  }
}

// Knot range [kb, ke] of view v that holds every pixel edge of the pixel
// tile [r0, r1) x [c0, c1) (image rows x columns): the tile's axis extent is
// spanned by its corners (a pixel edge's axis point is monotone along and
// across the lines), widened by one knot each side against rounding.
__device__ __forceinline__ int2 knot_range(const Geo2& g, const ViewGeo& vg,
                                           const double* __restrict__ ev,
                                           const LineGeo* __restrict__ lv, int r0, int r1,
                                           int c0, int c1) {
  double amin = 1e300, amax = -1e300;
  auto corner = [&](int l, int i) {
    const LineGeo lg = lv[l];
    const double a = lg.a0 + i / lg.inv_p;
    amin = fmin(amin, a);
    amax = fmax(amax, a);
  };
  if (vg.xaxis) {  // lines = rows, pixel edges = columns
    corner(r0, c0), corner(r0, c1), corner(r1 - 1, c0), corner(r1 - 1, c1);
  } else {  // lines = columns, pixel edges from the bottom
    corner(c0, g.H - r1), corner(c0, g.H - r0), corner(c1 - 1, g.H - r1),
        corner(c1 - 1, g.H - r0);
  }
  // last knot <= amin, first knot >= amax (edges ascend in walk order),
  // from the closed-form guesses
  int lo = min(max(guess_bin_fast(g, vg, amin), 0), g.D);
  while (lo > 0 && ev[lo] > amin) --lo;
  while (lo < g.D && ev[lo + 1] <= amin) ++lo;
  const int kb = max(lo - 1, 0);
  int hi = min(max(guess_bin_fast(g, vg, amax) + 1, 0), g.D);
  while (hi < g.D && ev[hi] < amax) ++hi;
  while (hi > 0 && ev[hi - 1] >= amax) --hi;
  const int ke = min(hi + 1, g.D);
  return make_int2(kb, max(ke, kb + 1));
}

// Views are summed in chunks, the chunk sums added in order: the same
// partition and order in every sinogram -> image walk, whether one wavefront
// takes all chunks or each chunk has its own, so a slice gets the same bits
// alone and in any batch.  Chunks are what a small image is split over the
// chip by (a 64 x 64 image is 16 wavefronts); their sums are also shorter, so
// rounding grows less over the views.
__host__ __device__ inline int walk_chunks(int views) {
  const int n = views / 8;
  return n < 1 ? 1 : n > 8 ? 8 : n;
}

__host__ __device__ inline int walk_chunk_begin(int views, int ch) {
  return static_cast<int>(1LL * views * ch / walk_chunks(views));
}

// sinogram -> image for one pixel, all views.  Each view's search is
// started (line map, guess, first two edges loaded) before the previous
// view's walk, so those loads overlap the walk's instead of opening the
// view; per view the same bins in the same order as pixel_one_view.
template <int BT, int WM>
__device__ __forceinline__ void pixels_body(
    const Geo2& g, const ViewGeo* __restrict__ views, const double* __restrict__ edges,
    const LineGeo* __restrict__ lines, const float* __restrict__ pint,
    const float* __restrict__ sino, float* __restrict__ out, int r, int c, int b0,
    const Epi& ep = Epi{}) {
  float xcw = 0.0f, ycw = 0.0f;
  pixel_centre(g, 1, r, c, &xcw, &ycw);
  float acc[BT], sum[BT];
  ViewGeo vg = views[0];
  PixViewStart cur = pixel_view_start(g, vg, 0, edges, lines, pint, r, c, xcw, ycw);
  const int nc = walk_chunks(g.V);
  for (int ch = 0, v = 0; ch < nc; ++ch) {
#pragma unroll
    for (int b = 0; b < BT; ++b) acc[b] = 0.0f;
    for (const int v1 = walk_chunk_begin(g.V, ch + 1); v < v1; ++v) {
      const int vn = min(v + 1, g.V - 1);
      const ViewGeo vgn = const_load(views + vn);
      const PixViewStart nxt = pixel_view_start(g, vgn, vn, edges, lines, pint, r, c, xcw, ycw);
      pixel_view_from<BT, WM>(g, vg, v, edges, cur, sino, r, c, b0, xcw, ycw, acc);
      vg = vgn;
      cur = nxt;
    }
#pragma unroll
    for (int b = 0; b < BT; ++b) sum[b] = ch == 0 ? acc[b] : sum[b] + acc[b];
  }
#pragma unroll
  for (int b = 0; b < BT; ++b)
    if (b0 + b < g.B) {
      const size_t at = (static_cast<size_t>(b0 + b) * g.H + r) * g.W + c;
      out[at] = epi_value(ep, sum[b], at);
    }
}

// Adds view v to the two consecutive pixels i0, i0 + 1 of one line (i0 + 1 only
// when has1): one first-bin search, for i0, and one walk over the bins that
// reach either pixel, each loaded once.  A pixel's bins are those whose upper
// edge does not lie before it nor the lower past it, in its own frame: the set
// and order that pixel_one_view walks, so each sum is the same bit for bit.
template <int BT>
__device__ __forceinline__ void pixel_pair_view(
    const Geo2& g, const ViewGeo& vg, const double* __restrict__ ev, const LineGeo& lg, float pl,
    const float* __restrict__ sv, int i0, bool has1, float gw0, float gw1, float (&acc0)[BT],
    float (&acc1)[BT]) {
  const PixelFrame f0(lg.a0, lg.inv_p, i0), f1(lg.a0, lg.inv_p, i0 + 1);
  int k = min(max(guess_bin_fast(g, vg, lg.a0 + (i0 + 0.5) * static_cast<double>(pl)), 0),
              g.D - 1);
  double e1 = ev[k];
  while (k > 0 && f0.at(e1) >= 0.0) e1 = ev[--k];
  double e2 = ev[k + 1];
  while (f0.at(e2) < 0.0) {
    if (++k >= g.D) return;
    e1 = e2;
    e2 = ev[k + 1];
  }
  double u0 = f0.at(e1), u1 = f1.at(e1);
  while ((has1 ? u1 : u0) < 1.0) {
    const double v0 = f0.at(e2), v1 = f1.at(e2);
    float q[BT];
    load_sino<BT>(g, sv, k, q);
    if (u0 < 1.0) {
      const float w = (pixel_fraction(v0) - pixel_fraction(u0)) * gw0;
#pragma unroll
      for (int b = 0; b < BT; ++b) acc0[b] = fmaf(w, q[b], acc0[b]);
    }
    if (has1 && v1 >= 0.0) {
      const float w = (pixel_fraction(v1) - pixel_fraction(u1)) * gw1;
#pragma unroll
      for (int b = 0; b < BT; ++b) acc1[b] = fmaf(w, q[b], acc1[b]);
    }
    if (++k >= g.D) break;
    u0 = v0;
    u1 = v1;
    if ((has1 ? u1 : u0) >= 1.0) break;
    e2 = ev[k + 1];
  }
}

// sinogram -> image for the 2 x 2 pixels at (r0, c0), all views: per view two
// lines of two consecutive pixels, image rows r0, r0 + 1 or columns c0, c0 + 1
// (read bottom-up).  Equal bit for bit to pixels_body on each pixel.
template <int BT, int WM>
__device__ __forceinline__ void quads_body(
    const Geo2& g, const ViewGeo* __restrict__ views, const double* __restrict__ edges,
    const LineGeo* __restrict__ lines, const float* __restrict__ pint,
    const float* __restrict__ sino, float* __restrict__ out, int r0, int c0, int b0,
    const Epi& ep = Epi{}) {
  const bool hr = r0 + 1 < g.H, hc = c0 + 1 < g.W;
  float xc[2][2] = {}, yc[2][2] = {};  // [row][column]
  if constexpr (WM == W_BPW) {
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int c = 0; c < 2; ++c) pixel_centre(g, 1, r0 + r, c0 + c, &xc[r][c], &yc[r][c]);
  }
  float acc[2][2][BT], sum[2][2][BT];
  const int nc = walk_chunks(g.V);
  for (int ch = 0, v = 0; ch < nc; ++ch) {
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int b = 0; b < BT; ++b) acc[r][c][b] = 0.0f;
    for (const int v1 = walk_chunk_begin(g.V, ch + 1); v < v1; ++v) {
      const ViewGeo vg = const_load(views + v);
      const double* __restrict__ ev = edges + static_cast<size_t>(v) * (g.D + 1);
      const LineGeo* __restrict__ lv = lines + static_cast<size_t>(v) * g.Lmax;
      const float* __restrict__ pv = pint + static_cast<size_t>(v) * g.Lmax;
      const float* __restrict__ sv = sino_view<BT>(g, sino, v, b0);
      const float kbp = bp_const(g);
      auto weight = [&](float pl, int r, int c) {
        float w = (WM == W_FP) ? pl : kbp;
        if constexpr (WM == W_BPW) w *= fbp_weight(g, vg, xc[r][c], yc[r][c]);
        return w;
      };
      if (vg.xaxis) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          if (r == 1 && !hr) break;
          const float pl = pv[r0 + r];
          pixel_pair_view<BT>(g, vg, ev, lv[r0 + r], pl, sv, c0, hc, weight(pl, r, 0),
                              weight(pl, r, 1), acc[r][0], acc[r][1]);
        }
      } else {
        // pixel H - 1 - r: the pair is rows r0 + 1, r0, or the last row alone
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          if (c == 1 && !hc) break;
          const float pl = pv[c0 + c];
          const LineGeo lg = lv[c0 + c];
          if (hr)
            pixel_pair_view<BT>(g, vg, ev, lg, pl, sv, g.H - 2 - r0, true, weight(pl, 1, c),
                                weight(pl, 0, c), acc[1][c], acc[0][c]);
          else
            pixel_pair_view<BT>(g, vg, ev, lg, pl, sv, g.H - 1 - r0, false, weight(pl, 0, c), 0.0f,
                                acc[0][c], acc[1][c]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int b = 0; b < BT; ++b)
          sum[r][c][b] = ch == 0 ? acc[r][c][b] : sum[r][c][b] + acc[r][c][b];
  }
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < 2; ++c)
      if ((r == 0 || hr) && (c == 0 || hc))
#pragma unroll
        for (int b = 0; b < BT; ++b)
          if (b0 + b < g.B) {
            const size_t at = (static_cast<size_t>(b0 + b) * g.H + r0 + r) * g.W + c0 + c;
            out[at] = epi_value(ep, sum[r][c][b], at);
          }
}

// ---------------------------------------------------------------------------
// 3c. sinogram -> image: the staged walk, one wavefront per pixel tile
// ---------------------------------------------------------------------------
constexpr int kWalkW = 16;         // tile width in pixels (height 4 NP)
constexpr int kWalkRangeH = 8;     // rows of one entry of the range table
constexpr int kWalkSlots = 64;     // edge slots per view, one per lane
constexpr int kWalkEdges = 60;     // edges a view may stage; the rest is padding
constexpr float kWalkEarly = 0.0625f;  // bins a pixel's first bin is guessed early by

__host__ __device__ inline int walk_range_tiles(const Geo2& g) {
  return ((g.W + kWalkW - 1) / kWalkW) * ((g.H + kWalkRangeH - 1) / kWalkRangeH);
}

// First edge and edge count of one range entry (16 x 8 pixels of one view),
// packed; 255: not to be staged.
__device__ __forceinline__ unsigned pack_range(int2 r) {
  const int n = r.y - r.x + 1;
  return (static_cast<unsigned>(r.x) << 8) |
         static_cast<unsigned>(n > kWalkSlots || r.x >= (1 << 24) ? 255 : n);
}

// Entries [t0, ...) of one view's range table, every `step`th.
__device__ __forceinline__ void walk_ranges_view(const Geo2& g, const ViewGeo& vg,
                                                 const double* __restrict__ ev,
                                                 const LineGeo* __restrict__ lv, int t0, int step,
                                                 unsigned* __restrict__ out) {
  const int tx = (g.W + kWalkW - 1) / kWalkW, tiles = walk_range_tiles(g);
  for (int t = t0; t < tiles; t += step) {
    const int c0 = (t % tx) * kWalkW, r0 = (t / tx) * kWalkRangeH;
    out[t] = pack_range(
        knot_range(g, vg, ev, lv, r0, min(r0 + kWalkRangeH, g.H), c0, min(c0 + kWalkW, g.W)));
  }
}

// Rows per lane of the staged walk (tiles of 16 x 4 rows pixels), or 0 where
// the per-pixel kernel takes the op.  A taller tile shares each staged view
// over more pixels, but its edges have to fit the slots: a tile's diagonal
// spans at most its length over the bin's width at the image corner next to
// the source (beam divergence and a flat detector's slant included).  Where
// even 16 x 4 (8 rows of 16 below 8 instances) pixels do not fit, the walk
// would go back to single views' bins in memory all the time.
inline int walk_rows(const Geo2& g) {
  const double half = 0.5 * std::hypot(g.W * g.dx, g.H * g.dy) + std::hypot(g.shx, g.shy);
  double bin = std::fabs(g.det);  // smallest bin across the rays
  if (g.scan != DD_PARA) {
    const double near = g.sid - half;
    if (!(near > 0.0)) return 0;
    bin *= g.scan == DD_FAN_ARC ? near : near / g.sdd / std::hypot(1.0, half / near);
  }
  auto fits = [&](int rows) {
    return std::hypot(kWalkW * g.dx, 4.0 * rows * g.dy) / bin + 5.0 <= kWalkEdges;
  };
  const int most = g.BT >= 8 ? 2 : 4;
  if (fits(most)) return most;
  if (fits(most / 2)) return most / 2;
  return 0;
}

// Whether the walk takes the geometry at some instance tile (a plan's tables
// serve them all; the tiles of 8 and more stage the lower pixel tiles).
inline bool walk_stages(Geo2 g) {
  g.BT = 8;
  return walk_rows(g) > 0;
}

template <int BT>
struct WalkLds {
  double e[kWalkSlots];                    // bin edges from the tile's first on
  double2 line[kWalkW];                    // {a0, 1 / P} of the tile's lines
  float4 par[kWalkW];                      // {k0, k1, k2, P}: bin k0 + x (k1 + x k2) at tile pixel x
  __align__(16) float q[BT * kWalkSlots];  // sinogram values, quad planes [BT / 4][bin][4]
};

// What a lane fetches for one view ahead of its turn.
template <int BT>
struct WalkFetch {
  static constexpr int kQ = BT >= 8 ? BT / 2 : BT;  // values per lane
  double e;
  float q[kQ];
  LineGeo lg;
  float pl;
};

template <int BT>
__device__ __forceinline__ void walk_load_q(const float* __restrict__ q, int k, float (&v)[BT]) {
  if constexpr (BT >= 4) {
#pragma unroll
    for (int j = 0; j < BT / 4; ++j) {
      const float4 t = *reinterpret_cast<const float4*>(q + (j * kWalkSlots + k) * 4);
      v[4 * j] = t.x;
      v[4 * j + 1] = t.y;
      v[4 * j + 2] = t.z;
      v[4 * j + 3] = t.w;
    }
  } else if constexpr (BT == 2) {
    const float2 t = *reinterpret_cast<const float2*>(q + k * 2);
    v[0] = t.x;
    v[1] = t.y;
  } else {
    v[0] = q[k];
  }
}

// Whether a pixel's window starts at its first bin exactly (one more edge to
// place), or up to kWalkEarly before it (maybe one more bin to add, dear
// where a bin holds many values).
template <int BT>
constexpr bool walk_shift() {
  return BT >= 8;
}

// One staged view's bins for the tile: K bins per pixel from its first one on
// (K = 0: kd of them), every pixel's independent of the others', so that
// their LDS reads are in flight together.  Bins beside the pixel, and the
// padding before and past the detector, have weight or value 0.  Clears `ok`
// where a window does not hold the whole of a pixel inside the image.
// AXIS: the view's lines are image columns (0) or rows (1), or what the view
// says (-1).
template <int BT, int WM, int NP, int K, int AXIS>
__device__ __forceinline__ void walk_window(
    const Geo2& g, const ViewGeo& vg, const WalkLds<BT>& s, int n, int i0, int px, int py,
    const float (&xcw)[NP], const float (&ycw)[NP], const bool (&inside)[NP], int kd,
    float (&acc)[NP][BT], bool& ok) {
  constexpr int kTH = 4 * NP;
  // no code shared between the windows
  asm volatile("; window %0" ::"i"(4 * K + AXIS + 1) : "memory");
  // 16 values a bin: one bin after the other, or the loads that the scheduler
  // moves ahead spill
  constexpr bool kOneByOne = BT == 16;
  const int bins = K > 0 ? K : kd;
  const float klast = static_cast<float>(n - 2);
  // row j of the lane: line li + j dli, tile pixel x + j dx
  const bool rows = AXIS < 0 ? vg.xaxis != 0 : AXIS == 1;
  const int li = rows ? py : px, dli = rows ? 4 : 0;
  const int x0 = rows ? px : kTH - 1 - py, dx = rows ? 0 : -4;
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    const double2 lg = s.line[li + j * dli];
    const float4 par = s.par[li + j * dli];
    const PixelFrame fr(lg.x, lg.y, i0 + x0 + j * dx);
    const float x = static_cast<float>(x0 + j * dx);
    int k = static_cast<int>(
        __builtin_amdgcn_fmed3f(fmaf(x, fmaf(x, par.z, par.y), par.x), 0.0f, klast));
    float gw = (WM == W_FP) ? par.w : bp_const(g);
    if constexpr (WM == W_BPW) gw *= fbp_weight(g, vg, xcw[j], ycw[j]);
    float p0 = pixel_fraction(fr.at(s.e[k]));
    float p1 = pixel_fraction(fr.at(s.e[k + 1]));
    if constexpr (walk_shift<BT>()) {
      // leave out a bin that ends before the pixel
      const bool skip = p1 <= 0.0f;
      k += skip;
      p0 = skip ? p1 : p0;
      p1 = pixel_fraction(fr.at(s.e[k + 1]));
    }
    const float first = p0;
    auto add = [&](int m) {
      const float w = (p1 - p0) * gw;
      float q[BT];
      walk_load_q<BT>(s.q, K > 0 ? k + m : min(k + m, kWalkSlots - 1), q);
#pragma unroll
      for (int b = 0; b < BT; ++b) acc[j][b] = fmaf(w, q[b], acc[j][b]);
      if constexpr (kOneByOne) __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (K > 0) {
#pragma unroll
      for (int m = 0; m < K; ++m) {
        if (m > 0) {
          p0 = p1;
          p1 = pixel_fraction(fr.at(s.e[k + m + 1]));
        }
        add(m);
      }
    } else {
      add(0);
      for (int m = 1; m < bins; ++m) {
        p0 = p1;
        p1 = pixel_fraction(fr.at(s.e[min(k + m + 1, kWalkSlots - 1)]));
        add(m);
      }
    }
    ok = ok & ((p1 - first == 1.0f) | !inside[j]);
    if constexpr (kOneByOne) asm volatile("; row %0" ::"i"(j) : "memory");
  }
}

// Adds views [v0, v1) to the zeroed sums of the tile at (r0, c0): lane l owns
// column c0 + l % 16 and rows r0 + l / 16 + 4 j.  Per view the bin edges and
// sinogram values the tile can reach (range table) are staged in the
// wavefront's own LDS (no barrier; the next view's are fetched during this
// one), and every pixel takes its bins there: the first by a parabola through
// the bins under three pixel edges of its line, then as many as a pixel can
// meet at the view's bins per pixel (2 below one bin per pixel, 3 below two).
// Bins, order, overlaps and products are pixel_one_view's, beside terms of
// weight zero, so the sums are the same bit for bit.  If a view's range does
// not fit, a window does not hold its pixel, or a sum is not finite at the
// end (zero times an infinity is not zero), it returns false and the sums are
// to be formed by walk_views_again.
//
// Bound by VALU issue (about 60 instructions per pixel and view at one
// instance, two thirds of the cycles) and the LDS reads' latency.  The
// per-pixel walk it replaces searched and placed three to five edges per
// pixel in FP64 from global memory, one after the other, at about 200
// instructions.  ProjTrans of 512 x 512 x 720 views x 736 bins: one slice
// 1087 -> 350 us, 16 slices 1573 -> 939 us; 256 x 256 x 180 views parallel
// 206 -> 43 us.
// AXES: a window of its own for each direction of the lines.  Uneven batches
// gain 2.5 % by it (64 slices of 256^2 to 512^2: 5.73 -> 5.58 ms); a single
// slice of 512 x 512 x 720 views lost 1 %.
template <int BT, int WM, int NP, bool AXES = false>
__device__ __forceinline__ bool walk_views(
    const Geo2& g, const ViewGeo* __restrict__ views, const double* __restrict__ edges,
    const LineGeo* __restrict__ lines, const float* __restrict__ pint,
    const unsigned* __restrict__ ranges, const float* __restrict__ sino, int r0, int c0, int b0,
    int v0, int v1, float (&acc)[NP][BT], WalkLds<BT>& s) {
  constexpr int kTH = 4 * NP;  // tile height
  using F = WalkFetch<BT>;
  int lane = static_cast<int>(threadIdx.x) & 63;
  const int c = c0 + (lane & 15);
  const int rtx = (g.W + kWalkW - 1) / kWalkW;
  const int rty = (g.H + kWalkRangeH - 1) / kWalkRangeH;
  const int rtiles = rtx * rty;
  const size_t plane4 = static_cast<size_t>(g.V) * g.D * 4;
  float xcw[NP] = {}, ycw[NP] = {};
  if constexpr (WM == W_BPW) {
#pragma unroll
    for (int j = 0; j < NP; ++j)
      pixel_centre(g, 1, r0 + (lane >> 4) + 4 * j, c, &xcw[j], &ycw[j]);
  }
  bool inside[NP];
#pragma unroll
  for (int j = 0; j < NP; ++j) inside[j] = c < g.W && r0 + (lane >> 4) + 4 * j < g.H;
  // first edge and edge count of view v's range over the whole tile; a range
  // at the detector's start gets a padding edge before it
  auto range_of = [&](int v, int* kb) {
    const unsigned* __restrict__ rv =
        ranges + static_cast<size_t>(v) * rtiles + (r0 / kWalkRangeH) * rtx + c0 / kWalkW;
    unsigned w = const_load(rv);
    int lo = static_cast<int>(w >> 8), n = static_cast<int>(w & 255u), hi = lo + n;
    bool big = n == 255;
#pragma unroll
    for (int y = 1; y < (kTH + kWalkRangeH - 1) / kWalkRangeH; ++y) {
      w = const_load(rv + (r0 / kWalkRangeH + y < rty ? y * rtx : 0));
      const int l2 = static_cast<int>(w >> 8), n2 = static_cast<int>(w & 255u);
      big = big || n2 == 255;
      lo = min(lo, l2);
      hi = max(hi, l2 + n2);
    }
    if (lo == 0) lo = -1;
    *kb = lo;
    return big ? 255 : hi - lo;
  };
  auto load_quads = [&](const float* sv, int k, float* q) {  // BT >= 8: half the planes
#pragma unroll
    for (int m = 0; m < BT / 8; ++m) {
      const float4 t = *reinterpret_cast<const float4*>(
          sv + (2 * m + (lane >> 5)) * plane4 + static_cast<size_t>(k) * 4);
      q[4 * m] = t.x;
      q[4 * m + 1] = t.y;
      q[4 * m + 2] = t.z;
      q[4 * m + 3] = t.w;
    }
  };
  auto store_quads = [&](int slot, const float* q) {
#pragma unroll
    for (int m = 0; m < BT / 8; ++m)
      *reinterpret_cast<float4*>(s.q + ((2 * m + (lane >> 5)) * kWalkSlots + slot) * 4) =
          make_float4(q[4 * m], q[4 * m + 1], q[4 * m + 2], q[4 * m + 3]);
  };
  auto fetch = [&](const ViewGeo& vg, int v, int kb, int n, F& f) {
    const double* __restrict__ ev = edges + static_cast<size_t>(v) * (g.D + 1);
    const float* __restrict__ sv = sino_view<BT>(g, sino, v, b0);
    // padding lies before or past every pixel
    f.e = kb + lane < 0 ? -1e300 : 1e300;
    if (kb + lane >= 0 && lane < n) f.e = ev[kb + lane];
#pragma unroll
    for (int b = 0; b < F::kQ; ++b) f.q[b] = 0.0f;
    if constexpr (BT >= 8) {
      const int bin = lane & 31;
      if (kb + bin >= 0 && bin < n - 1) load_quads(sv, kb + bin, f.q);
    } else {
      if (kb + lane >= 0 && lane < n - 1)
        load_tile<BT>(sv + static_cast<size_t>(kb + lane) * g.Bp, f.q);
    }
    const int l = vg.xaxis ? min(r0 + (lane & 15), g.H - 1) : min(c0 + (lane & 15), g.W - 1);
    f.lg = lines[static_cast<size_t>(v) * g.Lmax + l];
    f.pl = pint[static_cast<size_t>(v) * g.Lmax + l];
  };
  bool ok = true;
  int kb = 0;
  ViewGeo vg = const_load(views + v0);
  int n = range_of(v0, &kb);
  F f;
  if (n <= kWalkEdges) fetch(vg, v0, kb, n, f);
  for (int v = v0; v < v1; ++v) {
    const int vn = min(v + 1, v1 - 1);
    const ViewGeo vgn = const_load(views + vn);
    int kbn = 0;
    const int nn = range_of(vn, &kbn);
    if (n > kWalkEdges || nn > kWalkEdges) {
      ok = false;
      break;
    }
    // what follows from the lane alone is cheaper formed again than kept in
    // registers over the views
    asm volatile("" : "+v"(lane));
    const int px = lane & 15, py = lane >> 4;
    // stage the view
    const int i0 = vg.xaxis ? c0 : g.H - r0 - kTH;  // the tile's first pixel on its lines
    s.e[lane] = f.e;
    if constexpr (BT >= 8) {
      store_quads(lane & 31, f.q);
      float q[F::kQ] = {};
      if (n > 32) {  // bins 32 on, not fetched ahead
        if (32 + (lane & 31) < n - 1)
          load_quads(sino_view<BT>(g, sino, v, b0), kb + 32 + (lane & 31), q);
        store_quads(32 + (lane & 31), q);
      } else if ((lane & 31) < 4) {
        store_quads(32 + (lane & 31), q);
      }
    } else if constexpr (BT == 4) {
      *reinterpret_cast<float4*>(s.q + lane * 4) = make_float4(f.q[0], f.q[1], f.q[2], f.q[3]);
    } else {
#pragma unroll
      for (int b = 0; b < BT; ++b) s.q[lane * BT + b] = f.q[b];
    }
    // the bins under each line's first, middle and last pixel edge in the
    // tile, and the parabola through them (off by hundredths of a bin)
    const int span = vg.xaxis ? kWalkW : kTH;
    const float inv = vg.xaxis ? 1.0f / kWalkW : 1.0f / kTH;
    const float k0 = guess_bin_real(
        g, vg, f.lg.a0 + (i0 + py * (span / 2)) * static_cast<double>(f.pl));
    const float km = __shfl_down(k0, 16), k1 = __shfl_down(k0, 32);
    const float b1 = (4.0f * km - 3.0f * k0 - k1) * inv;
    const float b2 = 2.0f * (k0 - 2.0f * km + k1) * inv * inv;
    float slope = 0.0f;  // most bins per pixel on the line
    if (lane < 16) {
      slope = fmaxf(b1, fmaf(2.0f * span, b2, b1));
      s.line[lane] = make_double2(f.lg.a0, f.lg.inv_p);
      s.par[lane] = make_float4(k0 - static_cast<float>(kb) - kWalkEarly, b1, b2, f.pl);
    }
    if (v + 1 < v1) fetch(vgn, vn, kbn, nn, f);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // bins of a pixel: those its extent (and an early start) can cross
    constexpr float kSlack = walk_shift<BT>() ? 0.03125f : 2 * kWalkEarly;
    auto window = [&](auto k, int kd) {
      constexpr int K = decltype(k)::value;
      auto go = [&](auto axis) {
        walk_window<BT, WM, NP, K, decltype(axis)::value>(g, vg, s, n, i0, px, py, xcw, ycw,
                                                          inside, kd, acc, ok);
      };
      if constexpr (!AXES)
        go(std::integral_constant<int, -1>{});
      else if (vg.xaxis)
        go(std::integral_constant<int, 1>{});
      else
        go(std::integral_constant<int, 0>{});
    };
    if (__all(slope < 1.0f - kSlack)) {
      window(std::integral_constant<int, 2>{}, 0);
    } else if (__all(slope < 2.0f - kSlack)) {
      window(std::integral_constant<int, 3>{}, 0);
    } else {
      int kd = 4;
      while (kd < kWalkEdges && !__all(slope < kd - 1 - kSlack)) ++kd;
      window(std::integral_constant<int, 0>{}, kd);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    vg = vgn;
    kb = kbn;
    n = nn;
  }
#pragma unroll
  for (int j = 0; j < NP; ++j)
#pragma unroll
    for (int b = 0; b < BT; ++b) ok = ok & (fabsf(acc[j][b]) < __builtin_inff());
  return __all(ok);
}

// The tile's sums of views [v0, v1) by pixel_one_view, chunk by chunk, given
// to put(row, value index, sum): what walk_views could not do.
template <int BT, int WM, int NP, typename Put>
__device__ __forceinline__ void walk_views_again(
    const Geo2& g, const ViewGeo* __restrict__ views, const double* __restrict__ edges,
    const LineGeo* __restrict__ lines, const float* __restrict__ pint,
    const float* __restrict__ sino, int r0, int c0, int b0, int ch0, int ch1, Put put) {
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const int c = c0 + (lane & 15);
#pragma unroll 1
  for (int j = 0; j < NP; ++j) {
    const int r = r0 + (lane >> 4) + 4 * j;
    if (c >= g.W || r >= g.H) continue;
    float xc = 0.0f, yc = 0.0f, sum[BT];
    if constexpr (WM == W_BPW) pixel_centre(g, 1, r, c, &xc, &yc);
#pragma unroll 1
    for (int ch = ch0; ch < ch1; ++ch) {
      float acc[BT];
#pragma unroll
      for (int b = 0; b < BT; ++b) acc[b] = 0.0f;
      const int v1 = walk_chunk_begin(g.V, ch + 1);
#pragma unroll 1
      for (int v = walk_chunk_begin(g.V, ch); v < v1; ++v)
        pixel_one_view<BT, WM>(g, views[v], v, edges, lines, pint, sino, r, c, b0, xc, yc, acc);
#pragma unroll
      for (int b = 0; b < BT; ++b) sum[b] = ch == ch0 ? acc[b] : sum[b] + acc[b];
    }
#pragma unroll
    for (int b = 0; b < BT; ++b) put(r, c, b, sum[b]);
  }
}

}  // namespace body2d
}  // namespace dd
