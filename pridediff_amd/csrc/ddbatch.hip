// Batched 2D projection of many instances of uneven size in one launch per
// phase.
//
// A batch is a list of instances, each with its own geometry (image size,
// detector, view count and angles) and its own slot in one packed image
// buffer and one packed sinogram buffer.  setup() builds every instance's
// FP64 geometry tables once and uploads a device descriptor table; run() is
// then a few launches per op for the whole batch — a layout phase, a gather
// phase (sinogram -> image: one launch per tile height of the staged walk and
// one for instances whose bins are too fine for it) and the sum over chunks —
// each a grid over a static list of work items (instance, view, bin block,
// line chunk), (instance, view, bin block) or (instance, pixel tile, view
// chunk), heaviest instances first: by default one workgroup per item, or a
// set number of workgroups that stride over the list.  No counters, no
// atomics, no host work: a run is capturable and replays bit-identically.
//
// The per-item arithmetic is the one of the one-call kernels
// (dd2d_body.h), so a batched result equals the per-instance call exactly.
// No counterpart in the reference (one launch per instance and op,
// deeprecon/cuda/dis2d/FanArcDisCUDA2d.cu:758-1016).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <new>
#include <numeric>
#include <vector>

#include "dd.h"
#include "dd2d_body.h"
#include "dd_common.h"
#include "dd_profile.h"

namespace dd {
namespace {

using namespace body2d;

// Device descriptor of one instance, as stored in the descriptor table at the
// start of the batch's device block: its tables and scratch are byte offsets
// into that block.  Kernels take the block's base as an argument and rebuild
// the pointers from it (BatchInst), so every access is a global-memory one
// (pointers read from memory would otherwise be generic: flat loads).
enum Region {
  kViews, kEdges, kWfp, kLines, kPint, kXrow, kXcol, kSino, kPart, kPrefRow, kPrefCol,
  kPrefSino, kKnotRange, kWalkRange, kWalkPart, kRegions
};

enum Phase {
  kLayoutImage = 0,
  kGatherBins = 1,
  kLayoutSino = 2,
  kGatherPixels = 3,  // sinogram -> image by the staged walk, tiles of 16 rows
  kReduceBins = 4,
  kGatherQuads = 5,   // running-sum sinogram -> image: 4 x 4 pixels a thread, same instances
  kLayoutPrefix = 6,  // running sums of every image row and column
  kSumPixels = 7,     // staged walk: partial images of the view chunks
  kGatherShort = 8,   // sinogram -> image by the staged walk, tiles of 8 rows
  kGatherFine = 9,    // sinogram -> image per pixel: bins too fine to stage
  kLayoutKnots = 10,  // running sums of the views of those instances
  kPhases = 11
};

struct BatchDesc {
  Geo2 g;
  int rows;    // rows per lane of the staged walk, 0: per-pixel gather
  int chunks;  // workgroups the views of a pixel tile are split over
  unsigned long long off[kRegions];
  long long img_off;   // floats, into the packed image buffer
  long long sino_off;  // floats, into the packed sinogram buffer
  int item0[kPhases];  // first work item of each phase
  int nitems[kPhases];
};

// One instance inside a kernel: the descriptor with typed pointers.
struct BatchInst {
  Geo2 g;
  int rows, chunks;
  ViewGeo* views;
  double* edges;
  float* wfp;
  LineGeo* lines;
  float* pint;
  float* xrow;         // layout scratch: image rows, interleaved
  float* xcol;         // layout scratch: image columns, bottom-up
  float* sino;         // layout scratch: sinogram in walk order
  float* part;         // partial bin sums per line chunk [kSplit][B][V][D]
  float4* prow;        // running sums of the rows [B][H][W + 1]
  float4* pcol;        // running sums of the columns, bottom-up [B][W][H + 1]
  double2* psino;      // running-sum knots over the bins per view [B][V][D + 1]
  unsigned* wrange;    // edges each 16 x 8 pixel tile needs, per view
  float* wpart;        // partial images [chunks][H][W] of the staged walk
  int2* krange;        // knots each 64 x 64 pixel tile needs, per view [V][tiles]
  long long img_off;
  long long sino_off;
};

constexpr int kBT = 1;  // one geometry per instance

// Block items of the running-sum adjoint: one thread per kBlockQ x kBlockQ
// pixel block (one first-bin search and one merge walk per line serve kBlockQ
// pixels), kQuadSide x kQuadSide threads per item.
constexpr int kBlockQ = 4;
constexpr int kQuadSide = 16;
constexpr int kQuadThreads = kQuadSide * kQuadSide;
constexpr int kQuadTile = kQuadSide * kBlockQ;  // pixels per quad item edge

__device__ __forceinline__ int find_inst(const char* __restrict__ mem, int n, int phase,
                                         int item) {
  const BatchDesc* __restrict__ desc = reinterpret_cast<const BatchDesc*>(mem);
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if (const_load(&desc[mid].item0[phase]) <= item) lo = mid; else hi = mid - 1;
  }
  return lo;
}

__device__ __forceinline__ BatchInst load_inst(char* __restrict__ mem, int i) {
  const BatchDesc& s = reinterpret_cast<const BatchDesc*>(mem)[i];
  BatchInst d;
  d.g = const_load(&s.g);
  d.rows = const_load(&s.rows);
  d.chunks = const_load(&s.chunks);
  d.wrange = reinterpret_cast<unsigned*>(mem + const_load(&s.off[kWalkRange]));
  d.wpart = reinterpret_cast<float*>(mem + const_load(&s.off[kWalkPart]));
  d.views = reinterpret_cast<ViewGeo*>(mem + const_load(&s.off[kViews]));
  d.edges = reinterpret_cast<double*>(mem + const_load(&s.off[kEdges]));
  d.wfp = reinterpret_cast<float*>(mem + const_load(&s.off[kWfp]));
  d.lines = reinterpret_cast<LineGeo*>(mem + const_load(&s.off[kLines]));
  d.pint = reinterpret_cast<float*>(mem + const_load(&s.off[kPint]));
  d.xrow = reinterpret_cast<float*>(mem + const_load(&s.off[kXrow]));
  d.xcol = reinterpret_cast<float*>(mem + const_load(&s.off[kXcol]));
  d.sino = reinterpret_cast<float*>(mem + const_load(&s.off[kSino]));
  d.part = reinterpret_cast<float*>(mem + const_load(&s.off[kPart]));
  d.prow = reinterpret_cast<float4*>(mem + const_load(&s.off[kPrefRow]));
  d.pcol = reinterpret_cast<float4*>(mem + const_load(&s.off[kPrefCol]));
  d.psino = reinterpret_cast<double2*>(mem + const_load(&s.off[kPrefSino]));
  d.krange = reinterpret_cast<int2*>(mem + const_load(&s.off[kKnotRange]));
  d.img_off = const_load(&s.img_off);
  d.sino_off = const_load(&s.sino_off);
  return d;
}

// First work item of instance i in a phase (read from the table, not the
// copy, so a runtime phase index does not put the copy in scratch memory).
__device__ __forceinline__ int item0_of(const char* __restrict__ mem, int i, int phase) {
  return const_load(&reinterpret_cast<const BatchDesc*>(mem)[i].item0[phase]);
}

__global__ __launch_bounds__(kThreads) void k_batch_setup(
    char* __restrict__ mem, const float* const* __restrict__ angles, int n_inst, int total) {
  const BatchDesc* __restrict__ desc = reinterpret_cast<const BatchDesc*>(mem);
  for (int item = blockIdx.x; item < total; item += gridDim.x) {
    // setup items: one per (instance, view); item0[kLayoutImage] is unused here,
    // so the per-instance view offsets are recomputed by a linear scan
    int i = 0, base = 0;
    while (i < n_inst - 1 && item >= base + desc[i].g.V) {
      base += desc[i].g.V;
      ++i;
    }
    const BatchInst d = load_inst(mem, i);
    setup2d_view(d.g, angles[i], d.views, d.edges, d.wfp, d.lines, d.pint, item - base);
    __syncthreads();
  }
}

// Per (instance, view): the edge range of every 16 x 8 pixels for the staged
// walk; where the bins are too fine for it, the knot range of every 64 x 64
// pixel tile for the LDS staging of k_batch_quads_prefix.  With few views in
// the whole batch, workgroup rows share a view's entries (setup of one 2048 x
// 2048 x 16 views 194 -> 40 us).
__global__ __launch_bounds__(kThreads) void k_batch_ranges(char* __restrict__ mem, int n_inst,
                                                           int total) {
  const BatchDesc* __restrict__ desc = reinterpret_cast<const BatchDesc*>(mem);
  for (int item = blockIdx.x; item < total; item += gridDim.x) {
    int i = 0, base = 0;
    while (i < n_inst - 1 && item >= base + desc[i].g.V) {
      base += desc[i].g.V;
      ++i;
    }
    const BatchInst d = load_inst(mem, i);
    const int v = item - base;
    const ViewGeo vg = const_load(d.views + v);
    const double* __restrict__ ev = d.edges + static_cast<size_t>(v) * (d.g.D + 1);
    const LineGeo* __restrict__ lv = d.lines + static_cast<size_t>(v) * d.g.Lmax;
    if (d.rows > 0) {
      walk_ranges_view(d.g, vg, ev, lv, blockIdx.y * blockDim.x + threadIdx.x,
                       gridDim.y * blockDim.x,
                       d.wrange + static_cast<size_t>(v) * walk_range_tiles(d.g));
    } else {
      const int tx = (d.g.W + kQuadTile - 1) / kQuadTile;
      const int tiles = tx * ((d.g.H + kQuadTile - 1) / kQuadTile);
      for (int t = blockIdx.y * blockDim.x + threadIdx.x; t < tiles;
           t += gridDim.y * blockDim.x) {
        const int c0 = (t % tx) * kQuadTile, r0 = (t / tx) * kQuadTile;
        d.krange[static_cast<size_t>(v) * tiles + t] =
            knot_range(d.g, vg, ev, lv, r0, min(r0 + kQuadTile, d.g.H), c0,
                       min(c0 + kQuadTile, d.g.W));
      }
    }
  }
}

template <bool FOLD_W>
__global__ __launch_bounds__(kThreads) void k_batch_layout(
    char* __restrict__ mem, int n_inst, int phase, int total,
    const float* __restrict__ in) {
  for (int item = blockIdx.x; item < total; item += gridDim.x) {
    const int i = find_inst(mem, n_inst, phase, item);
    const BatchInst d = load_inst(mem, i);
    const int local = item - item0_of(mem, i, phase);
    if (phase == kLayoutImage) {
      // item = (image row, instance tile); threads stride over the row
      const int h = local % d.g.H;
      const int b0 = (local / d.g.H) * kBT;
      for (int w = threadIdx.x; w < d.g.W; w += blockDim.x)
        interleave_image_px<kBT>(d.g, in + d.img_off, d.xrow, d.xcol, h, w, b0);
    } else {
      // item = (view, instance tile); threads stride over the bins
      const int v = local % d.g.V;
      const int b0 = (local / d.g.V) * kBT;
      for (int k = threadIdx.x; k < d.g.D; k += blockDim.x)
        interleave_sino_bin<kBT, FOLD_W>(d.g, d.views, d.wfp, in + d.sino_off, d.sino, v, k, b0);
    }
  }
}

// Running-sum items: (line, instance), the H rows first, then the W columns
// read bottom-up; one workgroup per line.
__global__ __launch_bounds__(kThreads) void k_batch_prefix(
    char* __restrict__ mem, int n_inst, int total, const float* __restrict__ in) {
  __shared__ double lds[kThreads];
  for (int item = blockIdx.x; item < total; item += gridDim.x) {
    const int i = find_inst(mem, n_inst, kLayoutPrefix, item);
    const BatchInst d = load_inst(mem, i);
    const int local = item - item0_of(mem, i, kLayoutPrefix);
    const int H = d.g.H, W = d.g.W;
    const int line = local % (H + W);
    const int b = local / (H + W);
    const float* __restrict__ img = in + d.img_off + static_cast<size_t>(b) * H * W;
    if (line < H)
      prefix_line(img + static_cast<size_t>(line) * W, 1, W,
                  d.prow + (static_cast<size_t>(b) * H + line) * prefix_entries(W), lds);
    else
      prefix_line(img + static_cast<size_t>(H - 1) * W + (line - H), -static_cast<long long>(W),
                  H, d.pcol + (static_cast<size_t>(b) * W + line - H) * prefix_entries(H), lds);
  }
}

// Gather-bins items: (block of kBinsPerWave bins, view, instance, line
// chunk), chunk fastest, one wavefront per item (a 64-thread workgroup), so
// instances whose bin count is not a multiple of 256 keep their lanes busy.
// Every instance's item count and first item are multiples of kSplit, so with
// a grid that is a multiple of 8 the chunk follows the XCD.
constexpr int kBinsWave = 64;  // threads per gather-bins workgroup

// PREFIX: the bins' line integrals come from the running-sum tables
// (bins_accumulate_prefix) instead of the pixel walk.
template <int WM, bool PREFIX>
__global__ __launch_bounds__(kBinsWave) void k_batch_bins(
    char* __restrict__ mem, int n_inst, int total) {
  for (int item = blockIdx.x; item < total; item += gridDim.x) {
    const int i = find_inst(mem, n_inst, kGatherBins, item);
    const BatchInst d = load_inst(mem, i);
    const int local = item - item0_of(mem, i, kGatherBins);
    const int chunk = local % kSplit;
    int rest = local / kSplit;
    const int kb_n = (d.g.D + kBinsPerWave - 1) / kBinsPerWave;
    const int lane = static_cast<int>(threadIdx.x);
    const int k = (rest % kb_n) * kBinsPerWave + lane;
    const bool edge_lane = lane == 63;
    rest /= kb_n;
    const int v = rest % d.g.V;
    const int b0 = (rest / d.g.V) * kBT;
    // the whole wave works every item (the edge exchange needs it); lanes
    // past the last bin use clamped edges and write nothing
    const ViewGeo vg = const_load(d.views + v);
    const int L = vg.xaxis ? d.g.H : d.g.W;
    const int N = vg.xaxis ? d.g.W : d.g.H;
    const double e1 = d.edges[static_cast<size_t>(v) * (d.g.D + 1) + min(k, d.g.D)];
    float acc[kBT];
#pragma unroll
    for (int b = 0; b < kBT; ++b) acc[b] = 0.0f;
    if constexpr (PREFIX) {
      const float4* __restrict__ tab =
          (vg.xaxis ? d.prow : d.pcol) + static_cast<size_t>(b0) * L * prefix_entries(N);
      acc[0] = bins_accumulate_prefix<WM>(e1, d.lines + static_cast<size_t>(v) * d.g.Lmax,
                                          d.pint + static_cast<size_t>(v) * d.g.Lmax, tab,
                                          bp_const(d.g), L * chunk / kSplit,
                                          L * (chunk + 1) / kSplit, N);
    } else {
      bins_accumulate<kBT, WM>(d.g, vg, e1, d.lines + static_cast<size_t>(v) * d.g.Lmax,
                               d.pint + static_cast<size_t>(v) * d.g.Lmax,
                               (vg.xaxis ? d.xrow : d.xcol) + b0, bp_const(d.g),
                               L * chunk / kSplit, L * (chunk + 1) / kSplit, N, acc, edge_lane);
    }
    if (edge_lane || k >= d.g.D) continue;
#pragma unroll
    for (int b = 0; b < kBT; ++b)
      d.part[((static_cast<size_t>(chunk) * d.g.Bp + b0 + b) * d.g.V + v) * d.g.D + k] = acc[b];
  }
}

// Reduce items: (view, bin block, instance): chunk sums in chunk order, times
// the bin weight, detector order (the arithmetic of k_bins_reduce).
template <int WM>
__global__ __launch_bounds__(kThreads) void k_batch_reduce(
    char* __restrict__ mem, int n_inst, int total, float* __restrict__ out) {
  for (int item = blockIdx.x; item < total; item += gridDim.x) {
    const int i = find_inst(mem, n_inst, kReduceBins, item);
    const BatchInst d = load_inst(mem, i);
    const int local = item - item0_of(mem, i, kReduceBins);
    const int kb_n = (d.g.D + kThreads - 1) / kThreads;
    const int k = (local % kb_n) * kThreads + threadIdx.x;
    const int v = (local / kb_n) % d.g.V;
    const int b = local / (kb_n * d.g.V);
    if (k >= d.g.D) continue;
    const size_t plane = static_cast<size_t>(d.g.Bp) * d.g.V * d.g.D;
    const size_t at = (static_cast<size_t>(b) * d.g.V + v) * d.g.D + k;
    float sum = d.part[at];
#pragma unroll
    for (int c = 1; c < kSplit; ++c) sum += d.part[c * plane + at];
    const ViewGeo vg = const_load(d.views + v);
    const int kk = vg.flip ? d.g.D - 1 - k : k;
    const float wk = (WM == W_FP) ? d.wfp[static_cast<size_t>(v) * d.g.D + k] : 1.0f;
    out[d.sino_off + (static_cast<size_t>(b) * d.g.V + v) * d.g.D + kk] = sum * wk;
  }
}

// One wavefront's share of a gather-pixels item: the staged walk of one pixel
// tile, over one view chunk (several workgroups per tile) or all of them.
template <int WM, int NP>
__device__ __forceinline__ void batch_walk_tile(const BatchInst& d, int tile, int chunk, int b0,
                                                float* __restrict__ out, WalkLds<kBT>& lds) {
  const int tx = (d.g.W + kWalkW - 1) / kWalkW;
  const int c0 = (tile % tx) * kWalkW, r0 = (tile / tx) * 4 * NP;
  const int nc = walk_chunks(d.g.V);
  const int ch0 = d.chunks > 1 ? chunk : 0, ch1 = d.chunks > 1 ? chunk + 1 : nc;
  const size_t n = static_cast<size_t>(d.g.H) * d.g.W;
  float* __restrict__ o = (d.chunks > 1 ? d.wpart + n * d.g.Bp * chunk : out + d.img_off) + n * b0;
  auto put = [&](int r, int c, int, float v) {
    if (c < d.g.W && r < d.g.H) o[static_cast<size_t>(r) * d.g.W + c] = v;
  };
  float acc[NP][kBT], sum[NP];
  for (int ch = ch0; ch < ch1; ++ch) {
#pragma unroll
    for (int j = 0; j < NP; ++j) acc[j][0] = 0.0f;
    if (!walk_views<kBT, WM, NP, true>(d.g, d.views, d.edges, d.lines, d.pint, d.wrange, d.sino,
                                       r0, c0, b0, walk_chunk_begin(d.g.V, ch),
                                       walk_chunk_begin(d.g.V, ch + 1), acc, lds)) {
      walk_views_again<kBT, WM, NP>(d.g, d.views, d.edges, d.lines, d.pint, d.sino, r0, c0, b0,
                                    ch0, ch1, put);
      return;
    }
#pragma unroll
    for (int j = 0; j < NP; ++j) sum[j] = ch == ch0 ? acc[j][0] : sum[j] + acc[j][0];
  }
  const int lane = static_cast<int>(threadIdx.x) & 63;
#pragma unroll
  for (int j = 0; j < NP; ++j) put(r0 + (lane >> 4) + 4 * j, c0 + (lane & 15), 0, sum[j]);
}

// Gather items of the staged walk: (four pixel tiles, view chunk) of the
// instances with NP rows per lane.  Bound by VALU issue and LDS latency, so
// waves count: one kernel for both heights, with views and descriptors in
// vector registers, had 155 of them (3 waves per SIMD), 8.25 ms for ProjTrans
// of 64 slices of 256^2 to 512^2; a kernel per height 7.95 (104 registers),
// views and descriptors through scalar loads (const_load) 5.6 (80).
template <int WM, int NP>
__global__ __launch_bounds__(kThreads)
__attribute__((amdgpu_waves_per_eu(WM == W_FP ? 6 : 4))) void k_batch_walk(
    char* __restrict__ mem, int n_inst, int total, float* __restrict__ out) {
  constexpr int kPhase = NP == 4 ? kGatherPixels : kGatherShort;
  __shared__ WalkLds<kBT> lds[kThreads / 64];
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / 64);
  for (int item = blockIdx.x; item < total; item += gridDim.x) {
    const int i = find_inst(mem, n_inst, kPhase, item);
    const BatchInst d = load_inst(mem, i);
    const int local = item - item0_of(mem, i, kPhase);
    const int tiles = ((d.g.W + kWalkW - 1) / kWalkW) * ((d.g.H + 4 * NP - 1) / (4 * NP));
    const int groups = (tiles + kThreads / 64 - 1) / (kThreads / 64);
    const int tile = (local / d.chunks) % groups * (kThreads / 64) + wave;
    if (tile < tiles)
      batch_walk_tile<WM, NP>(d, tile, local % d.chunks, local / d.chunks / groups * kBT, out,
                              lds[wave]);
  }
}

// Gather items of the instances whose bins are too fine to be staged: 16 x 16
// pixels.
template <int WM>
__global__ __launch_bounds__(kThreads) void k_batch_pixels(
    char* __restrict__ mem, int n_inst, int total, float* __restrict__ out) {
  for (int item = blockIdx.x; item < total; item += gridDim.x) {
    const int i = find_inst(mem, n_inst, kGatherFine, item);
    const BatchInst d = load_inst(mem, i);
    const int local = item - item0_of(mem, i, kGatherFine);
    const int tx = (d.g.W + kTile - 1) / kTile, ty = (d.g.H + kTile - 1) / kTile;
    const int t = local % (tx * ty);
    const int c = (t % tx) * kTile + (threadIdx.x % kTile);
    const int r = (t / tx) * kTile + (threadIdx.x / kTile);
    if (c < d.g.W && r < d.g.H)
      pixels_body<kBT, WM>(d.g, d.views, d.edges, d.lines, d.pint, d.sino, out + d.img_off, r, c,
                           local / (tx * ty) * kBT);
  }
}

// Sum items: 256 pixels of an instance whose views were split, chunk sums in
// chunk order.
__global__ __launch_bounds__(kThreads) void k_batch_sum(
    char* __restrict__ mem, int n_inst, int total, float* __restrict__ out) {
  for (int item = blockIdx.x; item < total; item += gridDim.x) {
    const int i = find_inst(mem, n_inst, kSumPixels, item);
    const BatchInst d = load_inst(mem, i);
    const size_t n = static_cast<size_t>(d.g.H) * d.g.W * d.g.Bp;
    const size_t at = static_cast<size_t>(item - item0_of(mem, i, kSumPixels)) * kThreads +
                      threadIdx.x;
    if (at >= n) continue;
    float s = d.wpart[at];
    for (int c = 1; c < d.chunks; ++c) s += d.wpart[c * n + at];
    out[d.img_off + at] = s;
  }
}

// Sinogram running-sum items: (view, instance) of the instances whose bins are
// too fine to be staged, one workgroup per view.
template <bool FOLD_W>
__global__ __launch_bounds__(kThreads) void k_batch_prefix_sino(
    char* __restrict__ mem, int n_inst, int total, const float* __restrict__ in) {
  __shared__ double lds[kThreads];
  for (int item = blockIdx.x; item < total; item += gridDim.x) {
    const int i = find_inst(mem, n_inst, kLayoutKnots, item);
    const BatchInst d = load_inst(mem, i);
    const int local = item - item0_of(mem, i, kLayoutKnots);
    const int v = local % d.g.V, b = local / d.g.V;
    prefix_sino_view<FOLD_W>(
        d.g, d.views, d.edges, d.wfp, in + d.sino_off + static_cast<size_t>(b) * d.g.V * d.g.D,
        v, d.psino + (static_cast<size_t>(b) * d.g.V + v) * (d.g.D + 1), lds);
  }
}

// Block items through the running sums over the bins: per view, the knots the
// item's 64 x 64 pixel tile needs are staged in LDS (one 16-byte load per
// thread, double-buffered: view v + 1's load is in flight while view v is
// walked, one barrier per view), and every 4-pixel run's merge walk reads
// them there.  A view whose range exceeds the buffer is walked from global
// memory; both give the same bits (the walk never leaves the range).  The
// walk keeps its positions and sums in FP32 relative to the run, so the
// kernel fits 5 waves per SIMD (96 VGPRs); at 4 (101) it measured 8 % slower.
constexpr int kKnotCap = kQuadThreads;  // knots staged per view

template <int WM>
__global__ __launch_bounds__(kQuadThreads)
__attribute__((amdgpu_waves_per_eu(5))) void k_batch_quads_prefix(
    char* __restrict__ mem, int n_inst, int total, float* __restrict__ out) {
  __shared__ double2 knots[2][kKnotCap];
  const int tid = static_cast<int>(threadIdx.x);
  for (int item = blockIdx.x; item < total; item += gridDim.x) {
    const int i = find_inst(mem, n_inst, kGatherQuads, item);
    const BatchInst d = load_inst(mem, i);
    const int local = item - item0_of(mem, i, kGatherQuads);
    const int tx = (d.g.W + kQuadTile - 1) / kQuadTile;
    const int tiles = tx * ((d.g.H + kQuadTile - 1) / kQuadTile);
    const int t = local % tiles;
    const int b = local / tiles;
    const int c0 = (t % tx) * kQuadTile + kBlockQ * (tid % kQuadSide);
    const int r0 = (t / tx) * kQuadTile + kBlockQ * (tid / kQuadSide);
    const bool active = c0 < d.g.W && r0 < d.g.H;
    const int nr = min(kBlockQ, d.g.H - r0), nc = min(kBlockQ, d.g.W - c0);
    const double2* __restrict__ tab = d.psino + static_cast<size_t>(b) * d.g.V * (d.g.D + 1);
    const int2* __restrict__ rng = d.krange + t;  // view v at rng[v * tiles]
    float acc[kBlockQ][kBlockQ];
#pragma unroll
    for (int dr = 0; dr < kBlockQ; ++dr)
#pragma unroll
      for (int dc = 0; dc < kBlockQ; ++dc) acc[dr][dc] = 0.0f;
    // stage view 0
    int2 r = rng[0];
    bool staged = r.y - r.x + 1 <= kKnotCap;
    if (staged && tid <= r.y - r.x) knots[0][tid] = tab[r.x + tid];
    __syncthreads();
    for (int v = 0; v < d.g.V; ++v) {
      // the next view's knot for this thread, in flight during this view's walks
      const int vn = min(v + 1, d.g.V - 1);
      const int2 rn = rng[static_cast<size_t>(vn) * tiles];
      const bool staged_n = rn.y - rn.x + 1 <= kKnotCap;
      double2 kn = make_double2(0.0, 0.0);
      const bool mine = v + 1 < d.g.V && staged_n && tid <= rn.y - rn.x;
      if (mine) kn = tab[static_cast<size_t>(vn) * (d.g.D + 1) + rn.x + tid];
      if (active) {
        const ViewGeo vg = const_load(d.views + v);
        const LineGeo* __restrict__ lv = d.lines + static_cast<size_t>(v) * d.g.Lmax;
        const float* __restrict__ pv = d.pint + static_cast<size_t>(v) * d.g.Lmax;
        if (staged)
          block_view_prefix<WM, kBlockQ>(
              d.g, vg, lv, pv, (const __attribute__((address_space(3))) double*)(knots[v & 1]),
              r.x, r.y, r0, c0, nr, nc, acc);
        else
          block_view_prefix<WM, kBlockQ>(
              d.g, vg, lv, pv,
              reinterpret_cast<const double*>(tab + static_cast<size_t>(v) * (d.g.D + 1)), 0,
              d.g.D, r0, c0, nr, nc, acc);
      }
      if (mine) knots[(v + 1) & 1][tid] = kn;
      __syncthreads();
      r = rn;
      staged = staged_n;
    }
    if (active) {
      float* __restrict__ o = out + d.img_off + static_cast<size_t>(b) * d.g.H * d.g.W;
#pragma unroll
      for (int dr = 0; dr < kBlockQ; ++dr)
#pragma unroll
        for (int dc = 0; dc < kBlockQ; ++dc)
          if (dr < nr && dc < nc) o[static_cast<size_t>(r0 + dr) * d.g.W + c0 + dc] = acc[dr][dc];
    }
  }
}

}  // namespace
}  // namespace dd

using namespace dd;

struct dd2d_batch {
  std::vector<dd2d_batch_item> items;
  std::vector<BatchDesc> inst;   // host copy of the descriptors
  std::vector<int> order;        // instance order (heaviest first)
  size_t desc_off = 0, angles_off = 0, bytes = 0;
  size_t total_views = 0;
  int total[kPhases] = {};
  int grid = 0;                  // workgroups per launch (0 = one per work item)
  bool prefix = false;           // fine bins through running sums (DD_ADJ_BLOCK_PREFIX)
  bool fwd_prefix = false;       // image -> sinogram through running sums (DD_FWD_PREFIX)
  char* dev = nullptr;           // device memory given to setup()
};

namespace {

size_t take(size_t* off, size_t bytes) {
  const size_t at = *off;
  *off = align_up(*off + bytes, static_cast<size_t>(256));
  return at;
}

// Workgroups of one launch: the set grid (each workgroup strides over the
// items), or by default one workgroup per item, which measured fastest on
// the 64-instance fan-arc batch (21.3 ms per FP + adjoint vs 23.5 ms at 16
// workgroups per compute unit and 24.8 ms at 8).
int grid_for(const dd2d_batch* b, int total) {
  const int g = b->grid > 0 ? b->grid : total;
  return std::max(1, std::min(g, total));
}

// Largest partial images of a whole batch that its pixel tiles are split over
// their view chunks for (as in one-call ops: what the Infinity Cache holds).
constexpr unsigned long long kWalkPartBytes = 256ull << 20;

}  // namespace

extern "C" {

dd2d_batch* dd2d_batch_create(const dd2d_batch_item* items, int n) {
  if (!items || n <= 0) return nullptr;
  auto* b = new (std::nothrow) dd2d_batch();
  if (!b) return nullptr;
  b->items.assign(items, items + n);
  for (int i = 0; i < n; ++i) {
    const auto& it = items[i];
    if (it.scan < DD_PARA || it.scan > DD_FAN_ARC || it.views <= 0 || it.batch <= 0 ||
        it.geom.width <= 0 || it.geom.height <= 0 || it.geom.num_det <= 0 || !it.angles ||
        it.image_offset < 0 || it.sino_offset < 0) {
      delete b;
      return nullptr;
    }
  }
  // heaviest instances first, so the static item lists balance
  b->order.resize(n);
  std::iota(b->order.begin(), b->order.end(), 0);
  std::stable_sort(b->order.begin(), b->order.end(), [&](int x, int y) {
    const auto& a = items[x];
    const auto& c = items[y];
    return 1.0 * a.views * a.geom.width * a.geom.height * a.batch >
           1.0 * c.views * c.geom.width * c.geom.height * c.batch;
  });
  size_t off = 0;
  b->desc_off = take(&off, sizeof(BatchDesc) * n);  // 0: kernels find it at the block base
  b->angles_off = take(&off, sizeof(float*) * n);
  b->inst.resize(n);
  // staged walk: partial images of the whole batch
  unsigned long long parts = 0;
  for (int j = 0; j < n; ++j)
    parts += sizeof(float) * 1ull * walk_chunks(items[j].views) * items[j].geom.width *
             items[j].geom.height * items[j].batch;
  int acc[kPhases] = {};
  for (int j = 0; j < n; ++j) {
    const auto& it = items[b->order[j]];
    BatchDesc d{};
    Geo2& g = d.g;
    g.W = it.geom.width;
    g.H = it.geom.height;
    g.D = it.geom.num_det;
    g.V = it.views;
    g.B = it.batch;
    g.BT = kBT;
    g.Bp = it.batch;
    g.Lmax = std::max(g.W, g.H);
    g.scan = it.scan;
    g.dx = it.geom.pix_x;
    g.dy = it.geom.pix_y;
    g.det = it.geom.det;
    g.sid = it.geom.iso_source;
    g.sdd = it.geom.source_detector;
    g.shx = it.geom.shift_x;
    g.shy = it.geom.shift_y;
    g.bin = it.geom.bin_shift;
    // geometry tables and layout scratch: byte offsets into the device block
    d.off[kViews] = take(&off, sizeof(ViewGeo) * g.V);
    d.off[kEdges] = take(&off, sizeof(double) * g.V * (g.D + 1));
    d.off[kWfp] = take(&off, sizeof(float) * g.V * g.D);
    d.off[kLines] = take(&off, sizeof(LineGeo) * g.V * g.Lmax);
    d.off[kPint] = take(&off, sizeof(float) * g.V * g.Lmax);
    const size_t img = static_cast<size_t>(g.W) * g.H * g.Bp;
    d.off[kXrow] = take(&off, sizeof(float) * img);
    d.off[kXcol] = take(&off, sizeof(float) * img);
    d.off[kSino] = take(&off, sizeof(float) * g.V * g.D * g.Bp);
    d.off[kPart] =
        take(&off, sizeof(float) * static_cast<size_t>(kSplit) * g.Bp * g.V * g.D);
    d.off[kPrefRow] = take(&off, sizeof(float4) * static_cast<size_t>(g.Bp) * g.H *
                                     prefix_entries(g.W));
    d.off[kPrefCol] = take(&off, sizeof(float4) * static_cast<size_t>(g.Bp) * g.W *
                                     prefix_entries(g.H));
    d.rows = walk_rows(g);
    d.chunks = d.rows > 0 && parts <= kWalkPartBytes ? walk_chunks(g.V) : 1;
    const int tiles = it.batch;  // kBT == 1
    const int quads = ((g.W + kQuadTile - 1) / kQuadTile) * ((g.H + kQuadTile - 1) / kQuadTile);
    d.nitems[kLayoutSino] = g.V * tiles;
    if (d.rows > 0) {
      d.off[kWalkRange] = take(&off, sizeof(unsigned) * g.V * walk_range_tiles(g));
      if (d.chunks > 1)
        d.off[kWalkPart] = take(&off, sizeof(float) * static_cast<size_t>(d.chunks) * img);
      const int wt = ((g.W + kWalkW - 1) / kWalkW) * ((g.H + 4 * d.rows - 1) / (4 * d.rows));
      d.nitems[d.rows == 4 ? kGatherPixels : kGatherShort] = (wt + 3) / 4 * d.chunks * tiles;
    } else {
      d.off[kPrefSino] =
          take(&off, sizeof(double2) * static_cast<size_t>(g.Bp) * g.V * (g.D + 1));
      d.off[kKnotRange] = take(&off, sizeof(int2) * static_cast<size_t>(g.V) * quads);
      d.nitems[kGatherFine] = ((g.W + kTile - 1) / kTile) * ((g.H + kTile - 1) / kTile) * tiles;
      d.nitems[kLayoutKnots] = g.V * tiles;
      d.nitems[kGatherQuads] = quads * tiles;
    }
    d.img_off = it.image_offset;
    d.sino_off = it.sino_offset;
    d.nitems[kLayoutImage] = g.H * tiles;
    d.nitems[kGatherBins] = kSplit * g.V * ((g.D + kBinsPerWave - 1) / kBinsPerWave) * tiles;
    d.nitems[kReduceBins] = g.V * ((g.D + kThreads - 1) / kThreads) * it.batch;
    d.nitems[kSumPixels] = d.chunks > 1 ? static_cast<int>((img + kThreads - 1) / kThreads) : 0;
    d.nitems[kLayoutPrefix] = (g.H + g.W) * tiles;
    for (int ph = 0; ph < kPhases; ++ph) {
      d.item0[ph] = acc[ph];
      acc[ph] += d.nitems[ph];
    }
    b->total_views += g.V;
    b->inst[j] = d;
  }
  for (int ph = 0; ph < kPhases; ++ph) b->total[ph] = acc[ph];
  b->bytes = off;
  return b;
}

size_t dd2d_batch_device_bytes(const dd2d_batch* b) { return b ? b->bytes : 0; }

void dd2d_batch_set_grid(dd2d_batch* b, int workgroups) {
  if (b) b->grid = workgroups > 0 ? workgroups : 0;
}

void dd2d_batch_set_variant(dd2d_batch* b, int variant) {
  if (!b) return;
  b->prefix = (variant & ~DD_FWD_PREFIX) == DD_ADJ_BLOCK_PREFIX;
  b->fwd_prefix = (variant & DD_FWD_PREFIX) != 0;
}

dd_status dd2d_batch_setup(dd2d_batch* b, void* device_mem, size_t bytes, void* stream) {
  if (!b || !device_mem || bytes < b->bytes) return DD_NO_WORKSPACE;
  b->dev = static_cast<char*>(device_mem);
  auto st = static_cast<hipStream_t>(stream);
  const int n = static_cast<int>(b->inst.size());
  std::vector<const float*> angles(n);
  for (int j = 0; j < n; ++j) angles[j] = b->items[b->order[j]].angles;
  if (hipMemcpyAsync(b->dev + b->desc_off, b->inst.data(), sizeof(BatchDesc) * n,
                     hipMemcpyHostToDevice, st) != hipSuccess ||
      hipMemcpyAsync(b->dev + b->angles_off, angles.data(), sizeof(float*) * n,
                     hipMemcpyHostToDevice, st) != hipSuccess)
    return DD_LAUNCH_FAIL;
  const int total = static_cast<int>(b->total_views);
  hipLaunchKernelGGL(k_batch_setup, dim3(grid_for(b, total)), dim3(kThreads), 0, st, b->dev,
                     reinterpret_cast<const float* const*>(b->dev + b->angles_off), n, total);
  int most = 0;  // entries of a view
  for (const auto& d : b->inst) most = std::max(most, walk_range_tiles(d.g));
  const unsigned share = std::max(std::min(most / (2 * kThreads), 2048 / total), 1);
  hipLaunchKernelGGL(k_batch_ranges, dim3(grid_for(b, total), share), dim3(kThreads), 0, st,
                     b->dev, n, total);
  if (hipGetLastError() != hipSuccess) return DD_LAUNCH_FAIL;
  // the host staging vectors die with this call: wait for the uploads
  return hipStreamSynchronize(st) == hipSuccess ? DD_OK : DD_LAUNCH_FAIL;
}

dd_status dd2d_batch_run(const dd2d_batch* b, int op, const float* input, float* output,
                         void* stream) {
  if (!b || !b->dev || !input || !output) return DD_BAD_ARG;
  if (op < DD_PROJ || op > DD_BPROJ_TW) return DD_BAD_ARG;
  for (const auto& it : b->items)
    if (it.scan == DD_PARA && op >= DD_BPROJ_W) return DD_UNSUPPORTED;
  auto st = static_cast<hipStream_t>(stream);
  const int n = static_cast<int>(b->inst.size());
  char* inst = b->dev;  // descriptor table at the block base
  const bool sino_out = (op == DD_PROJ || op == DD_BPROJ_T || op == DD_BPROJ_TW);
  if (sino_out) {
    const int tot = b->total[kGatherBins], rtot = b->total[kReduceBins];
    // one-wave workgroups: four times the workgroups of the 256-thread phases
    const int bgrid = std::max(1, std::min(4 * grid_for(b, tot), tot));
    if (b->fwd_prefix && op != DD_BPROJ_TW) {
      // running sums of every line, then one lookup per (bin, line); the
      // weighted transpose keeps the pixel walk (its weight varies per pixel)
      ProfileScope prof(DD_KERNEL_IMAGE_TO_SINO, st);
      const int ptot = b->total[kLayoutPrefix];
      hipLaunchKernelGGL(k_batch_prefix, dim3(grid_for(b, ptot)), dim3(kThreads), 0, st, inst,
                         n, ptot, input);
      if (op == DD_PROJ) {
        hipLaunchKernelGGL((k_batch_bins<W_FP, true>), dim3(bgrid), dim3(kBinsWave), 0, st,
                           inst, n, tot);
        hipLaunchKernelGGL((k_batch_reduce<W_FP>), dim3(grid_for(b, rtot)), dim3(kThreads), 0,
                           st, inst, n, rtot, output);
      } else {
        hipLaunchKernelGGL((k_batch_bins<W_BP, true>), dim3(bgrid), dim3(kBinsWave), 0, st,
                           inst, n, tot);
        hipLaunchKernelGGL((k_batch_reduce<W_BP>), dim3(grid_for(b, rtot)), dim3(kThreads), 0,
                           st, inst, n, rtot, output);
      }
      return hipGetLastError() == hipSuccess ? DD_OK : DD_LAUNCH_FAIL;
    }
    hipLaunchKernelGGL((k_batch_layout<false>), dim3(grid_for(b, b->total[kLayoutImage])),
                       dim3(kThreads), 0, st, inst, n, static_cast<int>(kLayoutImage),
                       b->total[kLayoutImage], input);
    ProfileScope prof(DD_KERNEL_IMAGE_TO_SINO, st);
    if (op == DD_PROJ) {
      hipLaunchKernelGGL((k_batch_bins<W_FP, false>), dim3(bgrid), dim3(kBinsWave), 0, st, inst, n,
                         tot);
      hipLaunchKernelGGL((k_batch_reduce<W_FP>), dim3(grid_for(b, rtot)), dim3(kThreads), 0,
                         st, inst, n, rtot, output);
    } else if (op == DD_BPROJ_T) {
      hipLaunchKernelGGL((k_batch_bins<W_BP, false>), dim3(bgrid), dim3(kBinsWave), 0, st, inst, n,
                         tot);
      hipLaunchKernelGGL((k_batch_reduce<W_BP>), dim3(grid_for(b, rtot)), dim3(kThreads), 0,
                         st, inst, n, rtot, output);
    } else {
      hipLaunchKernelGGL((k_batch_bins<W_BPW, false>), dim3(bgrid), dim3(kBinsWave), 0, st, inst, n,
                         tot);
      hipLaunchKernelGGL((k_batch_reduce<W_BPW>), dim3(grid_for(b, rtot)), dim3(kThreads), 0,
                         st, inst, n, rtot, output);
    }
  } else {
    // The running sums (prefix) take only the instances whose bins are too
    // fine for the staged walk.  64 slices of 256^2 to 512^2, about one bin per
    // pixel: running sums 7.1 ms, walk 5.6 ms; 16 of 512^2 2.05 and 2.01 ms, 32
    // of 64^2 0.24 and 0.03 ms.  At 2 to 6 bins per pixel from 256^2 on, where
    // a tile's bins no longer fit the staging: 1.16 to 3.5 and, per pixel, 1.74
    // to 3.6 ms (32 of 256^2, 180 views).
    const bool prefix = b->prefix && op != DD_BPROJ_W;
    const int lt = b->total[kLayoutSino], kt = b->total[kLayoutKnots];
    const int wt = b->total[kGatherPixels], ht = b->total[kGatherShort];
    const int ft = b->total[kGatherFine], qt = b->total[kGatherQuads];
    const int stot = b->total[kSumPixels];
    if (!prefix || wt + ht > 0) {
      if (op == DD_PROJ_T)
        hipLaunchKernelGGL((k_batch_layout<true>), dim3(grid_for(b, lt)), dim3(kThreads), 0, st,
                           inst, n, static_cast<int>(kLayoutSino), lt, input);
      else
        hipLaunchKernelGGL((k_batch_layout<false>), dim3(grid_for(b, lt)), dim3(kThreads), 0, st,
                           inst, n, static_cast<int>(kLayoutSino), lt, input);
    }
    ProfileScope prof(DD_KERNEL_SINO_TO_IMAGE, st);
    auto run = [&](auto wm) {
      constexpr int WM = decltype(wm)::value;
      if (wt > 0)
        hipLaunchKernelGGL((k_batch_walk<WM, 4>), dim3(grid_for(b, wt)), dim3(kThreads), 0, st,
                           inst, n, wt, output);
      if (ht > 0)
        hipLaunchKernelGGL((k_batch_walk<WM, 2>), dim3(grid_for(b, ht)), dim3(kThreads), 0, st,
                           inst, n, ht, output);
      if (ft == 0) return;
      if constexpr (WM != W_BPW) {
        if (prefix) {
          // running sums of every view, then one merge walk per 4-pixel run
          hipLaunchKernelGGL((k_batch_prefix_sino<WM == W_FP>), dim3(grid_for(b, kt)),
                             dim3(kThreads), 0, st, inst, n, kt, input);
          hipLaunchKernelGGL((k_batch_quads_prefix<WM>), dim3(grid_for(b, qt)),
                             dim3(kQuadThreads), 0, st, inst, n, qt, output);
          return;
        }
      }
      hipLaunchKernelGGL((k_batch_pixels<WM>), dim3(grid_for(b, ft)), dim3(kThreads), 0, st,
                         inst, n, ft, output);
    };
    if (op == DD_PROJ_T)
      run(std::integral_constant<int, W_FP>{});
    else if (op == DD_BPROJ)
      run(std::integral_constant<int, W_BP>{});
    else
      run(std::integral_constant<int, W_BPW>{});
    if (stot > 0)
      hipLaunchKernelGGL(k_batch_sum, dim3(grid_for(b, stot)), dim3(kThreads), 0, st, inst, n,
                         stot, output);
  }
  return hipGetLastError() == hipSuccess ? DD_OK : DD_LAUNCH_FAIL;
}

void dd2d_batch_destroy(dd2d_batch* b) { delete b; }

}  // extern "C"
