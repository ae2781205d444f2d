// swr_raster.hpp -- the tile rasteriser (gfx950).
//
//   raster_batch_kernel  one workgroup per screen tile, one wave per 8x8
//                    block, one pixel per lane (a 2x2 quad in lanes
//                    4k..4k+3); the block's depth / stencil / colour live in
//                    registers while the wave walks the tile's primitive
//                    list in order: coverage, stencil, depth, shading, blend.
//
// The kernel's variants are compiled in translation units of their own
// (swr_raster_{blend,opaque}_{common,general}.hip), in parallel with the rest.
//
// Reference semantics: src/Device/QuadRasterizer.cpp,
// src/Pipeline/PixelRoutine.cpp, src/Pipeline/PixelProgram.cpp,
// src/Pipeline/SamplerCore.cpp.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "swr_device.hpp"
#include "swr_params.hpp"
#include "swr_raster_launch.hpp"
#include "swr_shade.hpp"
#include "swr_srgb.hpp"

namespace swr {

// Standard 4x sample locations relative to the pixel centre
// (Constants.hpp:26-47) and their 28.4 offsets Xf/Yf (Constants.cpp:291-297).
constexpr float kSampleX[4] = {-0.125f, 0.375f, -0.375f, 0.125f};
constexpr float kSampleY[4] = {-0.375f, -0.125f, 0.125f, 0.375f};
constexpr int kXf[4] = {-2, 6, -6, 2};
constexpr int kYf[4] = {-6, -2, 2, 6};

// D16 compares and stores Min(Max(Round(z * 0xFFFF), 0), 0xFFFF) of the
// clamped depth (PixelRoutine.cpp:506-510, 686-711; Round is to nearest even).
__device__ __forceinline__ float d16_value(float z) {
  return rr_min(rr_max(__builtin_rintf(z * 65535.0f), 0.0f), 65535.0f);
}

// B8G8R8A8 keeps R and B exchanged in memory (PixelRoutine.cpp:1091-1110,
// 2130-2143): the tile holds R8G8B8A8 order.
__device__ __forceinline__ uint32_t bgra_swap(int bgra, uint32_t v) {
  return bgra ? (v & 0xFF00FF00u) | ((v >> 16) & 0xFFu) | ((v & 0xFFu) << 16) : v;
}

// ---------------------------------------------------------------------------
// Tile rasteriser
// ---------------------------------------------------------------------------
// Work decomposition: one workgroup per 16x16 bin, one wavefront per 8x8
// block of the bin, one pixel per lane (lanes 4k..4k+3 form a 2x2 quad).
// Each wave walks the bin's triangle list in API order; the entries that may
// reach its block are compacted into batches of 64, every lane tests and
// sets up one of them (triangle-parallel), and the wave then applies them
// one by one (pixel-parallel) to the block's depth / stencil / colour, which
// stay in registers throughout.
//
// Coverage is the reference's span rule evaluated per sample point.  The
// reference walks each edge with an exact integer DDA that stores
// x = ceil(Xe(y) / 16) for rows [ceil(Y1/16), ceil(Y2/16)) into the left or
// right span, later edges overwriting earlier ones (SetupRoutine.cpp:
// 550-621), and a sample is covered iff left <= x < right
// (QuadRasterizer.cpp:181-206).  With
//   E(x, y) = DY * (16 x - X1) - DX * (16 y - Y1),   DY = Y2 - Y1 > 0,
// "ceil(Xe/16) <= x" is exactly E >= 0 and "x < ceil(Xe/16)" is exactly
// E < 0, so the span test becomes two integer sign tests per sample.
//
// A convex polygon needs no spans: over the rows it meets, one left and one
// right edge bound each row, so the rule equals its half planes.  With an
// edge a -> b in the order the reference walks it (interior at F > 0),
//   F(x, y) = (Yb - Ya) * (16 x - Xa) - (Xb - Xa) * (16 y - Ya),
// a sample is covered iff F >= 0 for left edges (Yb > Ya) and for horizontal
// top edges (Yb == Ya, Xb < Xa), and F > 0 for the others: left edges have
// F = E, right ones F = -E, and the horizontal ones keep the row range.  The
// F of a polygon add up to a constant (twice the area, signed by the
// winding), so a degenerate polygon, or one whose winding the float
// determinant of the setup misjudged, covers nothing under either rule.  F
// at the block origin is formed in 64 bits and clamped to +-2^30: beyond that
// its sign cannot change inside the block.  Edge extents below 2^15 (2047
// pixels) make the step over the block one 16-bit dot product.  Longer edges
// cross few of a polygon's blocks: where every one of them has the whole block on
// one side, its half plane is a constant there (or the polygon is out), and only
// the blocks that one crosses take the spans, edge by edge (3840x2160, 400 blended
// triangles of up to 4 M pixels: 1331 us with spans in every block, 960 now).
// The setup marks the polygons that qualify (kRecHalfPlanes, kRecWide: every
// triangle with coordinates below 2^20, and what clipping leaves convex on the
// 28.4 grid); the rest take the spans everywhere.

// Edge a -> b of a convex polygon as its half plane over the block at
// (ox, oy): pk holds (Yb - Ya, Xb - Xa) as 16-bit halves, and the sample at
// 28.4 offset (x, y) from the block's origin is inside iff
// dot2(pk, (x, -y)) + f >= 0.
__device__ __forceinline__ void half_plane(int Xa, int Ya, int Xb, int Yb, int ox, int oy, int &f, int &pk) {
  const int DX = Xb - Xa, DY = Yb - Ya;
  const bool closed = DY > 0 || (DY == 0 && DX < 0);
  const long long v = (long long)DY * (long long)(16 * ox - Xa) - (long long)DX * (long long)(16 * oy - Ya);
  const long long lim = 1ll << 30;
  f = (int)(v > lim ? lim : (v < -lim ? -lim : v)) - (closed ? 0 : 1);
  pk = (int)(((uint32_t)DY & 0xFFFFu) | ((uint32_t)DX << 16));
}

// The span rule at one sample point (28.4): whether the last left-writing
// edge spanning its row lies at or left of it, and the last right-writing one
// right of it.  Wave-uniform polygon, one point per lane.
template <typename VFetch>
__device__ __forceinline__ bool span_covers(const VFetch &vtx, int n, int d, int x, int y) {
  bool left = false, right = false;
  for (int i = 0; i < n; i++) {
    int ia = i + 1 - d, ib = i + d;
    ia = ia >= n ? ia - n : ia;
    ib = ib >= n ? ib - n : ib;
    int Xa, Ya, Xb, Yb;
    vtx(ia, Xa, Ya);
    vtx(ib, Xb, Yb);
    const bool swap = Yb < Ya;
    const int X1 = swap ? Xb : Xa, X2 = swap ? Xa : Xb;
    const int Y1 = swap ? Yb : Ya, Y2 = swap ? Ya : Yb;
    const long long E = (long long)(Y2 - Y1) * (long long)(x - X1) - (long long)(X2 - X1) * (long long)(y - Y1);
    const bool spans = Y1 <= y && y < Y2;
    if (swap) right = spans ? E < 0 : right;
    else left = spans ? E >= 0 : left;
  }
  return left && right;
}

typedef short Short2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ int dot2_i16(int a, int b, int c) {
  return __builtin_amdgcn_sdot2(__builtin_bit_cast(Short2, a), __builtin_bit_cast(Short2, b), c, false);
}

// Largest value of v over the wave (wave-uniform), by DPP: the old value of
// lanes without a source is the identity, so each step is one instruction.
__device__ __forceinline__ int wave_max_i32(int v) {
  v = max(v, __builtin_amdgcn_update_dpp(INT32_MIN, v, 0x111, 0xf, 0xf, false));  // row_shr:1
  v = max(v, __builtin_amdgcn_update_dpp(INT32_MIN, v, 0x112, 0xf, 0xf, false));  // row_shr:2
  v = max(v, __builtin_amdgcn_update_dpp(INT32_MIN, v, 0x114, 0xf, 0xf, false));  // row_shr:4
  v = max(v, __builtin_amdgcn_update_dpp(INT32_MIN, v, 0x118, 0xf, 0xf, false));  // row_shr:8
  v = max(v, __builtin_amdgcn_update_dpp(INT32_MIN, v, 0x142, 0xa, 0xf, false));  // row_bcast:15
  v = max(v, __builtin_amdgcn_update_dpp(INT32_MIN, v, 0x143, 0xc, 0xf, false));  // row_bcast:31
  return __builtin_amdgcn_readlane(v, 63);
}

// The lanes where p holds (all of them must be asked: as __ballot, without its
// detour through a vector register).
__device__ __forceinline__ uint64_t lanes_where(bool p) { return __builtin_amdgcn_ballot_w64(p); }

// The depth compare op as its result where the stored depth is above the
// fragment's (or either is NaN), equal to it, and below it: every op, with its
// results for NaN, is a function of stored <= z and stored < z.
struct DepthPass {
  bool above, equal, below;
  __device__ __forceinline__ bool operator()(float stored, float z) const {
    const bool le = stored <= z, lt = stored < z;
    return (lt & below) | (le & !lt & equal) | (!le & above);
  }
};
__device__ __forceinline__ DepthPass depth_pass(const DrawParams &P) {
  const bool inv = P.zInv != 0;
  const int k = P.zPred;  // le, lt, eq, true
  return {(k == 3) != inv, (k != 1) != inv, (k != 2) != inv};
}

// What a wave keeps of its block, per lane one pixel.  With BLEND the colours
// themselves; without it the primitive that last wrote each sample: an
// unblended fragment is replaced whole by the next one, so only the last one
// of a sample is shaded, once the list is done (4.7 fragments a pixel pass
// the depth test where 20 to 60 layers overlap).
template <int MS, bool FCOL, bool BLEND>
struct PixelState {
  float zb[MS];
  uint32_t sb[MS];
  uint32_t cb[BLEND && !FCOL ? MS : 1];
  float4 cf[BLEND && FCOL ? MS : 1];
  uint32_t id[BLEND && FCOL ? MS : 1];  // primitive_id record (float targets only)
  uint32_t last[BLEND ? 1 : MS];        // 1 + record slot of the last writer, 0 for none
};

// Pixel of lane `l` inside its 8x8 block: lanes 4k..4k+3 form the 2x2 quad
// k, quads in row-major order over the block.
__device__ __forceinline__ int lane_cx(int l) { return 2 * ((l >> 2) & 3) + (l & 1); }
__device__ __forceinline__ int lane_cy(int l) { return 2 * (l >> 4) + ((l >> 1) & 1); }

// Blend a shaded colour into the samples of this lane's pixel selected by
// xMask, then write (PixelRoutine.cpp:1617-2936).
// srgbLut: srgb_to_linear of every 8-bit code (sRGB targets).
// FAST: the blend is SRC_ALPHA, ONE_MINUS_SRC_ALPHA, ADD.
template <int MS, bool FCOL, bool XF, bool FAST = false>
__device__ __forceinline__ void blend_write(const DrawParams &P, PixelState<MS, FCOL, true> &S, float4 s, int xMask,
                                            uint32_t tri, const float *srgbLut) {
#pragma unroll
  for (int q = 0; q < MS; q++) {
    if (!((xMask >> q) & 1)) continue;
    float4 dst;
    if (FCOL) {
      dst = S.cf[FCOL ? q : 0];
    } else {
      const uint32_t p = S.cb[FCOL ? 0 : q];
      dst = make_float4(unorm8_to_float(p & 0xFFu), unorm8_to_float((p >> 8) & 0xFFu),
                        unorm8_to_float((p >> 16) & 0xFFu), unorm8_to_float(p >> 24));
      if (XF && P.colorSRGB) {  // blended in linear space (PixelRoutine.cpp:1811-1827)
        dst.x = srgbLut[p & 0xFFu];
        dst.y = srgbLut[(p >> 8) & 0xFFu];
        dst.z = srgbLut[(p >> 16) & 0xFFu];
      }
    }
    float4 o = FAST ? blend_src_alpha(s, dst) : alpha_blend<XF>(P, s, dst);
    if (!FCOL && (XF && P.colorSRGB)) {  // writeColor encodes R, G, B first (PixelRoutine.cpp:1963-1969)
      o.x = linear_to_srgb(o.x);
      o.y = linear_to_srgb(o.y);
      o.z = linear_to_srgb(o.z);
    }
    // Masked channels keep their value (selects, not branches).
    if (FCOL) {
      float4 &c = S.cf[FCOL ? q : 0];
      c.x = (P.colorMask & 1) ? o.x : c.x;
      c.y = (P.colorMask & 2) ? o.y : c.y;
      c.z = (P.colorMask & 4) ? o.z : c.z;
      c.w = (P.colorMask & 8) ? o.w : c.w;
      S.id[FCOL ? q : 0] = tri - (uint32_t)P.triBase + 1u;
    } else {
      const uint32_t wm = ((P.colorMask & 1) ? 0x000000FFu : 0u) | ((P.colorMask & 2) ? 0x0000FF00u : 0u) |
                          ((P.colorMask & 4) ? 0x00FF0000u : 0u) | ((P.colorMask & 8) ? 0xFF000000u : 0u);
      const uint32_t o8 = float4_to_unorm8(o);
      S.cb[FCOL ? 0 : q] = (S.cb[FCOL ? 0 : q] & ~wm) | (o8 & wm);
    }
  }
}

// Writes an unblended shaded colour to a pixel's samples selected by xMask
// (masked channels keep what the attachment holds), and the primitive_id
// record of float targets.
template <int MS, bool FCOL, bool XF>
__device__ __forceinline__ void store_color(const DrawParams &P, int colorMask, int px, int py, float4 o, int xMask,
                                            uint32_t tri) {
  uint32_t o8 = 0;
  if (!FCOL) {
    if (XF && P.colorSRGB) {  // writeColor encodes R, G, B first (PixelRoutine.cpp:1963-1969)
      o.x = linear_to_srgb(o.x);
      o.y = linear_to_srgb(o.y);
      o.z = linear_to_srgb(o.z);
    }
    o8 = bgra_swap(XF && P.colorBGRA, float4_to_unorm8(o));
  }
#pragma unroll
  for (int q = 0; q < MS; q++) {
    if (!((xMask >> q) & 1)) continue;
    char *at = P.color + q * P.colorSlice + (long long)py * P.colorPitch + (FCOL ? 16ll : 4ll) * px;
    if (FCOL) {
      float4 c = o;
      if (colorMask != 15) {
        const float4 d = *reinterpret_cast<const float4 *>(at);
        c.x = (colorMask & 1) ? c.x : d.x;
        c.y = (colorMask & 2) ? c.y : d.y;
        c.z = (colorMask & 4) ? c.z : d.z;
        c.w = (colorMask & 8) ? c.w : d.w;
      }
      *reinterpret_cast<float4 *>(at) = c;
      if (P.primId)
        *reinterpret_cast<uint32_t *>(P.primId + q * P.primIdSlice + (long long)py * P.primIdPitch + 4ll * px) =
            tri - (uint32_t)P.triBase + 1u;
    } else {
      uint32_t c = o8;
      if (colorMask != 15) {
        const uint32_t wm = bgra_swap(XF && P.colorBGRA, ((colorMask & 1) ? 0x000000FFu : 0u) |
                                                             ((colorMask & 2) ? 0x0000FF00u : 0u) |
                                                             ((colorMask & 4) ? 0x00FF0000u : 0u) |
                                                             ((colorMask & 8) ? 0xFF000000u : 0u));
        c = (*reinterpret_cast<const uint32_t *>(at) & ~wm) | (c & wm);
      }
      *reinterpret_cast<uint32_t *>(at) = c;
    }
  }
}

constexpr int kQueue = 128;  // deferred-shading queue entries per wave: two batches of 64

// LDS of one wave.  A workgroup has one to four waves (a tile is 8 or 16 pixels
// a side) and takes one of these for each, dynamically: sized for four, the
// workgroups of smaller tiles left most of it unused and a CU had five or six of
// them (1280x720, 30,000 triangles, 8x8 tiles, us a draw: textured and blended
// 480 -> 339, 4x 1088 -> 559, sRGB with stencil 921 -> 490; 16x8: 317 -> 247,
// 735 -> 552, 568 -> 424).
template <int MS, int LEVEL, bool BLEND>
struct WaveLds {
  // Without blending, one pixel is one fragment unless it has samples.
  static constexpr bool kQueued = BLEND || MS > 1;
  // Chunks of the list that raster_tile loads at a time, and the ring of entries
  // that wait: at least 63 + 64 * kChunks, a power of two.
  static constexpr int kChunks = LEVEL == 0 || (MS > 1 && !BLEND) ? 2 : 4;
  static constexpr uint32_t kRing = 128 * kChunks;
  int4 cand[3][64];   // a batch of candidates (see raster_tile)
  int4 candMore[64];  // and the further half planes of polygons
  float4 qCol[kQueued ? 64 : 1];
  uint32_t qTri[kQueued ? kQueue : 2];
  uint32_t qPix[kQueued ? kQueue : 2];
  uint32_t ring[kRing];
};

extern __shared__ int4 waveLds[];

// One screen tile of draw P: `bin` is the tile's index in the draw's tile
// grid, [start, end) its range of the sorted (tile, primitive) list.  The
// workgroup has one wave per 8x8 block of the tile.
// LEVEL 1: the draw has no stencil and no depth bias, tests and writes
// depth and writes all four colour channels (the checks below fold away).
// LEVEL 2 (3): also the common shading state with REPEAT (CLAMP_TO_EDGE)
// addressing (shade's FA, blend_write's FAST).
// BLEND: the draw blends (see PixelState).
template <int MS, bool FCOL, bool FTEX, bool XF, int LEVEL, bool BLEND>
__device__ __forceinline__ void raster_tile(const DrawParams &P, int bin, uint32_t start, uint32_t end0,
                                            const TriRecord *__restrict__ rec, const int *__restrict__ poly,
                                            const uint32_t *__restrict__ binTri) {
  constexpr bool SIMPLE = LEVEL >= 1, FAST = LEVEL >= 2;
  constexpr int FA = LEVEL >= 2 ? LEVEL - 2 : -1;
  const bool stencilActive = !SIMPLE && P.stencilActive, stencilWrite = !SIMPLE && P.stencilWrite;
  const bool depthBias = !SIMPLE && P.depthBias, depthTest = SIMPLE || P.depthTest;
  const bool depthWrite = SIMPLE || P.depthWrite;
  const int colorMask = SIMPLE ? 15 : P.colorMask;
  // What the candidate loop asks of the draw, loaded here: read in the branches
  // that use them, the fields cost a scalar load and a wait each per candidate,
  // and a target of few blocks has one wave per SIMD, which nothing hides them
  // behind (300x169 pixels, 40,000 blended triangles in display formats with
  // stencil: 1137 us a draw, 830 with the stencil table and the compares below
  // as well).  With four samples the common states need the registers: their
  // depth range is read where it is used (4x frame 566 -> 562 us).
  constexpr bool KEEP_RANGE = !(SIMPLE && MS > 1);
  const int msMask = P.msMask, depthCompare = P.depthCompare;
  const DepthPass zp = depth_pass(P);
  const float rangeLo = P.depthClampLo, rangeHi = P.depthClampHi;
  auto range_lo = [&]() __attribute__((always_inline)) { return KEEP_RANGE ? rangeLo : P.depthClampLo; };
  auto range_hi = [&]() __attribute__((always_inline)) { return KEEP_RANGE ? rangeHi : P.depthClampHi; };
  const bool depth16 = XF && P.depth16, depthBounds = XF && P.depthBounds, alphaToCoverage = XF && P.alphaToCoverage;
  // Per-wave queue of fragments that passed the tests and await shading,
  // in API order: primitive, owner lane | sample mask << 8, shaded colour.
  using Lds = WaveLds<MS, LEVEL, BLEND>;
  constexpr bool QUEUE = Lds::kQueued;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // scalar, as what follows from it: frees up to 14 vector registers
  Lds &W = reinterpret_cast<Lds *>(waveLds)[wave];
  const int bx = bin % P.tilesX, by = bin / P.tilesX;
  const int bw = P.tileW >> 3;  // 8x8 blocks per tile row
  const int ox = bx * P.tileW + 8 * (wave % bw), oy = by * P.tileH + 8 * (wave / bw);
  const int cx = lane_cx(lane), cy = lane_cy(lane);
  const int px = ox + cx, py = oy + cy;
  const int myBit = cy * 8 + cx;

  // A block outside the scissor walks no list (no early return: the
  // workgroup reduces its counters together at the end).
  const bool waveActive = !(ox >= P.sx1 || oy >= P.sy1 || ox + 8 <= P.sx0 || oy + 8 <= P.sy0);
  const uint32_t end = waveActive ? end0 : start;

  uint64_t scissorMask = 0;
  {
    uint32_t cols = 0;
#pragma unroll
    for (int c = 0; c < 8; c++)
      if (ox + c >= P.sx0 && ox + c < P.sx1) cols |= 1u << c;
#pragma unroll
    for (int r = 0; r < 8; r++)
      if (oy + r >= P.sy0 && oy + r < P.sy1) scissorMask |= (uint64_t)cols << (8 * r);
  }
  const bool inside = (scissorMask >> myBit) & 1;

  PixelState<MS, FCOL, BLEND> S;
#pragma unroll
  for (int q = 0; q < MS; q++) {
    S.zb[q] = 0.0f;
    S.sb[q] = 0;
    if constexpr (!BLEND) S.last[q] = 0;
    else if constexpr (FCOL) S.cf[q] = make_float4(0, 0, 0, 0), S.id[q] = 0;
    else S.cb[q] = 0;
    if (!inside) continue;
    if constexpr (BLEND && FCOL)
      if (P.primId)
        S.id[q] = *reinterpret_cast<const uint32_t *>(P.primId + q * P.primIdSlice + (long long)py * P.primIdPitch +
                                                      4ll * px);
    if (depthTest || depthBounds)  // D16 holds the float of its integer (readDepth16, PixelRoutine.cpp:466-481)
      S.zb[q] = depth16 ? (float)*reinterpret_cast<const uint16_t *>(P.depth + q * P.depthSlice +
                                                                     (long long)py * P.depthPitch + 2ll * px)
                        : *reinterpret_cast<const float *>(P.depth + q * P.depthSlice +
                                                           (long long)py * P.depthPitch + 4ll * px);
    if (stencilActive) S.sb[q] = (uint8_t)P.stencil[q * P.stencilSlice + (long long)py * P.stencilPitch + px];
    if constexpr (BLEND) {
      if constexpr (FCOL)
        S.cf[q] =
            *reinterpret_cast<const float4 *>(P.color + q * P.colorSlice + (long long)py * P.colorPitch + 16ll * px);
      else
        S.cb[q] = bgra_swap(
            (XF && P.colorBGRA),
            *reinterpret_cast<const uint32_t *>(P.color + q * P.colorSlice + (long long)py * P.colorPitch + 4ll * px));
    }
  }

  // What a stencil value becomes: where its test fails in bits 0-7, where the
  // depth test fails in 8-15 and where both pass in 16-23, write mask applied;
  // bit 31: the test passes.  For each face one entry a value, so that a
  // candidate costs a read of LDS instead of the compare and three ops.
  __shared__ uint32_t stencilTable[SIMPLE ? 1 : 2][SIMPLE ? 1 : 256];
  if constexpr (!SIMPLE)
    if (stencilActive) {
      for (uint32_t i = threadIdx.x; i < 512; i += blockDim.x) {
        const StencilParams &SP = i < 256 ? P.front : P.back;
        const uint32_t v = i & 255u, keep = v & ~SP.writeMask, wm = SP.writeMask;
        stencilTable[i >> 8][v] = (keep | (stencil_apply_op(v, SP.fail) & wm)) |
                                  (keep | (stencil_apply_op(v, SP.depthFail) & wm)) << 8 |
                                  (keep | (stencil_apply_op(v, SP.pass) & wm)) << 16 |
                                  (stencil_compare(SP, v) ? 0x80000000u : 0u);
      }
      __syncthreads();
    }

  // The 256 decoded codes of an sRGB target that is blended, so that a blend
  // reads its three channels instead of evaluating three powers.
  __shared__ float srgbLut[XF && BLEND ? 256 : 1];
  if (XF && BLEND && P.colorSRGB) {
    for (uint32_t i = threadIdx.x; i < 256; i += blockDim.x) srgbLut[i] = srgb_to_linear(unorm8_to_float(i));
    __syncthreads();
  }

  // Hierarchical depth: a primitive whose evaluated depth is bounded below
  // by zlo cannot pass LESS (LESS_OR_EQUAL) anywhere in a block whose
  // largest stored depth is <= zlo (< zlo).  Only when a failing fragment
  // has no side effect (no stencil writes).
  const bool hiz = depthTest && !stencilWrite && (depthCompare == 1 || depthCompare == 3);

  // Wave totals; nTests, nCovers and nShaded (fragments that passed every test,
  // whether or not a later one replaces them unshaded) are statistics
  // (profiling only).
  unsigned long long occl = 0, nShaded = 0;
  uint32_t nTests = 0, nCovers = 0;
  // The queue is a ring of two batches; a batch is shaded when it is full
  // (and the last one at the end), so every lane of it has a fragment.
  int qHead = 0, qCount = 0;  // wave-uniform: first entry (0 or 64), entries
  // Entries holding fragments of this lane's pixel: of the first batch, and of the next.
  uint64_t mine = 0, mineNext = 0;

  // Shades the first batch of the queue and applies it.
  auto flush = [&]() __attribute__((always_inline)) {
    if constexpr (!QUEUE) return;
    // Shade the queued fragments, one per lane...
    if (lane < qCount) {
      const uint32_t t = W.qTri[qHead + lane];
      const uint32_t pix = W.qPix[qHead + lane];
      const int l = (int)(pix & 63u);
      W.qCol[lane] = shade<FCOL, FTEX, XF, FA>(P, rec[t], ox + lane_cx(l), oy + lane_cy(l));
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // ...then blend them into their pixels in queue (API) order, or write them.
    uint64_t m = mine;
    while (m) {
      const int k = __builtin_ctzll(m);
      m &= m - 1;
      const int xMask = MS > 1 ? (int)(W.qPix[qHead + k] >> 8) : 1;
      const uint32_t tri = FCOL ? W.qTri[qHead + k] : 0u;
      if constexpr (BLEND)
        blend_write<MS, FCOL, XF, FAST>(P, S, W.qCol[k], xMask, tri, srgbLut);
      else
        store_color<MS, FCOL, XF>(P, colorMask, px, py, W.qCol[k], xMask, tri);
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    mine = mineNext;
    mineNext = 0;
    qHead ^= 64;
    qCount = qCount > 64 ? qCount - 64 : 0;
  };

  // Queues the fragment of the lanes that `want` it: primitive tri on their
  // pixel's samples xMask.
  auto enqueue = [&](bool want, uint32_t tri, uint32_t xMask) __attribute__((always_inline)) {
    const uint64_t need = lanes_where(want);
    const int pos = qCount + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(need >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((uint32_t)need, 0));
    if (want) {
      W.qTri[(qHead + pos) & (kQueue - 1)] = tri;
      W.qPix[(qHead + pos) & (kQueue - 1)] = (uint32_t)lane | (xMask << 8);
      const uint64_t bit = 1ull << (pos & 63);
      mine |= pos < 64 ? bit : 0ull;
      mineNext |= pos < 64 ? 0ull : bit;
    }
    qCount += __builtin_popcountll(need);
    if (qCount >= 64) flush();
  };

  // Largest stored depth of the block (+inf when any is NaN): a primitive
  // whose depth is bounded below by zl cannot pass where zl >= it (LESS) or
  // zl > it (LESS_OR_EQUAL).  Reduced as integers that order like the floats.
  auto block_zmax = [&]() __attribute__((always_inline)) {
    float v = -__builtin_inff();
    bool nan = false;
    if (inside) {
#pragma unroll
      for (int q = 0; q < MS; q++) {
        v = fmaxf(v, S.zb[q]);
        nan |= S.zb[q] != S.zb[q];
      }
    }
    const int i = __float_as_int(v);
    const int m = wave_max_i32(i ^ ((i >> 31) & 0x7FFFFFFF));
    return __ballot(nan) ? __builtin_inff() : __int_as_float(m ^ ((m >> 31) & 0x7FFFFFFF));
  };
  auto hidden = [&](float zl, float zmax) __attribute__((always_inline)) {
    return depthCompare == 1 ? zl >= zmax : zl > zmax;
  };

  // One batch of candidates, set up one per lane and then read back one at a
  // time by the whole wave (a broadcast, which leaves the vector units the
  // arithmetic): half planes 0 to 2 as (f, pk), x0, y0, zA, zB, zC, zBias;
  // half planes 3 and 4 of the polygons that have them.
  int step[MS];  // the pixel's samples from the block's origin, as half_plane's operand
#pragma unroll
  for (int q = 0; q < MS; q++)
    step[q] = (int)(((uint32_t)(16 * cx + (MS > 1 ? kXf[q] : 0)) & 0xFFFFu) |
                    ((uint32_t)(-16 * cy - (MS > 1 ? kYf[q] : 0)) << 16));

  // Applies a batch of up to 64 candidates in list order.  Most candidates of
  // a deep block lie behind what the ones before them wrote, and the list of
  // a block is seldom more than a batch or two, so the depth bounds zl are
  // tested before the batch and again, all at once, after every kRetest
  // primitives that wrote depth: at 1080p with 50 layers a block meets 86
  // candidates, of which 20 are not hidden by the time their turn comes.
  constexpr int kRetest = 2;
  auto process_chunk = [&](bool act, uint32_t tid) __attribute__((always_inline)) {
    const float zmax0 = hiz ? block_zmax() : __builtin_inff();  // by every lane of the wave
    // ---- triangle-parallel setup: box, depth bound, half planes ----
    int nflags = 0;
    float zl = -__builtin_inff();
    int4 h1, h2, h3, h4;
    if (act) {
      const int4 *rp = reinterpret_cast<const int4 *>(rec + tid);
      const int4 h0 = rp[0];  // nflags, yMin, yMax, xMin
      h1 = rp[1];             // xMax, X0, X1, X2
      h2 = rp[2];             // Y0, Y1, Y2, zlo
      h3 = rp[3];             // x0, y0, zA, zB
      h4 = rp[4];             // zC, zBias, wA, wB
      nflags = h0.x;
      act = h0.y < oy + 8 && h0.z > oy && h0.w < ox + 8 && h1.x > ox;
      if (hiz) {
        // Lower bound of the evaluated plane over this block (sample offsets
        // included), tightened with the primitive's bound over its box.
        const float x0 = __int_as_float(h3.x), y0 = __int_as_float(h3.y), zA = __int_as_float(h3.z);
        const float zB = __int_as_float(h3.w), zC = __int_as_float(h4.x);
        const float zBias = depthBias ? __int_as_float(h4.y) : 0.0f;
        const float xa = (float)ox - 0.5f - x0, xb = (float)(ox + 7) + 0.5f - x0;
        const float ya = (float)oy - 0.5f - y0, yb = (float)(oy + 7) + 0.5f - y0;
        const float m =
            fminf(fminf(zA * xa + zB * ya, zA * xb + zB * ya), fminf(zA * xa + zB * yb, zA * xb + zB * yb)) + zC + zBias;
        const float mag = fabsf(zA) * fmaxf(fabsf(xa), fabsf(xb)) + fabsf(zC) +
                          2.0f * fabsf(zB) * fmaxf(fabsf(ya), fabsf(yb)) + 2.0f * fabsf(zBias);
        zl = fmaxf(__int_as_float(h2.w), m - mag * 0x1p-19f);
        if (!(zl == zl)) zl = -__builtin_inff();
        zl = fminf(zl, range_hi());
        if (depth16) zl = d16_value(fmaxf(zl, 0.0f));  // the bound in stored units (monotone map)
        act = act && !hidden(zl, zmax0);
      }
    }
    if (act) {
      const int n = nflags & 0xFF, d = (nflags >> 8) & 1;
      int f[3] = {0, 0, 0}, pk[3] = {0, 0, 0};
      if (nflags & (kRecHalfPlanes | kRecWide)) {
        // Edge i runs from vertex i to i + 1 (d), or back.
        auto edge = [&](int Xi, int Yi, int Xk, int Yk, int &fo, int &po) {
          half_plane(d ? Xi : Xk, d ? Yi : Yk, d ? Xk : Xi, d ? Yk : Yi, ox, oy, fo, po);
        };
        if (n == 3) {
          edge(h1.y, h2.x, h1.z, h2.y, f[0], pk[0]);
          edge(h1.z, h2.y, h1.w, h2.z, f[1], pk[1]);
          edge(h1.w, h2.z, h1.y, h2.x, f[2], pk[2]);
        } else {
          const int *pp = poly + (size_t)tid * (2 * kMaxPolygon);
          const int4 X = *reinterpret_cast<const int4 *>(pp), Y = *reinterpret_cast<const int4 *>(pp + kMaxPolygon);
          const int X4 = n > 4 ? pp[4] : X.x, Y4 = n > 4 ? pp[kMaxPolygon + 4] : Y.x;
          int4 m = make_int4(0, 0, 1 << 30, 0);  // no fifth half plane: always inside
          edge(X.x, Y.x, X.y, Y.y, f[0], pk[0]);
          edge(X.y, Y.y, X.z, Y.z, f[1], pk[1]);
          edge(X.z, Y.z, X.w, Y.w, f[2], pk[2]);
          edge(X.w, Y.w, X4, Y4, m.x, m.y);
          if (n > 4) edge(X4, Y4, X.x, Y.x, m.z, m.w);
          W.candMore[lane] = m;
        }
      }
      W.cand[0][lane] = make_int4(f[0], pk[0], f[1], pk[1]);
      W.cand[1][lane] = make_int4(f[2], pk[2], h3.x, h3.y);
      W.cand[2][lane] = make_int4(h3.z, h3.w, h4.x, h4.y);
      if (__builtin_expect((nflags & kRecWide) != 0, 0)) {
        const int *X = reinterpret_cast<const int *>(rec + tid) + offsetof(TriRecord, X) / 4;
        if (n != 3) X = poly + (size_t)tid * (2 * kMaxPolygon);
        const int *Y = X + (n == 3 ? 3 : kMaxPolygon);
        bool crossed = false;
#pragma nounroll
        for (int i = 0; i < n; i++) {
          int *h = i < 2 ? &W.cand[0][lane].x + 2 * i : i == 2 ? &W.cand[1][lane].x : &W.candMore[lane].x + 2 * (i - 3);
          const int k = i + 1 < n ? i + 1 : 0;
          const int ex = abs(X[k] - X[i]), ey = abs(Y[k] - Y[i]), reach = (ex + ey) * 128;  // below 2^29
          if (h[0] < -reach) act = false;
          else if (h[0] > reach) h[1] = 0;
          else crossed |= max(ex, ey) > 32767;
        }
        if (crossed) nflags &= ~kRecWide;
      }
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    uint64_t todo = __ballot(act);
    const uint64_t spanLanes = __ballot(!(nflags & (kRecHalfPlanes | kRecWide)));
    const uint64_t moreLanes = __ballot((nflags & 0xFF) > 3);
    const uint64_t frontLanes = SIMPLE ? 0ull : __ballot((nflags >> 9) & 1);
    int wrote = 0;

    // ---- pixel-parallel coverage and tests, in list order ----
    while (todo) {
      const int j = __builtin_ctzll(todo);
      todo &= todo - 1;
      const int4 c0 = W.cand[0][j], c1 = W.cand[1][j], c2 = W.cand[2][j];
      bool cov[MS];
      if (!((spanLanes >> j) & 1)) {
        int in[MS];
#pragma unroll
        for (int q = 0; q < MS; q++)
          in[q] = min(min(dot2_i16(c0.y, step[q], c0.x), dot2_i16(c0.w, step[q], c0.z)), dot2_i16(c1.y, step[q], c1.x));
        if ((moreLanes >> j) & 1) {
          const int4 m = W.candMore[j];
#pragma unroll
          for (int q = 0; q < MS; q++)
            in[q] = min(min(in[q], dot2_i16(m.y, step[q], m.x)), dot2_i16(m.w, step[q], m.z));
        }
#pragma unroll
        for (int q = 0; q < MS; q++) cov[q] = in[q] >= 0;
      } else {
        const uint32_t tj = __builtin_amdgcn_readlane(tid, j);
        const TriRecord &R = rec[tj];
        const int *pp = poly + (size_t)tj * (2 * kMaxPolygon);
        const int n = R.nflags & 0xFF, d = (R.nflags >> 8) & 1;
        auto vtx = [&](int i, int &Xo, int &Yo) {
          Xo = n == 3 ? R.X[i] : pp[i];
          Yo = n == 3 ? R.Y[i] : pp[kMaxPolygon + i];
        };
#pragma unroll
        for (int q = 0; q < MS; q++)
          cov[q] = span_covers(vtx, n, d, 16 * px + (MS > 1 ? kXf[q] : 0), 16 * py + (MS > 1 ? kYf[q] : 0));
      }
#pragma unroll
      for (int q = 0; q < MS; q++) cov[q] = cov[q] & inside & (((msMask >> q) & 1) != 0);
      nTests++;
      bool anyCov = false;
#pragma unroll
      for (int q = 0; q < MS; q++) anyCov |= cov[q];
      if (!lanes_where(anyCov)) continue;
      nCovers++;

      bool pass[MS];  // samples that pass every test
      if constexpr (SIMPLE) {
        const float xf = (float)px - __int_as_float(c1.z);  // xFragment (PixelRoutine.cpp:125)
        const float yf = (float)py - __int_as_float(c1.w);  // yFragment (QuadRasterizer.cpp:126)
        const float a = __int_as_float(c2.x), b = __int_as_float(c2.y), c = __int_as_float(c2.z);
        float zq[MS];
#pragma unroll
        for (int q = 0; q < MS; q++) {
          const float yy = (MS > 1) ? yf + kSampleY[q] : yf;
          const float xx = (MS > 1) ? xf - kSampleX[q] : xf;
          const float Dz = c + yy * b;
          // clampDepth; the common state's range is of ordinary floats, for
          // which the hardware's max and min equal the ordered selects.
          zq[q] = fminf(fmaxf(xx * a + Dz, range_lo()), range_hi());
        }
        // LESS on its own: one compare.
        if (depthCompare == 1) {
#pragma unroll
          for (int q = 0; q < MS; q++) pass[q] = cov[q] & !(S.zb[q] <= zq[q]);
        } else {
#pragma unroll
          for (int q = 0; q < MS; q++) pass[q] = cov[q] & zp(S.zb[q], zq[q]);
        }
#pragma unroll
        for (int q = 0; q < MS; q++) {
          S.zb[q] = pass[q] ? zq[q] : S.zb[q];
          occl += (unsigned)__builtin_popcountll(lanes_where(pass[q]));
        }
      } else {
        bool sPass[MS], zPass[MS];
        uint32_t st[MS];  // stencil table entries; all ones: no stencil test, which passes
#pragma unroll
        for (int q = 0; q < MS; q++) st[q] = ~0u;
        if (stencilActive) {
          const uint32_t *table = stencilTable[(frontLanes >> j) & 1 ? 0 : 1];
#pragma unroll
          for (int q = 0; q < MS; q++) st[q] = table[S.sb[q]];
        }
#pragma unroll
        for (int q = 0; q < MS; q++) sPass[q] = cov[q] & ((int)st[q] < 0);
        if (alphaToCoverage) {
          // The reference shades before the depth test and keeps sample q
          // only where !(alpha < a2c[q]) (alphaTest / alphaToCoverage,
          // PixelProgram.cpp:243-259, PixelRoutine.cpp:317-337, 643-657); the
          // alpha is clamped when the colour attachment is UNORM.  The
          // fragment is shaded again, identically, if it reaches the queue.
          float alpha = 0.0f;
          const uint32_t tj = __builtin_amdgcn_readlane(tid, j);  // read where every lane is active: lane j need not be covered
          if (anyCov) alpha = shade<FCOL, FTEX, XF, FA>(P, rec[tj], px, py, P.color != nullptr).w;
#pragma unroll
          for (int q = 0; q < MS; q++) {
            cov[q] = cov[q] & !(alpha < P.a2c[q]);
            sPass[q] = sPass[q] & cov[q];
          }
        }
        float zq[MS];
#pragma unroll
        for (int q = 0; q < MS; q++) zPass[q] = cov[q];
        if (depthTest) {
          const float xf = (float)px - __int_as_float(c1.z);  // xFragment (PixelRoutine.cpp:125)
          const float yf = (float)py - __int_as_float(c1.w);  // yFragment (QuadRasterizer.cpp:126)
          const float a = __int_as_float(c2.x), b = __int_as_float(c2.y), c = __int_as_float(c2.z);
          const float zbias = depthBias ? __int_as_float(c2.w) : 0.0f;
#pragma unroll
          for (int q = 0; q < MS; q++) {
            const float yy = (MS > 1) ? yf + kSampleY[q] : yf;
            const float xx = (MS > 1) ? xf - kSampleX[q] : xf;
            const float Dz = c + yy * b;
            float z = xx * a + Dz;
            if (depthBias) z = z + zbias;  // PixelRoutine.cpp:141-144, before the clamp
            z = rr_min(rr_max(z, range_lo()), range_hi());  // clampDepth
            if (depth16) z = d16_value(z);
            zq[q] = z;
            zPass[q] = sPass[q] & zp(S.zb[q], z);
          }
        }
        if (depthBounds) {
          // depthBoundsTest (PixelRoutine.cpp:576-641) on the stored depth, D16
          // as its code / 0xFFFF. With the depth test off the coverage loses
          // the sample while zPass keeps it, so the occlusion count does too.
#pragma unroll
          for (int q = 0; q < MS; q++) {
            const float zs = depth16 ? S.zb[q] * (1.0f / 65535.0f) : S.zb[q];
            const bool in = (P.depthBoundsMin <= zs) & (zs <= P.depthBoundsMax);
            if (depthTest) zPass[q] = zPass[q] & in;
            else cov[q] = cov[q] & in;
          }
        }
        if (stencilWrite) {
#pragma unroll
          for (int q = 0; q < MS; q++) {
            const uint32_t at = !sPass[q] ? 0u : depthTest & !zPass[q] ? 8u : 16u;
            S.sb[q] = cov[q] ? st[q] >> at & 255u : S.sb[q];
          }
        }
#pragma unroll
        for (int q = 0; q < MS; q++) {
          if (depthWrite) S.zb[q] = zPass[q] ? zq[q] : S.zb[q];
          occl += (unsigned)__builtin_popcountll(lanes_where(zPass[q] & sPass[q]));
          pass[q] = (depthTest ? zPass[q] : cov[q]) & sPass[q];
        }
      }

      uint32_t xMask = 0;
#pragma unroll
      for (int q = 0; q < MS; q++) xMask |= pass[q] ? 1u << q : 0u;
      bool any = false;
#pragma unroll
      for (int q = 0; q < MS; q++) any |= pass[q];
      const uint64_t need = lanes_where(any);
      if (!need) continue;
      if (colorMask) {
        const uint32_t tj = __builtin_amdgcn_readlane(tid, j);
        // Shading is deferred so that it runs with every lane busy: blended
        // fragments queue, others leave their primitive's slot.
        if constexpr (BLEND) {
          enqueue(any, tj, xMask);
        } else {
#pragma unroll
          for (int q = 0; q < MS; q++) S.last[q] = pass[q] ? tj + 1u : S.last[q];
        }
        nShaded += (unsigned)__builtin_popcountll(need);
      }
      // What the block shows now may hide the rest of the batch.
      if (hiz && depthWrite && ++wrote >= kRetest && todo) {
        wrote = 0;
        const float zmax = block_zmax();
        todo &= __ballot(!hidden(zl, zmax));
      }
    }
  };

  // The entries of the tile's list that may reach this wave's block (a binned
  // pair carries the blocks its primitive's edges may reach in bits 28-31)
  // wait, in list order, in a per-wave ring, and are set up in full batches
  // of 64: about a quarter of the entries reach a given block, so testing
  // each chunk of the list on its own would leave most lanes idle.  Four
  // chunks are loaded at a time (1080p frame 516 us, 528 with two; the general
  // kernels and the unblended 4x ones take two, for the LDS of their fifth
  // wave per SIMD).
  constexpr int kChunks = Lds::kChunks;
  constexpr uint32_t kRing = Lds::kRing;
  uint32_t ringHead = 0, ringCount = 0;  // wave-uniform
  for (uint32_t base = start;;) {
    while (ringCount < 64 && base < end) {
      uint32_t v[kChunks];
#pragma unroll
      for (int u = 0; u < kChunks; u++) {
        const uint32_t e = base + 64u * u + (uint32_t)lane;
        v[u] = binTri ? 0u : e | 0xF0000000u;
        if (binTri && e < end) v[u] = binTri[e];
      }
#pragma unroll
      for (int u = 0; u < kChunks; u++) {
        const uint32_t e = base + 64u * u + (uint32_t)lane;
        const bool want = e < end && ((v[u] >> (28 + wave)) & 1u);
        const uint64_t tb = __ballot(want);
        if (want)
          W.ring[(ringHead + ringCount +
                  __builtin_amdgcn_mbcnt_hi((uint32_t)(tb >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)tb, 0))) &
                     (kRing - 1)] = v[u] & kSlotMask;
        ringCount += (uint32_t)__builtin_popcountll(tb);
      }
      base = end - base > 64u * kChunks ? base + 64u * kChunks : end;
    }
    if (!ringCount) break;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const uint32_t nb = ringCount < 64 ? ringCount : 64;
    const bool act = (uint32_t)lane < nb;
    const uint32_t t2 = act ? W.ring[(ringHead + lane) & (kRing - 1)] : 0u;
    ringHead = (ringHead + nb) & (kRing - 1);
    ringCount -= nb;
    process_chunk(act, t2);
  }
  if constexpr (!BLEND && MS > 1) {
    // One fragment per pixel and distinct last writer of its samples.
#pragma unroll
    for (int q = 0; q < MS; q++) {
      bool first = S.last[q] != 0;
      uint32_t xMask = 0;
#pragma unroll
      for (int k = 0; k < MS; k++) {
        if (k < q) first = first && S.last[k] != S.last[q];
        else xMask |= S.last[k] == S.last[q] ? 1u << k : 0u;
      }
      enqueue(first, S.last[q] - 1u, xMask);
    }
  }
  if (qCount) flush();
  if constexpr (!BLEND && MS == 1)
    if (S.last[0]) {
      const uint32_t t = S.last[0] - 1u;
      store_color<MS, FCOL, XF>(P, colorMask, px, py, shade<FCOL, FTEX, XF, FA>(P, rec[t], px, py), 1, t);
    }

  // Write the block back.
  if (inside) {
#pragma unroll
    for (int q = 0; q < MS; q++) {
      if (P.depthWrite) {
        if (depth16)
          *reinterpret_cast<uint16_t *>(P.depth + q * P.depthSlice + (long long)py * P.depthPitch + 2ll * px) =
              (uint16_t)S.zb[q];
        else
          *reinterpret_cast<float *>(P.depth + q * P.depthSlice + (long long)py * P.depthPitch + 4ll * px) = S.zb[q];
      }
      if (P.stencilWrite) P.stencil[q * P.stencilSlice + (long long)py * P.stencilPitch + px] = (char)S.sb[q];
      if constexpr (BLEND && FCOL) {
        if (P.primId)
          *reinterpret_cast<uint32_t *>(P.primId + q * P.primIdSlice + (long long)py * P.primIdPitch + 4ll * px) =
              S.id[q];
        *reinterpret_cast<float4 *>(P.color + q * P.colorSlice + (long long)py * P.colorPitch + 16ll * px) = S.cf[q];
      } else if constexpr (BLEND) {
        *reinterpret_cast<uint32_t *>(P.color + q * P.colorSlice + (long long)py * P.colorPitch + 4ll * px) =
            bgra_swap((XF && P.colorBGRA), S.cb[q]);
      }
    }
  }

  // Counters: summed over the workgroup, so that one atomic per counter and
  // workgroup reaches the (single) global address.
  __shared__ unsigned long long red[4][4];
  if (P.occlusion || P.stats) {
    if (lane == 0) {
      red[wave][0] = occl;
      red[wave][1] = nTests;
      red[wave][2] = nCovers;
      red[wave][3] = nShaded;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
      const int k = threadIdx.x;
      const int nw = (int)(blockDim.x >> 6);
      unsigned long long t = red[0][k];
      for (int w = 1; w < nw; w++) t += red[w][k];
      if (k == 0) {
        if (P.occlusion && t) atomicAdd(P.occlusion, t);
      } else if (P.stats) {
        atomicAdd(P.stats + (k - 1), t);
      }
    }
  }
}

// Occupancy, in waves per SIMD.  A wave alternates between chains of scalar,
// LDS and vector work, so another wave pays even where the compiler makes room
// for it by spilling: up to 52 bytes of scratch a lane in the unblended and up
// to 60 in the blended kernels of the common states, up to 100 and 144 in the
// general ones.  At 1280x720 with 30,000 triangles, us a draw here and with one
// wave less:
//   one sample, unblended: common states 167 / 170; blended, general: sRGB with
//   stencil 392 / 413, additive 866 / 971; four samples, unblended: common
//   256 / 269, general (BGRA) 344 / 370, sRGB 624 / 682; blended: common 548 /
//   660, sRGB 848 / 930, float colours, whose 16 registers of colour leave them a
//   wave less, 362 / 425.
// On targets of a few hundred blocks, which do not fill the waves, the two are
// within 4 % but for the blended common kernels at 4x (282 / 318).  One wave
// more: unblended general (BGRA) 195 -> 205 at 6; the blended common kernels lost
// 7 % at 5 (1080p frame).
constexpr int raster_waves(int ms, bool floatColor, int level, bool blend) {
  if (ms == 1) return level == 0 ? 5 : blend ? 4 : 6;
  return blend ? (floatColor ? 3 : 4) : level == 0 ? 4 : 5;
}

// A batch of draws: persistent workgroups take global tiles [tileLo, tileHi)
// from an atomic counter (or, with counter == NULL, workgroup b renders tile
// tileLo + b once); tile t belongs to the draw d in [drawLo, drawHi) with
// tileBase[d] <= t < tileBase[d + 1].
//
// binTri == NULL selects the unbinned pass: every tile walks the record
// slots of its draw from *split on (the primitives the binned pass left out
// because their pairs exceeded the planned capacity) in slot order, testing
// each against its blocks as it would a binned list.  It does nothing when
// *split >= segT (everything was binned).  With binTri and `tail`, each tile
// walks its binned list and then those slots, so that one launch does both
// passes (the tiles of one launch never share pixels, so only the order
// within a tile matters).
template <int MS, bool FCOL, bool FTEX, bool XF, int LEVEL, bool BLEND>
__global__ __launch_bounds__(256, raster_waves(MS, FCOL, LEVEL, BLEND)) void raster_batch_kernel(
                                                           const DrawParams *__restrict__ params,
                                                           const uint32_t *__restrict__ tileBase, int drawLo,
                                                           int drawHi, uint32_t tileLo, uint32_t tileHi,
                                                           uint32_t *__restrict__ counter,
                                                           const TriRecord *__restrict__ rec,
                                                           const int *__restrict__ poly,
                                                           const uint32_t *__restrict__ binTri,
                                                           const uint32_t *__restrict__ tileStart,
                                                           const uint32_t *__restrict__ tileEnd,
                                                           const uint32_t *__restrict__ split, uint32_t segT,
                                                           int tail) {
  __shared__ uint32_t sTile;
  const uint32_t from = (binTri && !tail) ? segT : *split;
  if (!binTri && from >= segT) return;
  // Passes per tile: 0 = the binned list, 1 = the slots from *split on.
  const int pass0 = binTri ? 0 : 1, pass1 = from < segT ? 2 : 1;
  for (uint32_t iter = 0;; iter++) {
    uint32_t t;
    if (counter) {
      if (threadIdx.x == 0) sTile = tileLo + atomicAdd(counter, 1u);
      __syncthreads();
      t = __builtin_amdgcn_readfirstlane(sTile);
      __syncthreads();
    } else {
      if (iter) break;
      // Workgroups go round the 8 XCDs in turn: with four samples, whose planes
      // outgrow the caches, four neighbouring tiles go to one XCD, so that the
      // cache lines and records they share meet in one L2 (64-view step 14.84
      // -> 14.70 ms, 4x frame 576 -> 570 us; with one sample the frame of 50
      // layers loses 0.5 % to its uneven tiles).
      const uint32_t grp = blockIdx.x & ~31u, r = blockIdx.x & 31u;
      t = tileLo + (MS > 1 && grp + 32u <= gridDim.x ? grp + (r & 7u) * 4u + (r >> 3) : blockIdx.x);
    }
    if (t >= tileHi) break;
    int lo = drawLo, hi = drawHi;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (tileBase[mid] <= t) lo = mid;
      else hi = mid;
    }
    lo = __builtin_amdgcn_readfirstlane(lo);
#pragma nounroll
    for (int pass = pass0; pass < pass1; pass++) {
      // The counters of the pass before are summed up (raster_tile's red)
      // before a wave whose block has nothing left writes this pass's.
      if (pass > pass0) __syncthreads();
      uint32_t s, e;
      if (pass == 0) {
        s = tileStart[t];
        e = tileEnd[t];
      } else {
        const uint32_t b = (uint32_t)params[lo].triBase;
        s = from > b ? from : b;
        e = b + (uint32_t)params[lo].triCount;
      }
      if (s < e)
        raster_tile<MS, FCOL, FTEX, XF, LEVEL, BLEND>(params[lo], (int)(t - tileBase[lo]), s, e, rec, poly,
                                               pass == 0 ? binTri : nullptr);
    }
  }
}

template <int MS, bool FCOL, bool FTEX, bool XF, int LEVEL, bool BLEND>
void launch_raster_batch(dim3 grid, dim3 block, hipStream_t s, const RasterArgs &a) {
  // The kernels without a queue gain nothing from more small workgroups a CU,
  // and long lists lose to them in the caches (16x8 tiles, 30,000 untextured
  // triangles at 1280x720: 1494 us, 1619 with twice the workgroups).
  using Lds = WaveLds<MS, LEVEL, BLEND>;
  const uint32_t lds = (Lds::kQueued ? block.x / 64 : 4) * (uint32_t)sizeof(Lds);
  hipLaunchKernelGGL((raster_batch_kernel<MS, FCOL, FTEX, XF, LEVEL, BLEND>), grid, block, lds, s, a.params, a.tileBase,
                     a.lo, a.hi, a.tLo, a.tHi, a.counter, a.rec, a.poly, a.bin, a.ts, a.te, a.split, a.segT, a.tail);
}

// The raster kernel of variant v.
template <bool XF, int LEVEL, bool BLEND>
void launch_raster_variant(int v, dim3 grid, dim3 block, hipStream_t s, const RasterArgs &a) {
  switch (v & (kVarSamples | kVarFloatColor | kVarFloatTex)) {
    case 0: launch_raster_batch<1, false, false, XF, LEVEL, BLEND>(grid, block, s, a); break;
    case kVarFloatTex: launch_raster_batch<1, false, true, XF, LEVEL, BLEND>(grid, block, s, a); break;
    case kVarFloatColor: launch_raster_batch<1, true, false, XF, LEVEL, BLEND>(grid, block, s, a); break;
    case kVarFloatColor | kVarFloatTex: launch_raster_batch<1, true, true, XF, LEVEL, BLEND>(grid, block, s, a); break;
    case kVarSamples: launch_raster_batch<4, false, false, XF, LEVEL, BLEND>(grid, block, s, a); break;
    case kVarSamples | kVarFloatTex: launch_raster_batch<4, false, true, XF, LEVEL, BLEND>(grid, block, s, a); break;
    case kVarSamples | kVarFloatColor: launch_raster_batch<4, true, false, XF, LEVEL, BLEND>(grid, block, s, a); break;
    default: launch_raster_batch<4, true, true, XF, LEVEL, BLEND>(grid, block, s, a); break;
  }
}

// The kernels of the common output states (levels 1 to 3), and the rest.
template <bool BLEND>
void launch_raster_common(int v, dim3 grid, dim3 block, hipStream_t s, const RasterArgs &a) {
  switch ((v & kVarLevel) / kVarLevel1) {
    case 3: launch_raster_variant<false, 3, BLEND>(v, grid, block, s, a); break;
    case 2: launch_raster_variant<false, 2, BLEND>(v, grid, block, s, a); break;
    default: launch_raster_variant<false, 1, BLEND>(v, grid, block, s, a); break;
  }
}

template <bool BLEND>
void launch_raster_general(int v, dim3 grid, dim3 block, hipStream_t s, const RasterArgs &a) {
  if (v & kVarExtended) launch_raster_variant<true, 0, BLEND>(v, grid, block, s, a);
  else launch_raster_variant<false, 0, BLEND>(v, grid, block, s, a);
}

}  // namespace swr
