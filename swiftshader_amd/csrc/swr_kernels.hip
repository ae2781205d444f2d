// swr_kernels.hip -- HIP kernels of the fixed-function draw path (gfx950).
//
// Kernels of a draw (the front end between setup and raster, binning and
// the sort, is in swr_batch.hip, the tile rasteriser in swr_raster.hpp):
//   setup_kernel     one thread per triangle: vertex tail (clip flags,
//                    28.4 projection), trivial reject, clipping, culling,
//                    plane equations, pixel/tile bounding box (setup_one,
//                    shared with the batch front end).
//   clear_rect_kernel, resolve_*_kernel  clears and the 4x -> 1x resolve
//                    (compressed texture decoding is in swr_decode.hip).
//
// Reference semantics: src/Pipeline/VertexRoutine.cpp:116-154,601-611,
// src/Device/Clipper.cpp, src/Pipeline/SetupRoutine.cpp,
// src/Device/Blitter.cpp:1524-1545,2076-2200.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "swr_device.hpp"
#include "swr_params.hpp"
#include "swr_srgb.hpp"

namespace swr {

enum : int { CLIP_RIGHT = 1, CLIP_TOP = 2, CLIP_FAR = 4, CLIP_LEFT = 8, CLIP_BOTTOM = 16, CLIP_NEAR = 32,
             CLIP_FRUSTUM = 63, CLIP_SIDES = 27, CLIP_FINITE = 128 };

// ---------------------------------------------------------------------------
// Setup
// ---------------------------------------------------------------------------
struct ClipVtx { float v[4]; };

__device__ __forceinline__ float clip_dist(const ClipVtx &p, int plane) {
  switch (plane) {
    case 0: return p.v[2];
    case 1: return p.v[3] - p.v[2];
    case 2: return p.v[3] + p.v[0];
    case 3: return p.v[3] - p.v[0];
    case 4: return p.v[3] - p.v[1];
    default: return p.v[3] + p.v[1];
  }
}

__device__ __forceinline__ ClipVtx clip_edge(const ClipVtx &Vi, const ClipVtx &Vj, float di, float dj) {
  float D = rr_rcp(dj - di);
  ClipVtx o;
#pragma unroll
  for (int k = 0; k < 4; k++) o.v[k] = (dj * Vi.v[k] - di * Vj.v[k]) * D;
  return o;
}

// Sutherland-Hodgman against near, far, left, right, top, bottom in that
// order, stopping below 3 vertices (Clipper.cpp:271-299).  Returns the
// number of clip stages applied (the reference's Polygon::i).  tmp: the
// caller's second vertex buffer.
__device__ int clip_polygon(ClipVtx (&poly)[kMaxPolygon], int &n, int flagsOr, ClipVtx (&tmp)[kMaxPolygon]) {
  const int bits[6] = {CLIP_NEAR, CLIP_FAR, CLIP_LEFT, CLIP_RIGHT, CLIP_TOP, CLIP_BOTTOM};
  int stages = 0;
  for (int k = 0; k < 6; k++) {
    if (k > 0 && n < 3) break;
    if (!(flagsOr & bits[k])) continue;
    int t = 0;
    for (int i = 0; i < n; i++) {
      int j = (i == n - 1) ? 0 : i + 1;
      float di = clip_dist(poly[i], k), dj = clip_dist(poly[j], k);
      if (di >= 0) {
        if (t < kMaxPolygon) tmp[t] = poly[i];
        t++;
        if (dj < 0) {
          if (t < kMaxPolygon) tmp[t] = clip_edge(poly[i], poly[j], di, dj);
          t++;
        }
      } else if (dj > 0) {
        if (t < kMaxPolygon) tmp[t] = clip_edge(poly[j], poly[i], dj, di);
        t++;
      }
    }
    n = t < kMaxPolygon ? t : kMaxPolygon;
    for (int i = 0; i < n; i++) poly[i] = tmp[i];
    stages++;
  }
  return stages;
}

__device__ __forceinline__ int wadd(int a, int b) { return (int)((unsigned)a + (unsigned)b); }
__device__ __forceinline__ int wsub(int a, int b) { return (int)((unsigned)a - (unsigned)b); }

// Index p of the draw's index buffer, of its VkIndexType.
__device__ __forceinline__ uint32_t load_index(const DrawParams &P, uint32_t p) {
  if (P.idxBytes == 2) return reinterpret_cast<const uint16_t *>(P.idx)[p];
  if (P.idxBytes == 1) return reinterpret_cast<const uint8_t *>(P.idx)[p];
  return reinterpret_cast<const uint32_t *>(P.idx)[p];
}

// Vertex indices of primitive t in the reference's batch order
// (setBatchIndices, Renderer.cpp:50-145); out-of-range indices read the
// last vertex instead of faulting.
__device__ __forceinline__ void tri_vertices(const DrawParams &P, uint32_t t, uint32_t vi[3]) {
  const uint32_t f = P.provokeLast ? 0u : 1u;  // 1: first-vertex mode
  uint32_t p0, p1, p2;
  if (P.topology == 5) {
    p0 = p1 = p2 = t;  // a point's every setup vertex is its one
  } else if (P.topology >= 3) {
    // A line's vertices, exchanged in last-vertex mode; the setup's third
    // vertex is the second (SetupRoutine.cpp:52-54).
    const uint32_t b = P.topology == 3 ? 2u * t : t;
    p0 = b + (f ? 0u : 1u);
    p1 = b + f;
    p2 = p1;
  } else if (P.topology == 1) {
    p0 = t + (f ? 0u : 2u);
    p1 = t + (t & 1u) + f;
    p2 = t + (~t & 1u) + f;
  } else if (P.topology == 2) {
    const uint32_t a = t + 1u, b = t + 2u;
    p0 = f ? a : b;
    p1 = f ? b : 0u;
    p2 = f ? 0u : a;
  } else {
    p0 = 3u * t + (f ? 0u : 2u);
    p1 = 3u * t + (f ? 1u : 0u);
    p2 = 3u * t + (f ? 2u : 1u);
  }
  vi[0] = P.idx ? load_index(P, p0) : p0;
  vi[1] = P.idx ? load_index(P, p1) : p1;
  vi[2] = P.idx ? load_index(P, p2) : p2;
#pragma unroll
  for (int k = 0; k < 3; k++) vi[k] = vi[k] < (uint32_t)P.vertexCount ? vi[k] : (uint32_t)P.vertexCount - 1u;
}

// DrawCall::setupLine (Renderer.cpp:920-1163): the rectangle of width
// P.lineWidth centred on the segment P0-P1, or, in the Bresenham mode, the
// parallelogram joining P0's and P1's diamonds of half-width lineWidth / 2
// along the major axis, in clip space.  Returns false for a rejected line.
template <int N>
__device__ __forceinline__ bool line_polygon(const DrawParams &P, const float (&P0)[4], const float (&P1)[4],
                                             ClipVtx (&cp)[N]) {
  if (P0[3] <= 0.0f && P1[3] <= 0.0f) return false;
  const float W = P.WxF * (1.0f / 16.0f);
  const float H = P.HxF * (1.0f / 16.0f);
  float dx = W * (P1[0] / P1[3] - P0[0] / P0[3]);
  float dy = H * (P1[1] / P1[3] - P0[1] / P0[3]);
  if (dx == 0.0f && dy == 0.0f) return false;
  if (P.bresenham) {
    const float dx0 = P.lineWidth * 0.5f * P0[3] / W, dy0 = P.lineWidth * 0.5f * P0[3] / H;
    const float dx1 = P.lineWidth * 0.5f * P1[3] / W, dy1 = P.lineWidth * 0.5f * P1[3] / H;
    // Corners kept per major direction: right and down run P0, P1, P1, P0
    // along one diamond axis; up and left run P0, P0, P1, P1.
    const bool alongFirst = dx > -dy;
    const bool xMajor = dx > dy;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const bool first = alongFirst ? (k == 0 || k == 3) : (k < 2);
      for (int j = 0; j < 4; j++) cp[k].v[j] = first ? P0[j] : P1[j];
    }
    if (alongFirst && xMajor) {  // right: up and down corners
      cp[0].v[1] += +dy0; cp[1].v[1] += +dy1; cp[2].v[1] += -dy1; cp[3].v[1] += -dy0;
    } else if (alongFirst) {     // down: left and right corners
      cp[0].v[0] += -dx0; cp[1].v[0] += -dx1; cp[2].v[0] += +dx1; cp[3].v[0] += +dx0;
    } else if (xMajor) {         // up: left and right corners
      cp[0].v[0] += -dx0; cp[1].v[0] += +dx0; cp[2].v[0] += +dx1; cp[3].v[0] += -dx1;
    } else {                     // left: up and down corners
      cp[0].v[1] += +dy0; cp[1].v[1] += -dy0; cp[2].v[1] += -dy1; cp[3].v[1] += +dy1;
    }
  } else {
    const float scale = P.lineWidth * 0.5f / sqrtf(dx * dx + dy * dy);
    dx = dx * scale;
    dy = dy * scale;
    const float dx0h = dx * P0[3] / H, dy0w = dy * P0[3] / W;
    const float dx1h = dx * P1[3] / H, dy1w = dy * P1[3] / W;
#pragma unroll
    for (int k = 0; k < 4; k++)
      for (int j = 0; j < 4; j++) cp[k].v[j] = (k == 0 || k == 3) ? P0[j] : P1[j];
    cp[0].v[0] += -dy0w; cp[0].v[1] += +dx0h;
    cp[1].v[0] += -dy1w; cp[1].v[1] += +dx1h;
    cp[2].v[0] += +dy1w; cp[2].v[1] += -dx1h;
    cp[3].v[0] += +dy0w; cp[3].v[1] += -dx0h;
  }
  return true;
}

// DrawCall::setupPoint (Renderer.cpp:1166-1210): the square of side
// PointSize (clamped to [1, 1023] by two compares, so a NaN passes) centred
// on the vertex, offsets pSize * w * halfPixel, halfPixel = 0.5 / (viewport
// extent / 2).
template <int N>
__device__ __forceinline__ void point_polygon(const DrawParams &P, const float (&V)[4], float size,
                                              ClipVtx (&cp)[N]) {
  float pSize = size;
  if (pSize < 1.0f) pSize = 1.0f;
  if (pSize > 1023.0f) pSize = 1023.0f;
  const float halfPixelX = 0.5f / (P.WxF * (1.0f / 16.0f));
  const float halfPixelY = 0.5f / (P.HxF * (1.0f / 16.0f));
  const float X = pSize * V[3] * halfPixelX;
  const float Y = pSize * V[3] * halfPixelY;
#pragma unroll
  for (int k = 0; k < 4; k++)
    for (int j = 0; j < 4; j++) cp[k].v[j] = V[j];
  cp[0].v[0] -= X; cp[0].v[1] += Y;
  cp[1].v[0] += X; cp[1].v[1] += Y;
  cp[2].v[0] += X; cp[2].v[1] -= Y;
  cp[3].v[0] -= X; cp[3].v[1] -= Y;
}

template <typename T>
__device__ __forceinline__ T pick3(T a, T b, T c, int i) { return i == 0 ? a : (i == 1 ? b : c); }

// Vertex arrays of the polygon path (clipped triangles, lines and points),
// indexed at run time.
struct PolyWork {
  ClipVtx cp[kMaxPolygon], tmp[kMaxPolygon];
  int X[kMaxPolygon], Y[kMaxPolygon];
};

__device__ __forceinline__ int edge_mul(int a, int b) { return __mul24(a, b); }
__device__ __forceinline__ long long edge_mul(long long a, long long b) { return a * b; }

// Whether polygon X, Y (n >= 3) is convex on the 28.4 grid, with no repeated
// vertex: every turn goes the same way or straight on, and the edges change
// between downward and upward twice (one revolution).  T: int for extents up
// to 32767 (the products of 16-bit edges, and the sums of two, fit 32 bits),
// long long for longer ones.
template <typename T, int N>
__device__ __forceinline__ bool convex_polygon(const int (&X)[N], const int (&Y)[N], int n) {
  bool left = false, right = false, back = false;
  int changes = 0, dir = 0, firstDir = 0;
  T dx0 = X[0] - X[n - 1], dy0 = Y[0] - Y[n - 1];
  for (int i = 0; i < n; i++) {
    const int k = i + 1 < n ? i + 1 : 0;
    const T dx1 = X[k] - X[i], dy1 = Y[k] - Y[i];
    const T c = edge_mul(dx0, dy1) - edge_mul(dy0, dx1);
    left |= c > 0;
    right |= c < 0;
    // Straight on, and neither edge of zero length.
    back |= c == 0 && edge_mul(dx0, dx1) + edge_mul(dy0, dy1) <= 0;
    const int s = dy1 > 0 ? 1 : (dy1 < 0 ? -1 : 0);
    changes += s != 0 && firstDir != 0 && s != dir ? 1 : 0;
    firstDir = firstDir ? firstDir : s;
    dir = s ? s : dir;
    dx0 = dx1;
    dy0 = dy1;
  }
  if (dir != firstDir) changes++;
  return !(left && right) && !back && changes == 2;
}

// Setup of primitive t of the draw P into R (all but R.draw), and the tiles
// of its box into `tiles`; R's n and box and `tiles` are zero on entry and
// stay so when it is culled.  Polygons of more than three vertices also write
// `poly`; w holds the polygon path's arrays.  Without POLY, the primitives
// that need the polygon path (those that clipping changes) are left alone and
// false is returned (w is not touched), so that a kernel can give that path
// workspace in LDS for a few lanes at a time instead of scratch memory for
// every thread.  Points and lines inside the frustum keep their four corners
// in registers.
template <bool POLY = true>
__device__ __forceinline__ bool setup_one(const DrawParams &P, int t, TriRecord &R, int *__restrict__ poly,
                                          uint32_t &tiles, PolyWork &w) {
  uint32_t vi[3];
  tri_vertices(P, (uint32_t)t, vi);

  float pos[3][4], attr[3][6];
  int flags[3], PX[3], PY[3];
  float pz[3], pw[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    float4 p = reinterpret_cast<const float4 *>(P.pos)[vi[k]];
    pos[k][0] = p.x; pos[k][1] = p.y; pos[k][2] = p.z; pos[k][3] = p.w;
    if (P.col) {
      float4 c = reinterpret_cast<const float4 *>(P.col)[vi[k]];
      attr[k][0] = c.x; attr[k][1] = c.y; attr[k][2] = c.z; attr[k][3] = c.w;
    } else {
      attr[k][0] = attr[k][1] = attr[k][2] = attr[k][3] = 0.0f;
    }
    if (P.uv) {
      float2 u = reinterpret_cast<const float2 *>(P.uv)[vi[k]];
      attr[k][4] = u.x; attr[k][5] = u.y;
    } else {
      attr[k][4] = attr[k][5] = 0.0f;
    }
    // Clip flags (VertexRoutine.cpp:116-154).
    float x = p.x, y = p.y, z = p.z, w = p.w;
    int f = 0;
    if (w < x) f |= CLIP_RIGHT;
    if (w < y) f |= CLIP_TOP;
    if (!(-w <= x)) f |= CLIP_LEFT;
    if (!(-w <= y)) f |= CLIP_BOTTOM;
    if (P.depthClip) {  // near and far only with depth clipping (VertexRoutine.cpp:137-143)
      if (w < z) f |= CLIP_FAR;
      if (!(0.0f <= z)) f |= CLIP_NEAR;
    }
    const float maxPos = __uint_as_float(0x7F7FFFFFu);
    if (__builtin_fabsf(x) <= maxPos && __builtin_fabsf(y) <= maxPos && __builtin_fabsf(z) <= maxPos) f |= CLIP_FINITE;
    flags[k] = f;
    // Projection (VertexRoutine.cpp:601-611).
    float ww = __uint_as_float(__float_as_uint(w) | ((w == 0.0f) ? 0x3F800000u : 0u));
    float rhw = rr_rcp(ww);
    PX[k] = rr_round_int_clamped(P.X0xF + (x * rhw) * P.WxF);
    PY[k] = rr_round_int_clamped(P.Y0xF + (y * rhw) * P.HxF);
    pz[k] = z * rhw;
    pw[k] = rhw;
  }

  ClipVtx (&cp)[kMaxPolygon] = w.cp;
  int n = 3;
  int stages = 0;
  int d = 1;
  int frontFacing = 1;
  const bool quad = P.point || P.line;
  int QX[4] = {0, 0, 0, 0}, QY[4] = {0, 0, 0, 0};  // a point's or line's corners (without POLY)
  if (quad) {
    // setupPoint: the point's square; setupLine: the line's polygon.  Clipped
    // against every frustum plane; no culling, front-facing, d = 1
    // (SetupRoutine.cpp:115-119).
    n = 4;
    if constexpr (POLY) {
      if (P.point) point_polygon(P, pos[0], P.psize ? P.psize[vi[0]] : 1.0f, cp);
      else if (!line_polygon(P, pos[0], pos[1], cp)) return true;
      stages = clip_polygon(cp, n, P.depthClip ? CLIP_FRUSTUM : CLIP_SIDES, w.tmp);
      if (n < 3) return true;
    } else {
      ClipVtx q[4];
      if (P.point) point_polygon(P, pos[0], P.psize ? P.psize[vi[0]] : 1.0f, q);
      else if (!line_polygon(P, pos[0], pos[1], q)) return true;
      // Clipping keeps a polygon whose vertices all lie inside as it is.
      bool inside = true;
#pragma unroll
      for (int i = 0; i < 4; i++) {
#pragma unroll
        for (int k = 0; k < 6; k++) inside = inside && ((k < 2 && !P.depthClip) || clip_dist(q[i], k) >= 0);
        const float cw = q[i].v[3];
        const float rhw = (cw != 0.0f) ? rr_rcp(cw) : 1.0f;
        QX[i] = rr_round_int(P.X0xF + (q[i].v[0] * rhw) * P.WxF);
        QY[i] = rr_round_int(P.Y0xF + (q[i].v[1] * rhw) * P.HxF);
      }
      if (!inside) return false;
    }
  } else {
    // setupSolidTriangles (Renderer.cpp:733-776).
    if ((flags[0] & flags[1] & flags[2]) != CLIP_FINITE) return true;
    int flagsOr = flags[0] | flags[1] | flags[2];
    if (flagsOr != CLIP_FINITE) {
      if (!POLY) return false;
#pragma unroll
      for (int k = 0; k < 3; k++)
        for (int c = 0; c < 4; c++) cp[k].v[c] = pos[k][c];
      stages = clip_polygon(cp, n, flagsOr, w.tmp);
      if (n < 3) return true;
    }
    // Culling and facing (SetupRoutine.cpp:71-120).
    float x0 = (float)PX[0], x1 = (float)PX[1], x2 = (float)PX[2];
    float y0 = (float)PY[0], y1 = (float)PY[1], y2 = (float)PY[2];
    float A = (y0 - y2) * x1 + (y2 - y1) * x0 + (y1 - y0) * x2;
    int w012 = (int)(__float_as_uint(pos[0][3]) ^ __float_as_uint(pos[1][3]) ^ __float_as_uint(pos[2][3]));
    if (w012 < 0) A = -A;
    frontFacing = (P.frontFace == 0) ? (A >= 0.0f) : (A <= 0.0f);
    if ((P.cullMode & 1) && frontFacing) return true;
    if ((P.cullMode & 2) && !frontFacing) return true;
    d = (A > 0.0f) ? 1 : 0;
  }

  // Polygon in 28.4 (reprojected when clipped or a line,
  // SetupRoutine.cpp:122-143).
  // An unclipped triangle, point or line keeps its vertices in registers; only
  // a clipped polygon goes through the n-vertex arrays.
  const bool isPolygon = POLY && (stages != 0 || quad);
  int (&X)[kMaxPolygon] = w.X;
  int (&Y)[kMaxPolygon] = w.Y;
  int yMin, yMax, xLo, xHi;
  if (isPolygon) {
    for (int i = 0; i < n; i++) {
      float w = cp[i].v[3];
      float rhw = (w != 0.0f) ? rr_rcp(w) : 1.0f;
      X[i] = rr_round_int(P.X0xF + (cp[i].v[0] * rhw) * P.WxF);
      Y[i] = rr_round_int(P.Y0xF + (cp[i].v[1] * rhw) * P.HxF);
    }
    yMin = Y[0]; yMax = Y[0]; xLo = X[0]; xHi = X[0];
    for (int i = 1; i < n; i++) {
      yMin = min(yMin, Y[i]); yMax = max(yMax, Y[i]);
      xLo = min(xLo, X[i]); xHi = max(xHi, X[i]);
    }
  } else if (quad) {
    yMin = min(min(QY[0], QY[1]), min(QY[2], QY[3]));
    yMax = max(max(QY[0], QY[1]), max(QY[2], QY[3]));
    xLo = min(min(QX[0], QX[1]), min(QX[2], QX[3]));
    xHi = max(max(QX[0], QX[1]), max(QX[2], QX[3]));
  } else {
    yMin = min(min(PY[0], PY[1]), PY[2]);
    yMax = max(max(PY[0], PY[1]), PY[2]);
    xLo = min(min(PX[0], PX[1]), PX[2]);
    xHi = max(max(PX[0], PX[1]), PX[2]);
  }
  const int yLo = yMin, yHi = yMax;
  if (P.ms > 1) {
    yMin = wadd(yMin, 9) >> 4;   // yMinMultiSampleOffset (Constants.hpp:51)
    yMax = wadd(yMax, 21) >> 4;  // yMaxMultiSampleOffset (Constants.hpp:52)
  } else {
    yMin = wadd(yMin, 15) >> 4;
    yMax = wadd(yMax, 15) >> 4;
  }
  yMin = max(yMin, P.sy0);
  yMax = min(yMax, P.sy1);
  if (yMin >= yMax) return true;
  // Columns that can hold coverage: left >= ceil(min X / 16), right <= ceil(max X / 16).
  const int sxo = (P.ms > 1) ? 6 : 0;
  int xMin = max(wadd(wsub(xLo, sxo), 15) >> 4, P.sx0);
  int xMax = min(wadd(wadd(xHi, sxo), 15) >> 4, P.sx1);
  if (xMin >= xMax) return true;

  // Sort by minimum y, then by maximum w (SetupRoutine.cpp:270-294),
  // triangles only.
  int o0 = 0, o1 = 1, o2 = 2;
  if (!P.line && !P.point) {
    float y0 = pos[0][1], y1 = pos[1][1], y2 = pos[2][1];
    float ym = rr_min(rr_min(y0, y1), y2);
    if (ym == y1) { int tt = o0; o0 = o1; o1 = o2; o2 = tt; }
    if (ym == y2) { int tt = o2; o2 = o1; o1 = o0; o0 = tt; }
  }
  if (!P.line && !P.point) {
    float w0 = pick3(pos[0][3], pos[1][3], pos[2][3], o0), w1 = pick3(pos[0][3], pos[1][3], pos[2][3], o1),
          w2 = pick3(pos[0][3], pos[1][3], pos[2][3], o2);
    float wm = rr_max(rr_max(w0, w1), w2);
    if (wm == w1) { int tt = o0; o0 = o1; o1 = o2; o2 = tt; }
    if (wm == w2) { int tt = o2; o2 = o1; o1 = o0; o0 = tt; }
  }
  // Plane equations (SetupRoutine.cpp:296-548).
  // The rotated vertices are picked by selects, not by indexing the
  // per-vertex arrays with a run-time index (which would place them in
  // scratch memory).
  float w1 = pick3(pos[0][3], pos[1][3], pos[2][3], o1), w2 = pick3(pos[0][3], pos[1][3], pos[2][3], o2);
  float rhw0 = pick3(pw[0], pw[1], pw[2], o0);
  int X0 = pick3(PX[0], PX[1], PX[2], o0), X1 = pick3(PX[0], PX[1], PX[2], o1), X2 = pick3(PX[0], PX[1], PX[2], o2);
  int Y0 = pick3(PY[0], PY[1], PY[2], o0), Y1 = pick3(PY[0], PY[1], PY[2], o1), Y2 = pick3(PY[0], PY[1], PY[2], o2);
  if (P.line) {  // a third point across the line (SetupRoutine.cpp:317-321)
    X2 = wsub(wadd(X1, Y1), Y0);
    Y2 = wsub(wadd(Y1, X0), X1);
  }
  R.x0 = (float)X0 * (1.0f / 16.0f);
  R.y0 = (float)Y0 * (1.0f / 16.0f);
  X1 = wsub(X1, X0); Y1 = wsub(Y1, Y0);
  X2 = wsub(X2, X0); Y2 = wsub(Y2, Y0);
  float x1 = w1 * (1.0f / 16.0f) * (float)X1;
  float y1 = w1 * (1.0f / 16.0f) * (float)Y1;
  float x2 = w2 * (1.0f / 16.0f) * (float)X2;
  float y2 = w2 * (1.0f / 16.0f) * (float)Y2;
  float a = x1 * y2 - x2 * y1;
  float M00 = 0.0f, M01 = 0.0f, M02 = rhw0, M10 = 0.0f, M11 = 0.0f, M20 = 0.0f, M21 = 0.0f;
  if (a != 0.0f) {
    float A = rr_rcp(a);
    float D = A * rhw0;
    M00 = (y1 * w2 - y2 * w1) * D;
    M01 = (x2 * w1 - x1 * w2) * D;
    M10 = y2 * A;
    M11 = -x2 * A;
    M20 = -y1 * A;
    M21 = x1 * A;
  }
  R.wA = (M00 + M10) + M20;
  R.wB = (M01 + M11) + M21;
  R.wC = (M02 + 0.0f) + 0.0f;
  if (P.depthTest) {
    float z0 = pick3(pz[0], pz[1], pz[2], o0), z1 = pick3(pz[0], pz[1], pz[2], o1) - z0,
          z2 = pick3(pz[0], pz[1], pz[2], o2) - z0;
    float fx1 = (float)X1 * (1.0f / 16.0f), fy1 = (float)Y1 * (1.0f / 16.0f);
    float fx2 = (float)X2 * (1.0f / 16.0f), fy2 = (float)Y2 * (1.0f / 16.0f);
    if (!P.point) {
      float D = P.depthRange / (fx1 * fy2 - fx2 * fy1);
      R.zA = (fy2 * z1 - fy1 * z2) * D;
      R.zB = (fx1 * z2 - fx2 * z1) * D;
    } else {  // a point's depth is constant (SetupRoutine.cpp:393-409)
      R.zA = 0.0f;
      R.zB = 0.0f;
    }
    R.zC = z0 * P.depthRange + P.depthNear;
    // Depth bias (SetupRoutine.cpp:417-475), floating-point depth buffer:
    // r = 2^(e - 23) for the largest exponent e among the plane constant and
    // z1, z2 mapped through the depth range -- z1, z2 being the differences
    // from z0 formed above, as in the reference.
    float bias = 0.0f;
    if (P.biasConstant) {
      const float Z1 = z1 * P.depthRange + P.depthNear, Z2 = z2 * P.depthRange + P.depthNear;
      const int e0 = __float_as_int(R.zC) & 0x7F800000, e1 = __float_as_int(Z1) & 0x7F800000;
      const int e2 = __float_as_int(Z2) & 0x7F800000;
      const int e = max(max(e0, e1), e2);
      // D16: minimumResolvableDepthDifference (Renderer.cpp:427-430).
      const float r = P.depth16 ? 1.01f / 65535.0f : __int_as_float(e) * (1.0f / (float)(1 << 23));
      bias = r * P.constantDepthBias;
    }
    if (P.biasSlope) {
      const float aA = R.zA > 0.0f ? R.zA : -R.zA, aB = R.zB > 0.0f ? R.zB : -R.zB;  // Reactor's Abs
      const float m = rr_max(aA, aB);
      bias = bias + m * P.slopeDepthBias;
    }
    if ((P.biasConstant || P.biasSlope) && P.biasClamp)
      bias = P.depthBiasClamp > 0.0f ? rr_min(bias, P.depthBiasClamp) : rr_max(bias, P.depthBiasClamp);
    R.zBias = bias;
  } else {
    R.zA = R.zB = R.zC = 0.0f;
    R.zBias = 0.0f;
  }
#pragma unroll
  for (int k = 0; k < 6; k++) {
    float i0 = pick3(attr[0][k], attr[1][k], attr[2][k], o0), i1 = pick3(attr[0][k], attr[1][k], attr[2][k], o1),
          i2 = pick3(attr[0][k], attr[1][k], attr[2][k], o2);
    R.V[k][0] = (i0 * M00 + i1 * M10) + i2 * M20;
    R.V[k][1] = (i0 * M01 + i1 * M11) + i2 * M21;
    R.V[k][2] = (i0 * M02 + i1 * 0.0f) + i2 * 0.0f;
  }

  // Lower bound of z as the rasteriser evaluates it, x*A + (C + y*B) in
  // float: covered sample points lie in the polygon, so the affine minimum is
  // at one of its vertices; a sample's depth is taken at the point mirrored in
  // x about its pixel's centre, up to 3/4 pixel away; less a margin of 8 ulp
  // of the largest term over the bounding box.  Lets a tile skip primitives
  // that cannot pass its depth test (over the bounding box's corners, as this
  // bound once was, half the triangles of a deep scene reach down to 0).
  float zlo = -__builtin_inff();
  if (P.depthTest && __builtin_isfinite(R.zA) && __builtin_isfinite(R.zB) && __builtin_isfinite(R.zC) &&
      __builtin_isfinite(R.zBias)) {
    const double xa = (double)xMin - 0.5 - (double)R.x0, xb = (double)(xMax - 1) + 0.5 - (double)R.x0;
    const double ya = (double)yMin - 0.5 - (double)R.y0, yb = (double)(yMax - 1) + 0.5 - (double)R.y0;
    const double A = R.zA, B = R.zB, C = R.zC;
    const double Zb = P.depthBias ? (double)R.zBias : 0.0;
    auto at = [&](int vx, int vy) {
      return A * ((double)vx * 0.0625 - (double)R.x0) + B * ((double)vy * 0.0625 - (double)R.y0);
    };
    double m;
    if (isPolygon) {
      m = at(X[0], Y[0]);
      for (int i = 1; i < n; i++) m = fmin(m, at(X[i], Y[i]));
    } else if (quad) {
      m = fmin(fmin(at(QX[0], QY[0]), at(QX[1], QY[1])), fmin(at(QX[2], QY[2]), at(QX[3], QY[3])));
    } else {
      m = fmin(fmin(at(PX[0], PY[0]), at(PX[1], PY[1])), at(PX[2], PY[2]));
    }
    m += C + Zb - (P.ms > 1 ? 0.75 * fabs(A) : 0.0);
    const double mag =
        fabs(A) * fmax(fabs(xa), fabs(xb)) + fabs(C) + 2.0 * fabs(B) * fmax(fabs(ya), fabs(yb)) + 2.0 * fabs(Zb);
    const double lo = m - mag * 0x1p-21 - 1e-30;
    if (__builtin_isfinite(lo)) {
      float f = (float)lo;
      if ((double)f > lo) {  // step one float towards -inf
        const uint32_t u = __float_as_uint(f);
        f = (f > 0.0f) ? __uint_as_float(u - 1) : (f < 0.0f ? __uint_as_float(u + 1) : -1.17549435e-38f);
      }
      zlo = f;
    }
  }
  R.zlo = zlo;
  R.yMin = yMin;
  R.yMax = yMax;
  R.xMin = xMin;
  R.xMax = xMax;
  if (!POLY && quad) {
    int4 *pp = reinterpret_cast<int4 *>(poly);
    pp[0] = make_int4(QX[0], QX[1], QX[2], QX[3]);
    pp[kMaxPolygon / 4] = make_int4(QY[0], QY[1], QY[2], QY[3]);
  } else if (!isPolygon) {
#pragma unroll
    for (int i = 0; i < 3; i++) { R.X[i] = PX[i]; R.Y[i] = PY[i]; }
  } else if (n == 3) {
    for (int i = 0; i < 3; i++) { R.X[i] = X[i]; R.Y[i] = Y[i]; }
  } else {
    for (int i = 0; i < n; i++) { poly[i] = X[i]; poly[kMaxPolygon + i] = Y[i]; }
  }
  // A triangle is convex; a polygon is when its turns agree.
  const int big = 1 << 20, ext = 32767;
  const bool narrow = wsub(xHi, xLo) <= ext && wsub(yHi, yLo) <= ext;
  bool planes = xLo > -big && xHi < big && yLo > -big && yHi < big;
  if (planes && n > 3) {
    if (!POLY) planes = narrow ? convex_polygon<int>(QX, QY, 4) : convex_polygon<long long>(QX, QY, 4);
    else if (n > kMaxHalfPlanes) planes = false;
    else planes = narrow ? convex_polygon<int>(X, Y, n) : convex_polygon<long long>(X, Y, n);
  }
  R.nflags = n | (d << 8) | (frontFacing ? 1 << 9 : 0) | (planes ? (narrow ? kRecHalfPlanes : kRecWide) : 0);
  // Tiles are 8 or 16 pixels a side and xMin, yMin >= 0 (scissor-clamped to
  // a render area at x, y >= 0): shifts divide exactly.
  const int sw = __builtin_ctz((uint32_t)P.tileW), sh = __builtin_ctz((uint32_t)P.tileH);
  int tx0 = xMin >> sw, tx1 = (xMax - 1) >> sw;
  int ty0 = yMin >> sh, ty1 = (yMax - 1) >> sh;
  tiles = (uint32_t)((tx1 - tx0 + 1) * (ty1 - ty0 + 1));
  return true;
}

// Polygon-path workspaces per wave of the setup kernels (640 B each).
constexpr int kPolySlots = 16;
// A record's words as staged in LDS: all but the last, R.draw.  An odd stride,
// so that the lanes' writes of one word fall in different banks.
constexpr int kStageWords = (int)(sizeof(TriRecord) / 4) - 1;
static_assert(64 * kStageWords * 4 <= kPolySlots * sizeof(PolyWork) && kStageWords % 2 == 1, "record staging");

// Setup of primitive t (slot g, draw `draw`) by the calling lane, t < 0 for
// none: every lane first runs the setup without the polygon path; the lanes
// whose primitive needs it (what clipping changes) then run it
// kPolySlots at a time per wave, each with a workspace in `work` (the
// wave's kPolySlots entries in LDS), so that no thread uses scratch memory.
// Called by every lane of the wave, with consecutive slots.
//
// The kernel is bound by its record stores: 160 bytes a lane, 160 bytes
// apart, took some 13 store instructions of 64 cache lines each.  The wave's
// records are therefore staged in LDS (in the polygon path's workspaces, which
// are used afterwards) and leave as whole lines, 64 consecutive 16-byte pieces
// to an instruction; of a culled primitive's record only the first piece.
__device__ __forceinline__ void setup_lanes(const DrawParams &P, int t, size_t g, int draw, TriRecord *__restrict__ rec,
                                            int *__restrict__ poly, uint32_t *__restrict__ tileCount,
                                            PolyWork *work) {
  const int lane = threadIdx.x & 63;
  int *stage = reinterpret_cast<int *>(work);
  bool later = false;
  uint32_t tiles = 0;
  if (t >= 0) {
    TriRecord &R = *reinterpret_cast<TriRecord *>(stage + lane * kStageWords);
    R.nflags = R.yMin = R.yMax = R.xMin = R.xMax = 0;
    later = !setup_one<false>(P, t, R, poly + g * (2 * kMaxPolygon), tiles, work[0]);
    if (!later) tileCount[g] = tiles;
  }
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  {
    const uint64_t has = __ballot(t >= 0 && !later), full = __ballot(tiles != 0);
    int4 *out = reinterpret_cast<int4 *>(rec + (g - (size_t)lane));  // the wave's first record
    constexpr int kParts = (int)(sizeof(TriRecord) / 16);
#pragma unroll
    for (int i = 0; i < kParts; i++) {
      const int q = 64 * i + lane, r = q / kParts, part = q % kParts;
      if (!((part == 0 ? has : full) >> r & 1)) continue;
      const int *w = stage + r * kStageWords + 4 * part;
      out[q] = make_int4(w[0], w[1], w[2], part == kParts - 1 ? draw : w[3]);
    }
  }
  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  for (uint64_t m = __ballot(later); m; m = __ballot(later)) {  // wave-uniform
    // The next round's lanes reuse the workspaces.
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const uint32_t rank = (uint32_t)__builtin_popcountll(m & below);
    const bool mine = later && rank < (uint32_t)kPolySlots;
    if (mine) {
      TriRecord &R = rec[g];
      R.nflags = R.yMin = R.yMax = R.xMin = R.xMax = 0;
      R.draw = draw;
      setup_one<true>(P, t, R, poly + g * (2 * kMaxPolygon), tiles, work[rank]);
      tileCount[g] = tiles;
    }
    later = later && !mine;
  }
}

// One draw: one thread per primitive.
__global__ __launch_bounds__(256) void setup_kernel(DrawParams P, TriRecord *__restrict__ rec,
                                                    int *__restrict__ poly, uint32_t *__restrict__ tileCount) {
  __shared__ PolyWork work[4][kPolySlots];
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  setup_lanes(P, t < P.triCount ? t : -1, (size_t)t, 0, rec, poly, tileCount, work[threadIdx.x >> 6]);
}

__global__ void fill_u32_kernel(uint32_t *p, uint32_t v, uint32_t n) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// ---------------------------------------------------------------------------
// MSAA resolve (Blitter.cpp:2076-2200 for RGBA8, :1524-1545 for float)
// ---------------------------------------------------------------------------
// Fills a rectangle of every sample plane with one BYTES-wide value (the
// packed clear value).  Grid: x over the rectangle's width, y over its
// rows, z over the sample planes.
template <int BYTES>
__global__ void clear_rect_kernel(char *base, int rowPitch, long long slice, int x0, int y0, int w, int h,
                                  uint4 value) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
  if (x >= w || y >= h) return;
  char *p = base + (long long)blockIdx.z * slice + (long long)(y0 + y) * rowPitch + (long long)BYTES * (x0 + x);
  if (BYTES == 16) *reinterpret_cast<uint4 *>(p) = value;
  else if (BYTES == 4) *reinterpret_cast<uint32_t *>(p) = value.x;
  else if (BYTES == 2) *reinterpret_cast<uint16_t *>(p) = (uint16_t)value.x;
  else *reinterpret_cast<uint8_t *>(p) = (uint8_t)value.x;
}

// Up to kClearBatch clears of one element size in one launch (a kernel
// argument, so nothing is uploaded): rect k owns blocks [start[k],
// start[k + 1]), each block kClearPixels consecutive pixels of the rect's
// pixels in (sample, row, column) order, kClearPixels / 256 per thread.
constexpr int kClearBatch = 24;
constexpr int kClearPixels = 1024;
struct ClearRect {
  char *base;
  long long slice;
  int pitch, x0, y0, w, h, samples, bytes;
  uint4 value;
};
struct ClearBatch {
  ClearRect r[kClearBatch];
  uint32_t start[kClearBatch + 1];
  int n;
};

template <int BYTES>
__global__ void clear_batch_kernel(ClearBatch cb) {
  const uint32_t b = blockIdx.x;
  int k = 0;
  while (k + 1 < cb.n && cb.start[k + 1] <= b) k++;
  const ClearRect &r = cb.r[k];
  const uint64_t plane = (uint64_t)r.w * (uint64_t)r.h, total = plane * (uint64_t)r.samples;
  const uint64_t first = (uint64_t)(b - cb.start[k]) * kClearPixels;
#pragma unroll
  for (int j = 0; j < kClearPixels / 256; j++) {
    const uint64_t i = first + (uint64_t)threadIdx.x + 256u * (uint64_t)j;
    if (i >= total) break;
    const uint64_t q = i / plane, rem = i - q * plane;
    const uint32_t y = (uint32_t)(rem / (uint64_t)r.w), x = (uint32_t)(rem - (uint64_t)y * (uint64_t)r.w);
    char *p = r.base + (long long)q * r.slice + (long long)(r.y0 + (int)y) * r.pitch + (long long)BYTES * (r.x0 + (int)x);
    if (BYTES == 16) *reinterpret_cast<uint4 *>(p) = r.value;
    else if (BYTES == 4) *reinterpret_cast<uint32_t *>(p) = r.value.x;
    else if (BYTES == 2) *reinterpret_cast<uint16_t *>(p) = (uint16_t)r.value.x;
    else *reinterpret_cast<uint8_t *>(p) = (uint8_t)r.value.x;
  }
}

// 4x resolve of an sRGB attachment: the reference's blit routine (Blitter.cpp
// 1505-1545, 1427-1484, 676-690) decodes each sample to linear, averages in
// linear space and encodes the average: per R, G, B channel
// byte * (1 / 255) -> sRGBtoLinear -> * 255, summed in sample order, * 0.25,
// * (1 / 255) -> linearToSRGB -> * 255, rounded to nearest even and
// saturated; alpha takes the same path without the conversions.
__global__ void resolve_srgb8_kernel(const char *src, int srcPitch, long long slice, char *dst, int dstPitch, int w,
                                     int h) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
  if (x >= w || y >= h) return;
  uint32_t s[4];
#pragma unroll
  for (int q = 0; q < 4; q++) s[q] = *reinterpret_cast<const uint32_t *>(src + q * slice + (long long)y * srcPitch + 4ll * x);
  const float un = 1.0f / 255.0f;
  uint32_t o = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    float acc = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      float v = (float)((s[q] >> (8 * k)) & 0xFFu) * un;
      if (k < 3) v = srgb_to_linear(v);
      v = v * 255.0f;
      acc = q == 0 ? v : acc + v;
    }
    float c = acc * 0.25f;
    c = c * un;
    if (k < 3) c = linear_to_srgb(c);
    c = c * 255.0f;
    const int32_t i = rr_round_int(c);
    o |= (uint32_t)(i < 0 ? 0 : (i > 255 ? 255 : i)) << (8 * k);
  }
  *reinterpret_cast<uint32_t *>(dst + (long long)y * dstPitch + 4ll * x) = o;
}

__global__ void resolve_rgba8_kernel(const char *src, int srcPitch, long long slice, char *dst, int dstPitch, int w,
                                     int h) {
  int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
  if (x >= w || y >= h) return;
  uint32_t s[4];
#pragma unroll
  for (int q = 0; q < 4; q++) s[q] = *reinterpret_cast<const uint32_t *>(src + q * slice + (long long)y * srcPitch + 4ll * x);
  uint32_t o = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    uint32_t a = (s[0] >> (8 * k)) & 0xFF, b = (s[1] >> (8 * k)) & 0xFF, c = (s[2] >> (8 * k)) & 0xFF,
             dd = (s[3] >> (8 * k)) & 0xFF;
    uint32_t ab = (a + b + 1) >> 1, cd = (c + dd + 1) >> 1;
    o |= ((ab + cd + 1) >> 1) << (8 * k);
  }
  *reinterpret_cast<uint32_t *>(dst + (long long)y * dstPitch + 4ll * x) = o;
}

__global__ void resolve_rgba32f_kernel(const char *src, int srcPitch, long long slice, char *dst, int dstPitch, int w,
                                       int h) {
  int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
  if (x >= w || y >= h) return;
  float4 s[4];
#pragma unroll
  for (int q = 0; q < 4; q++) s[q] = *reinterpret_cast<const float4 *>(src + q * slice + (long long)y * srcPitch + 16ll * x);
  float4 o;
  o.x = (((s[0].x + s[1].x) + s[2].x) + s[3].x) * 0.25f;
  o.y = (((s[0].y + s[1].y) + s[2].y) + s[3].y) * 0.25f;
  o.z = (((s[0].z + s[1].z) + s[2].z) + s[3].z) * 0.25f;
  o.w = (((s[0].w + s[1].w) + s[2].w) + s[3].w) * 0.25f;
  *reinterpret_cast<float4 *>(dst + (long long)y * dstPitch + 16ll * x) = o;
}

}  // namespace swr
