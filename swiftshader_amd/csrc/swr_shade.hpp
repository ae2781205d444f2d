// swr_shade.hpp -- fragment shading from the primitive records: attribute
// interpolation, the quad's texture LOD and the fixed shader family (shared
// by the rasteriser and the gradients).
#pragma once

#include "swr_device.hpp"
#include "swr_params.hpp"

namespace swr {

// Interpolated attribute k at (xf, yf): (x*A + (C + y*B)) * rhw, the
// reference's operation order (QuadRasterizer.cpp:235-250).
__device__ __forceinline__ float interp(const TriRecord &R, int k, float xf, float yf, float rhw) {
  return (xf * R.V[k][0] + (R.V[k][2] + yf * R.V[k][1])) * rhw;
}

__device__ __forceinline__ float quad_rhw(const TriRecord &R, float xf, float yf) {
  const float Dw = R.wC + yf * R.wB;
  return rr_rcp(xf * R.wA + Dw);
}

// Texture LOD state of the 2x2 quad holding pixel (px, py): the lane
// differences of u, v over the quad's pixels (0,0), (1,0), (0,1), helper
// lanes included, evaluated from the plane equations (computeLod2D,
// SamplerCore.cpp:1376-1422).
template <int FA = -1>
__device__ __forceinline__ QuadLod quad_state(const DrawParams &P, const TriRecord &R, int px, int py) {
  const int qx = px & ~1, qy = py & ~1;
  float uq[4], vq[4];
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const float xi = (float)(qx + (i & 1)) - R.x0, yi = (float)(qy + (i >> 1)) - R.y0;
    const float ri = quad_rhw(R, xi, yi);
    uq[i] = interp(R, 4, xi, yi, ri);
    vq[i] = interp(R, 5, xi, yi, ri);
  }
  uq[3] = 0.0f;
  vq[3] = 0.0f;
  return quad_lod<FA>(P.tex, uq, vq);
}

// Shades one queued fragment: the fixed shader family at pixel (px, py)
// of primitive R, with the texture LOD of the 2x2 quad the pixel belongs
// to (helper lanes evaluated from the plane equations).  Output clamped
// for UNORM targets (PixelProgram::clampColor).
// FA >= 0: the draw's shader is MODULATE and its sampler state the common
// one with address mode FA (tex_filter and the other readers of the sampler
// state).
template <bool FCOL, bool FTEX, bool XF, int FA = -1>
__device__ __forceinline__ float4 shade(const DrawParams &P, const TriRecord &R, int px, int py,
                                        bool clampUnorm = true) {
  const int shader = FA >= 0 ? (int)SHADER_MODULATE : P.shader;
  const float xf = (float)px - R.x0, yf = (float)py - R.y0;
  const float rhw = quad_rhw(R, xf, yf);
  float4 col = make_float4(0, 0, 0, 0);
  if (shader != SHADER_SAMPLE) {
    col.x = interp(R, 0, xf, yf, rhw);
    col.y = interp(R, 1, xf, yf, rhw);
    col.z = interp(R, 2, xf, yf, rhw);
    col.w = interp(R, 3, xf, yf, rhw);
  }
  if (shader != SHADER_INTERPOLATE) {
    const float u = interp(R, 4, xf, yf, rhw), v = interp(R, 5, xf, yf, rhw);
    const QuadLod Lq = quad_state<FA>(P, R, px, py);
    float4 c = sample_lane<FTEX, XF, FA>(P.tex, u, v, Lq);
    if (shader == SHADER_MODULATE) {
      c.x = c.x * col.x;
      c.y = c.y * col.y;
      c.z = c.z * col.z;
      c.w = c.w * col.w;
    }
    col = c;
  }
  if (!FCOL && clampUnorm) {
    col.x = rr_min(rr_max(col.x, 0.0f), 1.0f);
    col.y = rr_min(rr_max(col.y, 0.0f), 1.0f);
    col.z = rr_min(rr_max(col.z, 0.0f), 1.0f);
    col.w = rr_min(rr_max(col.w, 0.0f), 1.0f);
  }
  return col;
}

}  // namespace swr
