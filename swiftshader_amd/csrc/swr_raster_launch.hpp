// swr_raster_launch.hpp -- host interface of the raster kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "swr_params.hpp"

namespace swr {

// Arguments of one raster launch over tiles [tLo, tHi) of draws [lo, hi).
struct RasterArgs {
  const DrawParams *params;
  const uint32_t *tileBase;
  int lo, hi;
  uint32_t tLo, tHi;
  uint32_t *counter;
  const TriRecord *rec;
  const int *poly;
  const uint32_t *bin;  // NULL: the unbinned pass
  const uint32_t *ts, *te;
  const uint32_t *split;
  uint32_t segT;
  int tail;  // with bin: each tile also walks the slots from *split on
};

// Raster variant of a draw, as bits: what the kernels are specialised for.
// The sample count is the highest bit, so that draws ordered by variant are
// also ordered by sample count.
enum : int {
  kVarFloatTex = 1,    // RGBA32F texture
  kVarFloatColor = 2,  // RGBA32F colour target
  kVarExtended = 4,    // a format or state outside the common set
  kVarLevel1 = 8,      // level (0 to 3), two bits
  kVarLevel = 24,
  kVarBlend = 32,
  kVarSamples = 64,    // 4 samples
  kVarCount = 80       // at most: (3 levels + general + extended) x 16
};

// Launches the raster kernel of a variant (levels 1 to 3; the rest).
template <bool BLEND>
void launch_raster_common(int v, dim3 grid, dim3 block, hipStream_t s, const RasterArgs &a);
template <bool BLEND>
void launch_raster_general(int v, dim3 grid, dim3 block, hipStream_t s, const RasterArgs &a);

}  // namespace swr
