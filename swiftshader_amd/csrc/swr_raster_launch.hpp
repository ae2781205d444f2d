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

// Launches the raster kernel of variant v (variant_of): the common output
// states (levels 1 to 3), and the rest.
void launch_raster_common(int v, dim3 grid, dim3 block, hipStream_t s, const RasterArgs &a);
void launch_raster_general(int v, dim3 grid, dim3 block, hipStream_t s, const RasterArgs &a);

}  // namespace swr
