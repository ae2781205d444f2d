// swr_raster_general.hip -- raster kernels of the general output state, and of the extended formats.
#include "swr_raster.hpp"

namespace swr {

void launch_raster_general(int v, dim3 grid, dim3 block, hipStream_t s, const RasterArgs &a) {
  if (v & 8) launch_raster_variant<true, 0>(v, grid, block, s, a);
  else launch_raster_variant<false, 0>(v, grid, block, s, a);
}

}  // namespace swr
