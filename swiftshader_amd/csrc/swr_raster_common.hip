// swr_raster_common.hip -- raster kernels of the common output states (variant_of's levels 1 to 3).
#include "swr_raster.hpp"

namespace swr {

void launch_raster_common(int v, dim3 grid, dim3 block, hipStream_t s, const RasterArgs &a) {
  switch (v >> 4) {
    case 3: launch_raster_variant<false, 3>(v, grid, block, s, a); break;
    case 2: launch_raster_variant<false, 2>(v, grid, block, s, a); break;
    default: launch_raster_variant<false, 1>(v, grid, block, s, a); break;
  }
}

}  // namespace swr
