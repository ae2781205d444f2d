// swr_raster_blend_common.hip -- raster kernels of draws that blend, for the common output states (levels 1 to 3).
#include "swr_raster.hpp"

template void swr::launch_raster_common<true>(int, dim3, dim3, hipStream_t, const swr::RasterArgs &);
