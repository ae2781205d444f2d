// swr_raster_blend_general.hip -- raster kernels of draws that blend, for the general output state and the extended formats.
#include "swr_raster.hpp"

template void swr::launch_raster_general<true>(int, dim3, dim3, hipStream_t, const swr::RasterArgs &);
