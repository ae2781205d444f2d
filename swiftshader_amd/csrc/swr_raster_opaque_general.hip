// swr_raster_opaque_general.hip -- raster kernels of draws that do not blend, for the general output state and the extended formats.
#include "swr_raster.hpp"

template void swr::launch_raster_general<false>(int, dim3, dim3, hipStream_t, const swr::RasterArgs &);
