// device_numerics.hip -- the device arithmetic of swr_device.hpp that replaces
// longer forms, against those forms over all 2^32 float arguments.  Compiled
// with the library's flags into tests/libswr_numerics.so.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../swiftshader_amd/csrc/swr_device.hpp"

namespace {

using namespace swr;

enum { RCP, PACK, FRAC, ADDRESS16, CHECKS };

// NaN results included, bit for bit.
__device__ bool same(float a, float b) { return __float_as_uint(a) == __float_as_uint(b); }

// rr_round_int of the clamped and scaled channel, the form of the reference.
__device__ uint32_t unorm8(float c) {
  const int32_t i = rr_round_int(rr_min(rr_max(c, 0.0f), 1.0f) * 255.0f);
  return (uint32_t)(i < 0 ? 0 : (i > 255 ? 255 : i));
}

// bad[k]: arguments for which check k differs; arg[k]: the bits of one of them.
// Thread t of 2^20 takes the arguments t, t + 2^20, ...
__global__ __launch_bounds__(256) void sweep_kernel(unsigned long long *bad, uint32_t *arg) {
  unsigned long long n[CHECKS] = {};
  uint32_t last[CHECKS] = {};
  for (uint32_t i = 0; i < 4096; i++) {
    const uint32_t bits = (i << 20) | (blockIdx.x * 256u + threadIdx.x);
    const float x = __uint_as_float(bits);
    const uint32_t u = unorm8(x);
    const float frac = rr_min(x - __builtin_floorf(x), __uint_as_float(0x3F7FFFFFu));
    const uint32_t clamped =
        (uint32_t)rr_trunc_int(rr_min(rr_max(x, 0.0f), 65535.0f / 65536.0f) * 65536.0f) & 0xFFFFu;
    // Each channel at its own place, beside channels that saturate both ways.
    const bool packed = float4_to_unorm8(make_float4(x, 2.0f, -1.0f, x)) == (u | 0xFF00u | (u << 24)) &&
                        float4_to_unorm8(make_float4(-1.0f, x, x, 2.0f)) == ((u << 8) | (u << 16) | 0xFF000000u);
    const bool ok[CHECKS] = {same(rr_rcp(x), 1.0f / x), packed, same(rr_frac(x), frac),
                             address16<false>(x, 1) == clamped};
#pragma unroll
    for (int k = 0; k < CHECKS; k++)
      if (!ok[k]) {
        n[k]++;
        last[k] = bits;
      }
  }
#pragma unroll
  for (int k = 0; k < CHECKS; k++)
    if (n[k]) {
      atomicAdd(bad + k, n[k]);
      arg[k] = last[k];
    }
}

}  // namespace

// Runs the sweep; bad and arg are device arrays of 4 entries, zeroed.
extern "C" int swr_numerics_sweep(unsigned long long *bad, uint32_t *arg) {
  hipLaunchKernelGGL(sweep_kernel, dim3(4096), dim3(256), 0, nullptr, bad, arg);
  return (int)hipGetLastError();
}
