// sqrt_rn_f32 and rcp_rn (openabl_amd/csrc/abl_device.hpp) on the device for every
// bit pattern of a float they are for -- a root's argument has no sign, but for
// zero -- against the double root rounded to float (correctly rounded, innocuously
// rounded twice) and the IEEE divisions.
#include "abl_device.hpp"

namespace {

// 2^20 threads, 4,096 patterns each; bad[0]: roots, bad[1]: reciprocals.
__global__ void k_check(unsigned long long *bad) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  unsigned long long roots = 0, rcps = 0;
  for (uint32_t h = 0; h < 4096u; h++) {
    const uint32_t bits = (h << 20) | t;
    const float f = __builtin_bit_cast(float, bits);
    const float r = abl::sqrt_rn_f32(f), want = (float) __builtin_sqrt((double) f);
    const bool same = __builtin_bit_cast(uint32_t, r) == __builtin_bit_cast(uint32_t, want);
    if (bits <= 0x80000000u && !same && !(r != r && want != want)) roots++;
    const float m = __builtin_fabsf(f);
    if (m >= 0x1p-100f && m <= 0x1p100f) {
      if (abl::rcp_rn<double>(f) != 1.0 / (double) f) rcps++;
      if (abl::rcp_rn<float>(f) != 1.0f / f) rcps++;
    }
  }
  if (roots) atomicAdd(&bad[0], roots);
  if (rcps) atomicAdd(&bad[1], rcps);
}

}  // namespace

extern "C" int root_rcp_check(unsigned long long out[2]) {
  unsigned long long *bad = nullptr;
  out[0] = out[1] = 0;
  if (hipMalloc(&bad, 16) != hipSuccess) return 1;
  int rc = hipMemcpy(bad, out, 16, hipMemcpyHostToDevice) != hipSuccess;
  if (!rc) hipLaunchKernelGGL(k_check, 4096, 256, 0, 0, bad);
  rc = rc || hipGetLastError() != hipSuccess ||
       hipMemcpy(out, bad, 16, hipMemcpyDeviceToHost) != hipSuccess;
  return hipFree(bad) != hipSuccess || rc;
}
