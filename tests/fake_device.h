// Included before each source of tests/fake_device.cpp's library: what
// wf_noalloc.hip uses that only a device compiler declares.
#ifndef FAKE_DEVICE_H
#define FAKE_DEVICE_H
#include <hip/hip_runtime.h>

#define __align__(n) __attribute__((aligned(n)))
#define HIP_SYMBOL(x) x
#define hipLaunchKernelGGL(...) ((void)0)
#define hipGetSymbolAddress(p, symbol) (*(p) = (symbol), hipSuccess)
static const dim3 blockIdx, blockDim, threadIdx, gridDim;

#endif
