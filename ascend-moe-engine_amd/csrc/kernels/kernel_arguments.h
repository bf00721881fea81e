// Kernel arguments at the start of a launch (device code).
#pragma once

#include <hip/hip_runtime.h>

namespace mlakv {

// Asks for the first `kLines` cache lines (64 bytes) of the kernel's arguments and waits for them once. Read where
// they are used, the arguments come in as many trips as there are lines met in a row, each a miss of the scalar
// cache at the start of a launch. For kernels whose workgroups are one chain of latencies.
template <int kLines>
__device__ __forceinline__ void TouchArguments() {
  const __attribute__((address_space(4))) unsigned* words = (const __attribute__((address_space(4))) unsigned*)__builtin_amdgcn_kernarg_segment_ptr();
  unsigned seen[kLines];
#pragma unroll
  for (int i = 0; i < kLines; ++i) seen[i] = words[16 * i];
#pragma unroll
  for (int i = 0; i < kLines; ++i) asm volatile("" ::"s"(seen[i]));
}

}  // namespace mlakv
