// Kernel arguments at the start of a launch (device code).
#pragma once

#include <hip/hip_runtime.h>

namespace mlakv {

// Asks for the first `kLines` cache lines (64 bytes) of the kernel's arguments and waits for them once. Read where
// they are used, the arguments come in as many trips as there are lines met in a row, each a miss of the scalar
// cache at the start of a launch. In the kernels that measured faster with it at some sizes and slower at none: the
// units of 16 heads and the appends (figures beside each). Not in the split units and their merge, which lose (beside
// the units of 16 heads), nor in the index-key append (recorded launches of 32 keys 1.91 -> 1.90 us without it, 65536
// keys 8.5 -> 8.4) and the index scores and selection, which were level.
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
