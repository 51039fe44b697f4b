// FP64 matrix-core and wave helpers.
#pragma once

#include <hip/hip_runtime.h>

namespace w2k {

typedef double d4 __attribute__((ext_vector_type(4)));

// Before FP64 MFMA results are read by another instruction: 64 clocks more
// than the compiler leaves after the last MFMA.  It leaves 19 wait
// states (16 passes + 3) after its issue; where that MFMA accumulates onto the
// one just before it, whose end it has to wait for, item 3 of the result was
// read three passes early.
__device__ __forceinline__ void mfma_settle()
{
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_sleep(1);
  __builtin_amdgcn_sched_barrier(0);
}

// LDS written by this wave is read by its other lanes
__device__ __forceinline__ void wave_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// the value of one lane, the same for all
__device__ __forceinline__ double lane_value(double v, int lane)
{
  const long long b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((int)b, lane), hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

}  // namespace w2k
