// FP64 matrix-core and wave helpers.
#pragma once

#include <hip/hip_runtime.h>

namespace w2k {

typedef double d4 __attribute__((ext_vector_type(4)));

// To stand between an FP64 MFMA that accumulates onto the one just before it and
// the first other instruction that reads its result.  The compiler leaves 19
// wait states there (the MFMA's 16 passes and 3), counted from its issue; but it
// may have had to wait for the one before: read 19 wait states after its issue,
// item 3 of a result was three passes old.  36 wait states by count cover 16
// passes of the one before, its own 16 and 3; they are enough whether or not
// the compiler adds its own.
//
// An accumulator in AGPRs is copied out in front of whatever stands here: the
// block Cholesky read its sums 19 wait states after a chain's end that way.  A
// kernel whose launch bounds ask for two waves a SIMD (up to 256 registers a
// lane) has its accumulators in VGPRs, if its LDS leaves room for two
// work-groups; where it does not, the chains of two accumulators alternate.
// Neither is the source's to promise: tests/test_mfma_waits.py checks the
// assembly of every kernel, also of those that alternate accumulators and do
// without this (gemm.hip).
__device__ __forceinline__ void mfma_settle()
{
  __builtin_amdgcn_sched_barrier(0);
#ifdef __AMDGCN__
  asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 3");
#endif
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
