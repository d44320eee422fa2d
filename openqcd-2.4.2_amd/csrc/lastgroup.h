// lastgroup.h -- sums over a launch by the work-group that finishes last.
//
// The work-groups leave their shares in memory and count themselves in; the
// one that completes the count adds the shares, in a fixed order whichever it
// is, so no second kernel is needed and results do not depend on the timing.
// For launches of up to a few hundred work-groups per count: with 1024 the
// count takes 9 us, where a second kernel takes 5 (Gram-Schmidt of the solver at
// 24^4).  The shares go through agent-scope atomic stores and loads, which bypass
// the caches that are not coherent between the XCDs; with ordinary stores and
// __threadfence every work-group writes the dirty lines of its L2 back.
#ifndef LASTGROUP_H
#define LASTGROUP_H

#include <hip/hip_runtime.h>

namespace oqh {

__device__ inline void put_share(double *p, double v)
{
   __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline double get_share(const double *p)
{
   return __hip_atomic_load(const_cast<double *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// true in the work-group that is the last of n to call this; the shares that
// lane 0 of the others has put before are there then.  cnt is 0 before and after
__device__ inline bool last_group(unsigned *cnt, unsigned n)
{
   __shared__ int last;
   if (threadIdx.x == 0)
   {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      last = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
      if (last) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
   }
   __syncthreads();
   return last;
}

}  // namespace oqh

#endif
