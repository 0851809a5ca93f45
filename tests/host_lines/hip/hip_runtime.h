// Host stand-in for the part of the HIP runtime header that the line kernels
// use: one thread per lane, barriers between them, no wave-level lock step.
#pragma once
#include <cstddef>
#include <cstdint>

#define __device__
#define __host__
#define __global__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ static

struct HostDim {
  unsigned x = 0, y = 0, z = 0;
};
extern thread_local HostDim threadIdx, blockIdx;

void host_barrier();
bool host_wave_votes(bool vote, unsigned long long* mask);
double host_wave_swap(double v, int from);

inline void __syncthreads() { host_barrier(); }
inline unsigned long long __ballot(bool b)
{
  unsigned long long m = 0;
  host_wave_votes(b, &m);
  return m;
}
inline double __shfl_xor(double v, int off, int) { return host_wave_swap(v, (int)(threadIdx.x & 63) ^ off); }
inline int __popcll(unsigned long long m) { return __builtin_popcountll(m); }
inline int atomicAdd(int* p, int v)
{
  const int old = *p;
  *p += v;
  return old;
}
#define __builtin_amdgcn_s_barrier host_barrier
#define __builtin_amdgcn_readfirstlane(v) (v) /* the kernels pass wave-uniform values */
