// TEST INFRASTRUCTURE -- CPU emulation of the HIP kernel model, used only by
// tests/test_emulated_kernels.py to run the library's own .hip sources on a
// machine without a GPU (optionally under AddressSanitizer).  The product
// library never includes or links this.
//
// Every work-item of a workgroup is a fiber on one host thread;
// __syncthreads and each half of a __shfl_xor or __all switch back to a
// scheduler that runs the workgroup's items round-robin until all of them, or
// all lanes of the wave, have come that far.  Workgroups of 1,024 items
// (grid-resident loops, which wait for one another) run side by side, a
// thread each, others one after another; __shared__ is storage of the thread.
// Items that leave a kernel before a barrier that others of their workgroup
// wait at end the process.  Kernel arguments are copied at launch
// (as a real launch does), and launches made during stream capture are
// recorded and replayed by the graph launch.
#pragma once
#include <cmath>
#include <cstdint>
#include <cstring>
#include <functional>
using std::isfinite;
using std::sqrt;
using std::fabs;

#undef __global__
#undef __device__
#undef __host__
#undef __shared__
#undef __forceinline__
#undef __launch_bounds__
#define __global__
#define __device__
#define __host__
#define __shared__ static thread_local
#define __forceinline__ inline
#define __launch_bounds__(...)
#ifndef HIP_SYMBOL
#define HIP_SYMBOL(X) X
#endif
#ifndef __align__
#define __align__(n) __attribute__((aligned(n)))
#endif

namespace emu {
struct Idx { unsigned x, y, z; };
extern thread_local Idx tIdx, bIdx;
extern Idx gDim, bDim;
extern thread_local int lane;
void sync_block();
double shfl(double v, int src);
int all(int v);
bool late(unsigned long long slot);
void launch_fn(std::function<void()> f, unsigned grid, unsigned block);
unsigned long long clock();
template <class F, class... A>
void launch(F k, dim3 g, dim3 b, A... args)
{
  launch_fn([k, args...]() { k(args...); }, g.x, b.x);
}
}  // namespace emu

#define threadIdx emu::tIdx
#define blockIdx emu::bIdx
#define gridDim emu::gDim
#define blockDim emu::bDim

inline void __syncthreads() { emu::sync_block(); }
template <class T>
inline T __shfl_xor(T v, int off, int width = 64)
{
  const int l = emu::lane;
  const int src = (l & ~(width - 1)) | ((l & (width - 1)) ^ off);
  return (T)emu::shfl((double)v, src);
}
inline unsigned long long wall_clock64() { return emu::clock(); }

#define hipLaunchKernelGGL(K, G, B, SHM, S, ...) emu::launch(K, dim3(G), dim3(B), __VA_ARGS__)
inline int __builtin_amdgcn_readfirstlane(int v) { return v; }
template <class T> inline T __builtin_nontemporal_load(const T *p) { return *p; }
template <class T> inline void __builtin_nontemporal_store(T v, T *p) { *p = v; }
// what the grid-resident loops use to publish and to wait
#define __HIP_MEMORY_SCOPE_AGENT 0
namespace emu {
template <class T> inline T load(const T *p)
{
  const T v = __atomic_load_n(p, __ATOMIC_SEQ_CST);
  if (sizeof(T) == 8 && late((unsigned long long)v)) return 0;
  return v;
}
}  // namespace emu
#define __hip_atomic_load(P, ORDER, SCOPE) emu::load(P)
#define __hip_atomic_store(P, V, ORDER, SCOPE) __atomic_store_n(P, V, __ATOMIC_SEQ_CST)
#define __builtin_amdgcn_fence(ORDER, SCOPE) __atomic_thread_fence(__ATOMIC_SEQ_CST)
#define __builtin_amdgcn_s_waitcnt(IMM) ((void)0)
inline int __all(int v) { return emu::all(v); }
