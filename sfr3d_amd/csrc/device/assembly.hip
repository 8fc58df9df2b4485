// Device assembly: per-cell coefficients scattered into a resident matrix's
// raw value arrays by a plan made once on the host (see host/assembly.c), and
// the device-format values, diagonal and Jacobi inverse that follow from them.
//
// One launch for all of it.  A device-format value is taken from where its raw
// value comes from, by a map that is composed with the plan when that is
// made: one index, one load.  What bounds it is memory, about 440 MB at 128^3
// cells, so long as a cell's coefficients (56 bytes of lA) come from there
// once: a workgroup takes all slots, the diagonal and the right-hand side of
// 256 rows and the raw values that lie at the same place of their array, and
// an XCD works on one stretch of rows (workgroups in turn over all: 43, 119,
// 236 us for the first three sizes below).
//
// us an assembly with its right-hand side, CSRD, 80x64x56 / 100^3 / 128^3 / 140^3
// cells: scatters, then a gather and a diagonal kernel 41 / 103 / 197 / 254;
// one launch that took a slot plane after another, and so lA from memory for
// each, 54 / 183 / 340 / not timed; this one 29 / 72 / 170 / 253.
#include "dev_common.hpp"

// plan entry m of a value whose old value is at old[-1 - m]
__device__ __forceinline__ double planned(int32_t m, const double *__restrict__ src,
                                          const double *__restrict__ old)
{
  return m > 0 ? src[m - 1] : m == 0 ? 0.0 : old[-1 - m];
}

// Plan and new values pass the caches by (NT) where the assembly's footprint
// exceeds the last-level cache: 205 -> 170 us at 128^3.  Below, the next
// assembly finds the plan there: 72 us plain, 86 without at 100^3.
template <bool NT, class T>
__device__ __forceinline__ T get(const T *p)
{
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}
template <bool NT>
__device__ __forceinline__ void put(double *p, double v)
{
  if constexpr (NT) __builtin_nontemporal_store(v, p);
  else *p = v;
}

// entries lo .. hi of a value array, four a thread in flight
template <bool NT, class F>
__device__ __forceinline__ void stretch(int64_t lo, int64_t hi, const int32_t *__restrict__ map, F each)
{
  constexpr int U = 4;
  for (int64_t k0 = lo + threadIdx.x; k0 < hi; k0 += U * SFR_BLOCK) {
    int32_t m[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int64_t k = k0 + u * SFR_BLOCK;
      m[u] = k < hi ? get<NT>(map + k) : 0;
    }
#pragma unroll
    for (int u = 0; u < U; u++)
      if (k0 + u * SFR_BLOCK < hi) each(k0 + u * SFR_BLOCK, m[u]);
  }
}

// S: slots of an ELL matrix, 0: read at run time, -1: CSR rows
template <int S, bool NT>
__global__ __launch_bounds__(SFR_BLOCK) void k_assemble(sfr_asm_args a)
{
  const int64_t n = a.n, chunks = (n + SFR_BLOCK - 1) / SFR_BLOCK;
  for (int64_t c = xcd_chunk(blockIdx.x, gridDim.x); c < chunks; c += gridDim.x) {
    const int64_t i = c * SFR_BLOCK + threadIdx.x;
    if (i < n && a.matrix) {
      if constexpr (S > 0) {
        int32_t m[S];
        double v[S];
#pragma unroll
        for (int f = 0; f < S; f++) m[f] = get<NT>(a.vsrc + f * n + i);
#pragma unroll
        for (int f = 0; f < S; f++) v[f] = planned(m[f], a.lA, a.raw);
#pragma unroll
        for (int f = 0; f < S; f++) put<NT>(a.val + f * n + i, v[f]);
      } else if constexpr (S == 0) {
        for (int f = 0; f < a.slots; f++)
          a.val[f * n + i] = planned(a.vsrc[f * n + i], a.lA, a.raw);
      }
      const int32_t m = a.dsrc[i];
      // a diagonal of its own that the plan leaves alone stays where it is
      const double d = m < 0 && a.raw_ad ? a.raw_ad[i] : planned(m, a.lA, a.raw);
      if (a.raw_ad) a.raw_ad[i] = d;
      a.ad[i] = d;
      a.dinv[i] = 1.0 / d;                 // preCondDiag, src/PreCond.c:18-26
    }
    if (i < n && a.b) {
      const int32_t m = a.bmap[i];
      if (m >= 0) a.b[i] = m > 0 ? a.lB[m - 1] : 0.0;
    }
    if (!a.matrix) continue;
    if constexpr (S < 0)
      stretch<NT>(a.nnz * c / chunks, a.nnz * (c + 1) / chunks, a.vsrc,
              [&](int64_t k, int32_t m) { a.val[k] = planned(m, a.lA, a.raw); });
    stretch<NT>(a.nraw * c / chunks, a.nraw * (c + 1) / chunks, a.amap, [&](int64_t k, int32_t m) {
      if (m >= 0) a.raw[k] = m > 0 ? a.lA[m - 1] : 0.0;
    });
  }
}

extern "C" int sfr_k_assemble(hipStream_t s, const sfr_asm_args *a)
{
  int64_t g = ((a->n + SFR_BLOCK - 1) / SFR_BLOCK + 7) & ~(int64_t)7;
  if (g > 16 * SFR_GRIDCAP) g = 16 * SFR_GRIDCAP;
  if (g <= 0) return hipSuccess;
  // maps, values written, coefficients read, the diagonal and b: see SFR_LLC_BYTES
  const bool nt = 12 * (a->nnz + a->nraw) + 120 * a->n > SFR_LLC_BYTES;
#define GO(S)                                                                       \
  do {                                                                              \
    const dim3 grid((unsigned)g), block(SFR_BLOCK);                                 \
    if (nt) hipLaunchKernelGGL((k_assemble<S, true>), grid, block, 0, s, *a);       \
    else hipLaunchKernelGGL((k_assemble<S, false>), grid, block, 0, s, *a);         \
  } while (0)
  switch (a->slots) {
  case -1: GO(-1); break;
  case 4: GO(4); break;
  case 6: GO(6); break;
  default: GO(0); break;
  }
#undef GO
  return hipGetLastError();
}

// Where the values that read raw entry map[k] come from: the plan's entry, or
// -1 - map[k] where it leaves the raw value alone; 0 for padding (map < 0)
__global__ __launch_bounds__(SFR_BLOCK) void k_compose(int64_t n, const int32_t *__restrict__ map,
    const int32_t *__restrict__ plan, int32_t *__restrict__ out)
{
  for (int64_t k = (int64_t)blockIdx.x * SFR_BLOCK + threadIdx.x; k < n;
       k += (int64_t)gridDim.x * SFR_BLOCK) {
    const int32_t r = map[k], m = r < 0 ? 0 : plan[r];
    out[k] = m < 0 ? -1 - r : m;
  }
}

extern "C" int sfr_k_compose(hipStream_t s, int64_t n, const int32_t *map, const int32_t *plan,
                             int32_t *out)
{
  int64_t g = (n + SFR_BLOCK - 1) / SFR_BLOCK;
  if (g > SFR_GRIDCAP) g = SFR_GRIDCAP;
  if (g <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_compose, dim3((unsigned)g), dim3(SFR_BLOCK), 0, s, n, map, plan, out);
  return hipGetLastError();
}
