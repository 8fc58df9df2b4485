// Device assembly: per-cell coefficients scattered into a resident matrix's
// raw value arrays by a plan made once on the host (see host/assembly.c), and
// the device-format values, diagonal and Jacobi inverse that follow from them.
//
// One launch for all of it.  A device-format entry k holds raw value vmap[k],
// which this launch may be writing; it is therefore taken from where that
// value comes from, the coefficient amap names, and from the raw array only
// where the plan leaves the raw value alone.  In five launches (three
// scatters, a gather, the diagonal) an assembly of 287 k cells took 27 us of
// kernels and four launch gaps; the second read of the coefficients costs
// less than the gaps: two such assemblies with their two cell kernels (172 us)
// went from 255 to 249 us.  What bounds it is memory: plan, coefficients, raw
// and device-format values, about 30 bytes a stored value.
#include "dev_common.hpp"

// what plan entry m puts there: a coefficient, 0, or (m < 0) the old value
__device__ __forceinline__ double planned(int32_t m, const double *__restrict__ src, double old)
{
  return m > 0 ? src[m - 1] : old;
}

__global__ __launch_bounds__(SFR_BLOCK) void k_assemble(sfr_asm_args a)
{
  const int64_t total = a.nnz + a.nraw + a.nd + (a.b ? a.n : 0);
  for (int64_t q = (int64_t)blockIdx.x * SFR_BLOCK + threadIdx.x; q < total;
       q += (int64_t)gridDim.x * SFR_BLOCK) {
    int64_t k = q;
    if (k < a.nnz) {                       // device-format values
      const int32_t r = a.vmap[k];
      double v = 0.0;
      if (r >= 0) {
        const int32_t m = a.amap[r];
        v = planned(m, a.lA, m < 0 ? a.raw[r] : 0.0);
      }
      a.val[k] = v;
      continue;
    }
    k -= a.nnz;
    if (k < a.nraw) {                      // raw values
      const int32_t m = a.amap[k];
      if (m >= 0) a.raw[k] = planned(m, a.lA, 0.0);
      continue;
    }
    k -= a.nraw;
    if (k < a.nd) {                        // diagonal and its inverse
      const int32_t r = a.dmap ? 0 : a.rawd[k];
      const int32_t m = a.dmap ? a.dmap[k] : a.amap[r];
      const double v = planned(m, a.lA, m < 0 ? (a.dmap ? a.raw_ad[k] : a.raw[r]) : 0.0);
      if (a.dmap && m >= 0) a.raw_ad[k] = v;
      a.ad[k] = v;
      a.dinv[k] = 1.0 / v;                 // preCondDiag, src/PreCond.c:18-26
      continue;
    }
    k -= a.nd;                             // right-hand side
    const int32_t m = a.bmap[k];
    if (m >= 0) a.b[k] = planned(m, a.lB, 0.0);
  }
}

extern "C" int sfr_k_assemble(hipStream_t s, const sfr_asm_args *a)
{
  const int64_t total = a->nnz + a->nraw + a->nd + (a->b ? a->n : 0);
  if (total <= 0) return hipSuccess;
  int64_t g = (total + SFR_BLOCK - 1) / SFR_BLOCK;
  if (g > 16 * SFR_GRIDCAP) g = 16 * SFR_GRIDCAP;
  hipLaunchKernelGGL(k_assemble, dim3((unsigned)g), dim3(SFR_BLOCK), 0, s, *a);
  return hipGetLastError();
}
