// Jacobi-preconditioned CG in FP64 as one grid-resident launch (resident.hpp):
// the recurrences, tests and products of pcg.hip (reference src/Cg.c:47-209)
// with two grid-wide sums an iteration in place of three kernels.
//
// Per iteration, each thread for its own rows:
//   1  p = z + beta p; q = A p, formed as A (z + beta p) from the neighbours'
//      z and p of the last iteration; sum p.q
//   2  alpha = d / p.q; x += alpha p, r -= alpha q, z = D^-1 r; sum r.z;
//      z and p are published for the next gathers
// x and D^-1 live in LDS, r, p, q in registers, so an iteration moves 16
// bytes a row of published vectors each way, plus the matrix where it does
// not fit the registers.  pcg.hip's loop moves 140.
//
// Measured, whole solves, loop of kernels -> here: 32x32 (one workgroup)
// 3.26 -> 0.53 ms, 128x128 12.6 -> 7.0 ms, 61x47x38 8.9 -> 6.2 ms, 128^3 (1,140
// iterations) 63.1 -> 45.5 ms.  Up to about 130 k rows the two sums bound an
// iteration (1.2 us each in one workgroup, 1.9 over 128, 2.8 over 256); at
// 128^3 the rows do: 52.8 k L1 accesses a CU (counted), 60 % of an
// iteration's 88 k cycles at one a cycle, for the gathers of z and p and the
// streamed matrix.  The vector unit has 2.8 k instructions a SIMD, and 72 MB read
// and 34 MB written beyond L2 are 2.7 TB/s: neither is near its rate.
//
// z_j + beta p_j is formed in every gather exactly as row j forms its own p
// (one fused multiply-add), so the products are those with the stored p.
#include "resident.hpp"

// what a row publishes
struct ZP {
  double z, p;
};

template <class M, int RPT>
__global__ __launch_bounds__(SFR_RT) void k_pcg_res(M A, const double *__restrict__ dinv,
    double *x, double *r, double *z, double *p, GridSync g, unsigned limit, sfr_scalars *sc)
{
  __shared__ double sx[RPT * SFR_RT], sd[RPT * SFR_RT];
  if (sc->done) return;
  g.id = blockIdx.x;
  const int n = A.rows();
  int t = threadIdx.x;
  const double conv = sc->conv;
  const unsigned maxit = sc->maxit;
  double rv[RPT], pv[RPT], qv[RPT];
  typename M::template State<RPT> st;
  unsigned it = sc->iter;
  unsigned ep = sc->ep;
  double d = sc->d, beta = it ? sc->beta : 0.0;
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    const int i = res_row<RPT>(k, t);
    const bool valid = i < n;
    A.template load<RPT>(st, k, i, valid);
    rv[k] = valid ? r[i] : 0.0;
    pv[k] = valid && it ? p[i] : 0.0;
    sx[k * SFR_RT + t] = valid ? x[i] : 0.0;
    sd[k * SFR_RT + t] = valid ? dinv[i] : 0.0;
  }
  // the first direction is z: beta 0 over a p that has not been written
  const double *pg = it ? p : z;
  const auto ld = [&](int j) { return ZP{at_row((const double *)z, j), at_row(pg, j)}; };
  const auto cj = [&](ZP w) { return fmad(beta, w.p, w.z); };
  unsigned done = SFR_DONE_RUN;
  bool ok = true;
  for (unsigned turn = 0; turn < limit; turn++) {
    double acc[1] = {0.0};
    SFR_OPAQUE(t);
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      // a pass at a time behind a branch of its own: in one block the passes'
      // loads were scheduled for low register pressure, one after another
      // (41.5 against 37.4 us an iteration at 128^3)
      const int i = res_row<RPT>(k, t);
      if (i < n) {
        pv[k] = fmad(beta, pv[k], rv[k] * sd[k * SFR_RT + t]);
        qv[k] = A.row(st, k, i, pv[k], ld, cj);
        acc[0] += qv[k] * pv[k];
      }
      SFR_SCHED_FENCE();
    }
    if (!(ok = grid_total<1, false>(acc, g, ++ep))) break;
    const double alpha = d / acc[0];
    if (!(acc[0] != 0.0) || !isfinite(alpha)) {
      done = SFR_DONE_BREAK;
      break;
    }
    acc[0] = 0.0;
    pg = p;
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int i = res_row<RPT>(k, t);
      const int s = k * SFR_RT + t;
      if (i < n) {
        sx[s] += alpha * pv[k];
        rv[k] -= alpha * qv[k];
        const double zi = rv[k] * sd[s];
        acc[0] += rv[k] * zi;
        agent_store(z + i, zi);
        agent_store(p + i, pv[k]);
      }
    }
    if (!(ok = grid_total<1, true>(acc, g, ++ep))) break;
    const double di = acc[0];
    beta = di / d;
    d = di;
    it++;
    if (sqrt(fabs(di)) < conv || di == 0.0) done = SFR_DONE_CONV;
    else if (!isfinite(di)) done = SFR_DONE_BREAK;
    else if (it >= maxit) done = SFR_DONE_MAXIT;
    if (done) break;
  }
  if (!ok) return;
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    const int i = res_row<RPT>(k, t);
    if (i < n) {
      x[i] = sx[k * SFR_RT + t];
      if (!done) r[i] = rv[k];
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    sc->iter = it;
    sc->d = d;
    sc->beta = beta;
    sc->ep = ep;
    sc->done = done;
  }
}

// The same loop in one workgroup (up to 4 x 1,024 rows): the direction is
// gathered from LDS, the sums and the exchange are workgroup barriers.
template <class M, int RPT>
__global__ __launch_bounds__(SFR_RT) void k_pcg_one(M A, const double *__restrict__ dinv,
    double *x, double *r, double *p, unsigned limit, sfr_scalars *sc)
{
  __shared__ double sp[RPT * SFR_RT], sx[RPT * SFR_RT], sd[RPT * SFR_RT];
  if (sc->done) return;
  const int n = A.rows();
  int t = threadIdx.x;
  const double conv = sc->conv;
  const unsigned maxit = sc->maxit;
  double rv[RPT], pv[RPT], qv[RPT];
  typename M::template State<RPT> st;
  unsigned it = sc->iter;
  double d = sc->d;
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    const int i = res_row<RPT>(k, t);
    const int s = k * SFR_RT + t;
    const bool valid = i < n;
    A.template load<RPT>(st, k, i, valid);
    rv[k] = valid ? r[i] : 0.0;
    sx[s] = valid ? x[i] : 0.0;
    sd[s] = valid ? dinv[i] : 0.0;
    pv[k] = it ? (valid ? p[i] : 0.0) : rv[k] * sd[s];
    sp[s] = pv[k];
  }
  __syncthreads();
  const auto ld = [&](int j) { return sp[j]; };
  const auto cj = [](double w) { return w; };
  unsigned done = SFR_DONE_RUN;
  for (unsigned turn = 0; turn < limit; turn++) {
    double acc[1] = {0.0};
    SFR_OPAQUE(t);
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int i = res_row<RPT>(k, t);
      qv[k] = A.row(st, k, clamp_row(i, n), pv[k], ld, cj);
      acc[0] += i < n ? qv[k] * pv[k] : 0.0;
    }
    one_total<1>(acc, 0);
    const double alpha = d / acc[0];
    if (!(acc[0] != 0.0) || !isfinite(alpha)) {
      done = SFR_DONE_BREAK;
      break;
    }
    acc[0] = 0.0;
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int s = k * SFR_RT + t;
      if (res_row<RPT>(k, t) < n) {
        sx[s] += alpha * pv[k];
        rv[k] -= alpha * qv[k];
        acc[0] += rv[k] * (rv[k] * sd[s]);
      }
    }
    one_total<1>(acc, 1);
    const double di = acc[0], beta = di / d;
    d = di;
    it++;
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int s = k * SFR_RT + t;
      pv[k] = fmad(beta, pv[k], rv[k] * sd[s]);
      sp[s] = pv[k];
    }
    __syncthreads();
    if (sqrt(fabs(di)) < conv || di == 0.0) done = SFR_DONE_CONV;
    else if (!isfinite(di)) done = SFR_DONE_BREAK;
    else if (it >= maxit) done = SFR_DONE_MAXIT;
    if (done) break;
  }
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    const int i = res_row<RPT>(k, t);
    if (i < n) {
      x[i] = sx[k * SFR_RT + t];
      r[i] = rv[k];
      p[i] = pv[k];
    }
  }
  if (threadIdx.x == 0) {
    sc->iter = it;
    sc->d = d;
    sc->done = done;
  }
}

template <int RPT>
static void launch(hipStream_t s, const sfr_mat_view *A, int wgs, double *x, double *r,
                   double *z, double *p, const GridSync &g, unsigned limit, sfr_scalars *sc)
{
  with_rows<double, RPT>(A, A->val, [&](auto rows) {
    using M = decltype(rows);
    if constexpr (RPT <= 4)
      if (wgs == 1) {
        hipLaunchKernelGGL((k_pcg_one<M, RPT>), dim3(1), dim3(SFR_RT), 0, s, rows, A->dinv, x,
                           r, p, limit, sc);
        return;
      }
    hipLaunchKernelGGL((k_pcg_res<M, RPT>), dim3(wgs), dim3(SFR_RT), 0, s, rows, A->dinv, x, r,
                       z, p, g, limit, sc);
  });
}

extern "C" int sfr_k_pcg_res(hipStream_t s, const sfr_mat_view *A, sfr_res shape, double *x,
                             double *r, double *z, double *p, sfr_scalars *sc, double *part,
                             unsigned limit, unsigned long long patience)
{
  // what the kernels assume of the grid: every row has one place in it, and
  // the polling lanes cover all workgroups
  const int64_t room = (int64_t)shape.wgs * shape.rpt * SFR_RT;
  if (A->fmt != SFR_FMT_ELL || room < A->n || shape.wgs > SFR_RES_WG ||
      (shape.wgs != 1 && shape.wgs % 8) || (shape.wgs == 1 && shape.rpt > 4))
    return hipErrorInvalidValue;
  const GridSync g = {(unsigned long long *)part, &sc->stall, patience, shape.wgs, 0};
  switch (shape.rpt) {
  case 1: launch<1>(s, A, shape.wgs, x, r, z, p, g, limit, sc); break;
  case 2: launch<2>(s, A, shape.wgs, x, r, z, p, g, limit, sc); break;
  case 4: launch<4>(s, A, shape.wgs, x, r, z, p, g, limit, sc); break;
  case 8: launch<8>(s, A, shape.wgs, x, r, z, p, g, limit, sc); break;
  default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
