// Right-Jacobi BiCGSTAB in FP64 as one grid-resident launch (resident.hpp):
// the recurrences and tests of bicgstab.hip (reference src/Bicgstab.c:50-245)
// with three grid-wide sums an iteration in place of five kernels.
//
// Per iteration, each thread for its own rows, with the scaled words
// a = D^-1 r, b = D^-1 (p - w v) and c = D^-1 v published for the gathers:
//   1  p = r + beta (p - w v), z = a + beta b; v = A z, formed from the
//      neighbours' a and b; c published; sum v.r0
//   2  alpha; s = r - alpha v, z' = a - alpha c; t = A z' from the
//      neighbours' a and c; sums s.s, t.s, t.t
//   3  half-step test; w; x += alpha z + w z', r = s - w t; a and b
//      published; sums r.r, r.r0; full-step test, beta
// The half-step test follows the second product instead of preceding it (one
// sum fewer; the last iteration of a solve that stops there computes a t it
// does not use).  x, r0, z and D^-1 live in LDS, r, p, v, t in registers: an
// iteration publishes 24 bytes a row and gathers as much, plus the matrix
// twice where it does not fit the registers; bicgstab.hip's five kernels move
// 216 plus the matrix twice.
//
// Measured, loop of kernels -> here: 45^3 momentum solve 402 -> 228 us; u, v and w
// on 96^3 one after another 1.96 -> 1.22 ms against the batched kernels, which
// read the pattern once for the three.  Solves of a few iterations are bound
// by their set-up and final norms, longer ones by three sums an iteration
// (1.9-2.8 us each) and two gathers (at 96^3 39 k L1 accesses a CU and
// iteration, counted: 39 % of its cycles at one a cycle).
#include "resident.hpp"

struct Two {
  double a, b;
};

template <class M, int RPT>
__global__ __launch_bounds__(SFR_RT) void k_bicg_res(M A, const double *__restrict__ dinv,
    const double *__restrict__ r0, double *x, double *r, double *u, double *za, double *zb,
    double *zc, GridSync g, unsigned limit, const sfr_scalars *carry, sfr_scalars *sc)
{
  __shared__ double sx[RPT * SFR_RT], sd[RPT * SFR_RT], sh[RPT * SFR_RT], sz[RPT * SFR_RT];
  // the system before in the batch has stalled, in a launch that is over
  const bool stalled = carry && carry->stall;
  if (sc->done || stalled) {
    if (stalled && blockIdx.x == 0 && threadIdx.x == 0) sc->stall = 1;
    return;
  }
  g.id = blockIdx.x;
  const int n = A.rows();
  const double conv = sc->conv;
  const unsigned maxit = sc->maxit;
  int t = threadIdx.x;
  double rv[RPT], pv[RPT], vv[RPT], tv[RPT];
  typename M::template State<RPT> st;
  unsigned it = sc->iter, ep = sc->ep;
  double rr0 = sc->d, beta = it ? sc->beta : 0.0, alpha = 0.0, w = 0.0;
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    const int i = res_row<RPT>(k, t), s = k * SFR_RT + t;
    const bool valid = i < n;
    A.template load<RPT>(st, k, i, valid);
    rv[k] = valid ? r[i] : 0.0;
    pv[k] = valid && it ? u[i] : 0.0;     // p - w v of the last iteration
    sx[s] = valid ? x[i] : 0.0;
    sd[s] = valid ? dinv[i] : 0.0;
    sh[s] = valid ? r0[i] : 0.0;
  }
  // the first direction is r: beta 0 over a b that has not been written
  const double *bg = it ? zb : za;
  const auto ld1 = [&](int j) { return Two{at_row((const double *)za, j), at_row(bg, j)}; };
  const auto cj1 = [&](Two q) { return fmad(beta, q.b, q.a); };
  const auto ld2 = [&](int j) {
    return Two{at_row((const double *)za, j), at_row((const double *)zc, j)};
  };
  const auto cj2 = [&](Two q) { return fmad(-alpha, q.b, q.a); };
  unsigned done = SFR_DONE_RUN;
  bool ok = true;
  for (unsigned turn = 0; turn < limit; turn++) {
    double a1[1] = {0.0};
    SFR_OPAQUE(t);
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int i = res_row<RPT>(k, t), s = k * SFR_RT + t;
      if (i < n) {
        const double z = fmad(beta, pv[k] * sd[s], rv[k] * sd[s]);
        pv[k] = fmad(beta, pv[k], rv[k]);
        sz[s] = z;
        vv[k] = A.row(st, k, i, z, ld1, cj1);
        agent_store(zc + i, vv[k] * sd[s]);
        a1[0] += vv[k] * sh[s];
      }
      SFR_SCHED_FENCE();
    }
    bg = zb;
    if (!(ok = grid_total<1, true>(a1, g, ++ep))) break;
    alpha = rr0 / a1[0];
    if (!(a1[0] != 0.0) || !isfinite(alpha)) {
      done = SFR_DONE_BREAK;
      break;
    }
    double a3[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int i = res_row<RPT>(k, t), s = k * SFR_RT + t;
      if (i < n) {
        const double si = fmad(-alpha, vv[k], rv[k]);
        tv[k] = A.row(st, k, i, fmad(-alpha, vv[k] * sd[s], rv[k] * sd[s]), ld2, cj2);
        a3[0] += si * si;
        a3[1] += tv[k] * si;
        a3[2] += tv[k] * tv[k];
      }
      SFR_SCHED_FENCE();
    }
    if (!(ok = grid_total<3, false>(a3, g, ++ep))) break;
    const bool half = sqrt(a3[0]) < conv || a3[0] == 0.0;
    w = a3[1] / a3[2];
    if (half) {
      it++;
      done = SFR_DONE_CONV;
    } else if (!isfinite(a3[0]) || !(a3[2] != 0.0) || !(w != 0.0) || !isfinite(w)) {
      done = SFR_DONE_BREAK;
    }
    if (done) {
#pragma unroll
      for (int k = 0; k < RPT; k++) sx[k * SFR_RT + t] += alpha * sz[k * SFR_RT + t];
      break;
    }
    double a2[2] = {0.0, 0.0};
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int i = res_row<RPT>(k, t), s = k * SFR_RT + t;
      if (i < n) {
        const double zs = fmad(-alpha, vv[k] * sd[s], rv[k] * sd[s]);
        sx[s] = fmad(w, zs, fmad(alpha, sz[s], sx[s]));
        rv[k] = fmad(-w, tv[k], fmad(-alpha, vv[k], rv[k]));
        pv[k] = fmad(-w, vv[k], pv[k]);
        agent_store(za + i, rv[k] * sd[s]);
        agent_store(zb + i, pv[k] * sd[s]);
        a2[0] += rv[k] * rv[k];
        a2[1] += rv[k] * sh[s];
      }
    }
    if (!(ok = grid_total<2, true>(a2, g, ++ep))) break;
    beta = (a2[1] / rr0) * (alpha / w);
    const bool brk = !isfinite(a2[0]) || !(rr0 != 0.0) || !isfinite(beta);
    rr0 = a2[1];
    it++;
    if (sqrt(a2[0]) < conv || a2[0] == 0.0) done = SFR_DONE_CONV;
    else if (brk) done = SFR_DONE_BREAK;
    else if (it >= maxit) done = SFR_DONE_MAXIT;
    if (done) break;
  }
  if (!ok) return;
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    const int i = res_row<RPT>(k, t);
    if (i < n) {
      x[i] = sx[k * SFR_RT + t];
      if (!done) {
        r[i] = rv[k];
        u[i] = pv[k];
      }
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    sc->iter = it;
    sc->d = rr0;
    sc->alpha = alpha;
    sc->omega = w;
    sc->beta = beta;
    sc->ep = ep;
    sc->done = done;
  }
}

template <int RPT>
static void launch(hipStream_t s, const sfr_mat_view *A, int wgs, double *x, double *const *w,
                   const GridSync &g, unsigned limit, const sfr_scalars *carry,
                   sfr_scalars *sc)
{
  with_rows<double, RPT>(A, A->val, [&](auto rows) {
    using M = decltype(rows);
    // w: r, r0, p, z, v, t of the set-up: r, r0, u, a, c, b here
    hipLaunchKernelGGL((k_bicg_res<M, RPT>), dim3(wgs), dim3(SFR_RT), 0, s, rows, A->dinv,
                       w[1], x, w[0], w[2], w[3], w[5], w[4], g, limit, carry, sc);
  });
}

extern "C" int sfr_k_bicg_res(hipStream_t s, const sfr_mat_view *A, sfr_res shape, double *x,
                              double *const *w, const sfr_scalars *carry, sfr_scalars *sc,
                              unsigned long long *slot, unsigned limit,
                              unsigned long long patience)
{
  const int64_t room = (int64_t)shape.wgs * shape.rpt * SFR_RT;
  if (A->fmt != SFR_FMT_ELL || room < A->n || shape.wgs > SFR_RES_WG ||
      (shape.wgs != 1 && shape.wgs % 8))
    return hipErrorInvalidValue;
  const GridSync g = {slot, &sc->stall, patience, shape.wgs, 0};
  switch (shape.rpt) {
  case 1: launch<1>(s, A, shape.wgs, x, w, g, limit, carry, sc); break;
  case 2: launch<2>(s, A, shape.wgs, x, w, g, limit, carry, sc); break;
  case 4: launch<4>(s, A, shape.wgs, x, w, g, limit, carry, sc); break;
  default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
