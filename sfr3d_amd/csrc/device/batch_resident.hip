// The uneven batch (mixed_batch.hip) as one grid-resident launch: each system
// gets workgroups of its own, which sum among themselves (resident.hpp) and
// run the whole of its solve -- FP32 CG on the Jacobi-scaled matrix, FP64
// folds, stop test -- independently of the others' iteration counts.
//
// What bounds the loop of kernels on such a batch is not the rows but three
// kernel boundaries an iteration over the slowest system's count, each kernel
// looking its work up and summing its systems' partials.  Here an iteration
// of a system costs its own sums (1.2-1.9 us each) and its rows' gathers; the
// system with the longest solve bounds the batch.  48 systems of 12^3 to 40^3
// rows: 28.3 -> 5.9 ms, the same bits.
//
// Per system the states, tests and recurrences are those of mixed_batch.hip;
// y, r, q and p live in LDS, the scaled matrix in registers, and {r, p} pairs
// are published for the gathers as in mixed_resident.hip.  A fold adds
// D^-1/2 y to its x (published, then gathered for b - A x in FP64).  A launch
// leaves a system that still runs before the fold that follows `limit`
// iterations, with y and p in the batch's vectors; the next starts there.
#include "resident.hpp"

template <int RPT, bool ESC>
__global__ __launch_bounds__(SFR_RT) void k_ub_res(sfr_ub_view v, const sfr_ub_place *places,
    unsigned long long *pairs, unsigned long long *slots, unsigned *stall, unsigned limit,
    unsigned long long patience)
{
  __shared__ float sy[RPT * SFR_RT], sr[RPT * SFR_RT], sq[RPT * SFR_RT], sp[RPT * SFR_RT];
  typedef KeptRows<float, 6, true, ESC> Kept;
  const sfr_ub_place pl = places[blockIdx.x];
  const sfr_ub_sys S = v.sys[pl.sys];
  sfr_scalars *c = &v.sc[pl.sys];
  // 16 slot words a workgroup, the system's next to one another
  const GridSync g = {slots + 16 * (size_t)(blockIdx.x - pl.id), stall, patience, pl.wgs, pl.id};
  const int n = S.n, slot_n = S.slots;
  double *x = v.x + S.row0;
  const double *b = v.b + S.row0;
  unsigned long long *pair = pairs + S.row0;
  const double conv = c->conv, delta2 = c->delta2;
  const unsigned maxit = c->maxit;
  unsigned it = c->iter, outer = c->outer, ep = c->ep, done = SFR_DONE_RUN;
  const unsigned from = it + outer, was = c->ru;
  double d = 0.0, d_prev = c->d_prev, rho = 0.0, rmr = 0.0, rr64 = 0.0;
  if (c->done) return;
  const Kept A = {S.val32, nullptr, nullptr, S.col16, n, S.exc_k, S.exc_col, (int)S.nexc};
  typename Kept::template State<RPT> st;
  st.esc = 0;
  int t = threadIdx.x;
  const auto row_of = [&](int k) { return (k * pl.wgs + pl.id) * SFR_RT + t; };
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    const int i = row_of(k), s = k * SFR_RT + t;
    const auto off = [&](int f) {
      const int o = i < n && f < slot_n ? (int)S.col16[(size_t)f * n + i] : 0;
      st.esc |= o == SFR_D16_ESC ? 1u << k : 0u;
      return o == SFR_D16_ESC ? 0 : o;
    };
#pragma unroll
    for (int f = 0; f < 6; f++)
      st.v[k][f] = i < n && f < slot_n ? S.val32[(size_t)f * n + i] : 0.0f;
#pragma unroll
    for (int f = 0; f < 3; f++) {
      const int a = off(2 * f), b = off(2 * f + 1);
      st.c[k][f] = (a & 0xffff) | (int)((unsigned)b << 16);
    }
    sy[s] = sr[s] = sq[s] = sp[s] = 0.0f;
  }
  enum { INIT, FOLD, RESTART } mode = INIT;
  double dummy[1] = {0.0};
  float fb = 0.0f;
  const auto ld = [&](int j) { return at_row((const unsigned long long *)pair, j); };
  const auto cj = [&](unsigned long long w) { return comb(w, fb); };
  if (ep) {                                // an earlier launch left off at a fold
    mode = was == RESTART ? RESTART : FOLD;
    for (int k = 0; k < RPT; k++) {
      const int i = row_of(k), s = k * SFR_RT + t;
      if (i < n) {
        sy[s] = v.y[S.row0 + i];
        sp[s] = v.p[S.row0 + i];
      }
    }
  }
  for (;;) {
    // fold: x += D^-1/2 y (INIT: x is given), the FP64 residual, the test
    if (mode != INIT) {
      for (int k = 0; k < RPT; k++) {
        const int i = row_of(k), s = k * SFR_RT + t;
        if (i < n) {
          const double xi = of_bits(__hip_atomic_load((unsigned long long *)(x + i),
                                                      __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT));
          agent_store(x + i, xi + S.dscale[i] * (double)sy[s]);
          sy[s] = 0.0f;
        }
      }
      outer++;
    }
    if (!grid_total<1, true>(dummy, g, ++ep)) return;
    double a4[4] = {0.0, 0.0, 0.0, 0.0};
    for (int k = 0; k < RPT; k++) {
      const int i = row_of(k), s = k * SFR_RT + t;
      if (i < n) {
        double ax = S.ad[i] * x[i];
        for (int f = 0; f < slot_n; f++) {
          const size_t e = (size_t)f * n + i;
          ax = fmad(S.val[e], x[d16_col(S.col16, S.exc_k, S.exc_col, S.nexc, e, i)], ax);
        }
        const double ri = b[i] - ax;
        const float ci = (float)(ri * S.dscale[i]);
        sr[s] = ci;
        a4[0] += ri * (ri * S.dinv[i]);
        a4[1] += ri * ri;
        a4[2] += (double)ci * (double)ci;
        a4[3] += (double)ci * (double)sp[s];
      }
    }
    if (!grid_total<4, false>(a4, g, ++ep)) return;
    rmr = a4[0];
    rr64 = a4[1];
    const double c2 = a4[2];
    const bool stop = sqrt(fabs(rmr)) < conv || rmr == 0.0;
    if (stop) done = SFR_DONE_CONV;
    else if (!isfinite(rmr) || !isfinite(c2) || c2 == 0.0) done = SFR_DONE_BREAK;
    else if (it >= maxit || outer >= maxit) done = SFR_DONE_MAXIT;
    if (done) break;
    const float fo = (float)(c2 / d_prev), fg = (float)(a4[3] / c2);
    for (int k = 0; k < RPT; k++) {
      const int i = row_of(k), s = k * SFR_RT + t;
      if (i < n) {
        const float ri = sr[s];
        const float pi = mode == FOLD ? ri + fo * (sp[s] - fg * ri) : ri;
        sp[s] = pi;
        __hip_atomic_store(pair + i, pair_bits(pi, 0.0f), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    d = rho = c2;
    if (!grid_total<1, true>(dummy, g, ++ep)) return;
    // FP32 iterations to the next fold
    fb = 0.0f;
    for (unsigned turn = 0;; turn++) {
      double acc[1] = {0.0};
      SFR_OPAQUE(t);
#pragma unroll
      for (int k = 0; k < RPT; k++) {
        const int i = row_of(k), ic = clamp_row(i, n), s = k * SFR_RT + t;
        const float pi = turn ? fmad(fb, sp[s], sr[s]) : sp[s];
        const float qi = A.row(st, k, ic, pi, ld, cj);
        sp[s] = pi;
        sq[s] = qi;
        acc[0] += i < n ? (double)qi * (double)pi : 0.0;
        SFR_SCHED_FENCE();
      }
      if (!grid_total<1, false>(acc, g, ++ep)) return;
      const double alpha = d / acc[0];
      if (!(acc[0] > 0.0) || !isfinite(alpha)) {
        // FP32 lost positive definiteness: fold, then go on with p = r
        mode = RESTART;
        break;
      }
      if (d > rho) rho = d;
      d_prev = d;
      const float fa = (float)alpha;
      acc[0] = 0.0;
#pragma unroll
      for (int k = 0; k < RPT; k++) {
        const int i = row_of(k), s = k * SFR_RT + t;
        if (i < n) {
          const float ri = sr[s] - fa * sq[s];
          sr[s] = ri;
          sy[s] = fmad(fa, sp[s], sy[s]);
          acc[0] += (double)ri * (double)ri;
          __hip_atomic_store(pair + i, pair_bits(ri, sp[s]), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      if (!grid_total<1, true>(acc, g, ++ep)) return;
      const double rr = acc[0];
      it++;
      d = rr;
      if (rr < delta2 * rho || rr <= conv * conv || !isfinite(rr) || it >= maxit ||
          turn + 1 >= limit) {
        mode = FOLD;
        break;
      }
      fb = (float)(rr / d_prev);
    }
    if (it + outer - from >= limit) break;
  }
  if (!done)
    for (int k = 0; k < RPT; k++) {
      const int i = row_of(k), s = k * SFR_RT + t;
      if (i < n) {
        v.y[S.row0 + i] = sy[s];
        v.p[S.row0 + i] = sp[s];
      }
    }
  if (pl.id == 0 && threadIdx.x == 0) {
    c->iter = it;
    c->outer = outer;
    c->done = done;
    c->ep = ep;
    c->d_prev = d_prev;
    c->ru = mode;
    c->res[2] = rmr;
    c->res[3] = rr64;
    v.ts[pl.sys] = wall_clock64();
  }
}

extern "C" int sfr_k_ub_res(hipStream_t s, const sfr_ub_view *v, const sfr_ub_place *places,
                            int wgs, int rpt, int esc, unsigned long long *pairs,
                            unsigned long long *slots, unsigned *stall,
                            unsigned limit, unsigned long long patience)
{
  if (wgs < 1 || wgs > SFR_RES_WG) return hipErrorInvalidValue;
#define GO(R)                                                                   \
  do {                                                                          \
    if (esc)                                                                    \
      hipLaunchKernelGGL((k_ub_res<R, true>), dim3(wgs), dim3(SFR_RT), 0, s,    \
                         *v, places, pairs, slots, stall, limit, patience);            \
    else                                                                        \
      hipLaunchKernelGGL((k_ub_res<R, false>), dim3(wgs), dim3(SFR_RT), 0, s,   \
                         *v, places, pairs, slots, stall, limit, patience);            \
  } while (0)
  switch (rpt) {
  case 1: GO(1); break;
  case 2: GO(2); break;
  case 4: GO(4); break;
  case 8: GO(8); break;
  default: return hipErrorInvalidValue;
  }
#undef GO
  return hipGetLastError();
}
