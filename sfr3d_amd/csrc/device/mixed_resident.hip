// The FP32 iterations of the mixed-precision PCG (mixed.hip) between two
// folds as one grid-resident launch (resident.hpp): the same recurrences,
// roundings, fold rule and breakdown test, with two grid-wide sums an
// iteration in place of two kernels.
//
// Per iteration, each thread for its own rows:
//   1  p = r + beta p; q = A^ p, formed as A^ (r + beta p) from the
//      neighbours' published r and p; sum p.q
//   2  alpha = r.r / p.q; y += alpha p, r -= alpha q; r and p published as
//      one 8-byte pair; sum r.r; fold decision
// y, r and q live in LDS, p in registers, and with 16-bit offsets the matrix
// too, up to 8 rows a thread (a 128^3 system on 256 CUs): an iteration then
// moves 8 bytes a row of published pairs each way, where the two kernels
// move 72.
//
// Measured: the whole 128^3 solve (1,142 FP32 iterations, 8 folds) 37.9 -> 20.6
// ms, the same bits.  Of an iteration's 17.9 us there the two sums are 5.6;
// counted, its 17.6 k L1 accesses a CU are 43 % of its cycles at one a cycle and
// 2.3 k vector instructions a SIMD 23 % at four each, and it reads 10 MB
// and writes 17 beyond L2.
#include "resident.hpp"

template <class M, int RPT>
__global__ __launch_bounds__(SFR_RT) void k_mx_res(M A, float *y, const float *r, float *pd,
    unsigned long long *pair, GridSync g, unsigned limit, sfr_scalars *sc)
{
  __shared__ float sy[RPT * SFR_RT], sr[RPT * SFR_RT], sq[RPT * SFR_RT], sp[RPT * SFR_RT];
  if (sc->done) return;
  g.id = blockIdx.x;
  const int n = A.rows();
  const double conv = sc->conv, delta2 = sc->delta2;
  const unsigned maxit = sc->maxit;
  int t = threadIdx.x;
  typename M::template State<RPT> st;
  unsigned it = sc->iter, ep = sc->ep, ru = 0;
  double rr = sc->dd[1], rr_old = rr, rho = sc->rho_max, alpha = 0.0;
  // the fold left the direction in pd: published as the pair (p, 0), which
  // beta 0 reads back as p
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    const int i = res_row<RPT>(k, t), s = k * SFR_RT + t;
    const bool valid = i < n;
    A.template load<RPT>(st, k, i, valid);
    const float pi = valid ? pd[i] : 0.0f;
    sp[s] = pi;
    sy[s] = valid ? y[i] : 0.0f;
    sr[s] = valid ? r[i] : 0.0f;
    if (valid)
      __hip_atomic_store(pair + i, pair_bits(pi, 0.0f), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  }
  float fb = 0.0f;
  const auto ld = [&](int j) { return at_row((const unsigned long long *)pair, j); };
  const auto cj = [&](unsigned long long w) { return comb(w, fb); };
  double acc[1] = {0.0};
  bool ok = grid_total<1, true, true>(acc, g, ++ep);
  for (unsigned turn = 0; ok; turn++) {
    acc[0] = 0.0;
    SFR_OPAQUE(t);
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int i = res_row<RPT>(k, t), ic = clamp_row(i, n), s = k * SFR_RT + t;
      // the same rounding as each neighbour's own direction
      const float pi = turn ? fmad(fb, sp[s], sr[s]) : sp[s];
      const float qi = A.row(st, k, ic, pi, ld, cj);
      sp[s] = pi;
      sq[s] = qi;
      acc[0] += i < n ? (double)qi * (double)pi : 0.0;
      SFR_SCHED_FENCE();
    }
    if (!(ok = grid_total<1, false>(acc, g, ++ep))) break;
    alpha = rr / acc[0];
    if (!(acc[0] > 0.0) || !isfinite(alpha)) {
      // FP32 lost positive definiteness: restart from the true residual
      ru = 2;
      break;
    }
    if (rr > rho) rho = rr;
    const float fa = (float)alpha;
    acc[0] = 0.0;
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int i = res_row<RPT>(k, t), s = k * SFR_RT + t;
      if (i < n) {
        const float ri = sr[s] - fa * sq[s];
        sr[s] = ri;
        sy[s] = fmad(fa, sp[s], sy[s]);
        acc[0] += (double)ri * (double)ri;
        __hip_atomic_store(pair + i, pair_bits(ri, sp[s]), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    if (!(ok = grid_total<1, true>(acc, g, ++ep))) break;
    it++;
    rr_old = rr;
    rr = acc[0];
    if (rr < delta2 * rho || rr <= conv * conv || !isfinite(rr) || it >= maxit ||
        turn + 1 >= limit) {
      ru = 1;
      break;
    }
    fb = (float)(rr / rr_old);
  }
  if (!ok) return;
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    const int i = res_row<RPT>(k, t);
    if (i < n) {
      y[i] = sy[k * SFR_RT + t];
      pd[i] = sp[k * SFR_RT + t];
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    sc->iter = it;
    sc->alpha = alpha;
    sc->rho_max = rho;
    sc->d_prev = rr_old;
    sc->ep = ep;
    sc->ru = ru;
  }
}

template <int RPT>
static void launch(hipStream_t s, const sfr_mat_view *A, int wgs, float *y, const float *r,
                   float *pd, double *pair, const GridSync &g, unsigned limit, sfr_scalars *sc)
{
  with_rows<float, RPT>(A, A->val32, [&](auto rows) {
    using M = decltype(rows);
    hipLaunchKernelGGL((k_mx_res<M, RPT>), dim3(wgs), dim3(SFR_RT), 0, s, rows, y, r, pd,
                       (unsigned long long *)pair, g, limit, sc);
  });
}

extern "C" int sfr_k_mx_res(hipStream_t s, const sfr_mat_view *A, sfr_res shape, float *y,
                            const float *r, float *pd, double *pair, sfr_scalars *sc,
                            double *part, unsigned limit, unsigned long long patience)
{
  const int64_t room = (int64_t)shape.wgs * shape.rpt * SFR_RT;
  if (A->fmt != SFR_FMT_ELL || room < A->n || shape.wgs > SFR_RES_WG ||
      (shape.wgs != 1 && shape.wgs % 8))
    return hipErrorInvalidValue;
  const GridSync g = {(unsigned long long *)part, &sc->stall, patience, shape.wgs, 0};
  switch (shape.rpt) {
  case 1: launch<1>(s, A, shape.wgs, y, r, pd, pair, g, limit, sc); break;
  case 2: launch<2>(s, A, shape.wgs, y, r, pd, pair, g, limit, sc); break;
  case 4: launch<4>(s, A, shape.wgs, y, r, pd, pair, g, limit, sc); break;
  case 8: launch<8>(s, A, shape.wgs, y, r, pd, pair, g, limit, sc); break;
  default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
