/*
 * Host side of the grid-resident loops (device/resident.hpp): which matrices
 * take one and at what shape, the count of resident workgroups in flight, and
 * how long a context stays away from them after a stall.
 *
 * A resident launch makes progress only when all its workgroups are on CUs at
 * once, and each takes a whole CU.  Two launches that together want more than
 * the device has could each hold half and wait for the other, so a launch
 * enters here first and waits until its workgroups fit beside those of the
 * process's other contexts and threads (small solves run side by side).
 * Kernels that do not wait for one another only delay a launch: they end.  But
 * the resident launches of another process are not counted here, and two
 * that hold CUs from each other wait in vain.  The device side then gives up
 * after the context's resident_wait (two seconds) and the loop of kernels
 * takes over, for the rest of that call and for RES_AWAY such waits: a device
 * that stays shared costs its solves at most one part in RES_AWAY of their time
 * in waits, and one that was shared for a moment goes resident again.
 */
#define _POSIX_C_SOURCE 200809L
#include <pthread.h>
#include <time.h>
#include "../sfr_internal.h"

#define MAXDEV 64
static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static pthread_cond_t freed = PTHREAD_COND_INITIALIZER;
static int in_flight[MAXDEV];

/* Workgroups go to the XCDs in turn, so a launch takes up to ceil(wgs / 8) CUs
 * of each.  Counted singly, 130 and 126 workgroups would fit 256 CUs, yet
 * want 33 of the first XCD's 32 and 33 of the second's: each launch could
 * be left waiting for a CU that the other holds. */
static int whole(int wgs)
{
  return (wgs + 7) & ~7;
}

void sfr_res_enter(int device, int ncu, int wgs)
{
  wgs = whole(wgs);
  pthread_mutex_lock(&mu);
  int *n = &in_flight[device % MAXDEV];
  while (*n && *n + wgs > ncu) pthread_cond_wait(&freed, &mu);
  *n += wgs;
  pthread_mutex_unlock(&mu);
}

void sfr_res_leave(int device, int wgs)
{
  pthread_mutex_lock(&mu);
  in_flight[device % MAXDEV] -= whole(wgs);
  pthread_cond_broadcast(&freed);
  pthread_mutex_unlock(&mu);
}

#define RES_AWAY 64

static double seconds(void)
{
  struct timespec t;
  clock_gettime(CLOCK_MONOTONIC, &t);
  return (double)t.tv_sec + 1e-9 * (double)t.tv_nsec;
}

int sfr_res_open(const sfr_context *ctx)
{
  if (ctx->res_wait < 0) return 0;
  return ctx->res_until == 0 || seconds() >= ctx->res_until;
}

void sfr_res_stalled(sfr_context *ctx)
{
  ctx->res_stalls++;
  ctx->res_until = seconds() + RES_AWAY * ctx->res_wait;
}

/* Workgroups and passes for n rows, `one` passes at most in a single
 * workgroup and `rpt` in several.  A grid sum costs 1.9 us over up to 128 workgroups and 2.8 us
 * over 256, a pass of 1,024 rows about 1 us on its CU, so two passes on 128
 * workgroups come before one on 256 (64^3: FP64 10.20 against 10.45 us an
 * iteration, mixed 9.46 against 10.32) and two on 256 before four on 128
 * (80^3: FP64 12.7 against 14.6 us, mixed 11.3 either way).  Eight passes
 * are what the registers and LDS of a CU hold of CG's vectors, four of
 * BiCGSTAB's. */
static sfr_res shape_of(const sfr_context *ctx, const sfr_matrix *A, int one, int rpt)
{
  static const sfr_res most[] = {{128, 1}, {128, 2}, {SFR_RES_WG, 2}, {SFR_RES_WG, 4},
                                 {SFR_RES_WG, 8}};
  const int64_t n = A->n;
  if (A->fmt != SFR_FMT_ELL || ctx->ncu < SFR_RES_WG || !sfr_res_open(ctx)) return (sfr_res){0, 0};
  for (int k = 1; k <= one; k *= 2)
    if (n <= k * SFR_RES_ROWS) return (sfr_res){1, k};
  for (int k = 0; k < (int)(sizeof most / sizeof most[0]) && most[k].rpt <= rpt; k++) {
    const int64_t rows = (int64_t)most[k].rpt * SFR_RES_ROWS;
    const int64_t wgs = ((n + rows - 1) / rows + 7) & ~(int64_t)7;
    if (wgs <= most[k].wgs) return (sfr_res){(int)wgs, most[k].rpt};
  }
  return (sfr_res){0, 0};
}

/* The FP64 loops gather two published words a neighbour from two arrays, the
 * loops of kernels one.  Where a wave's neighbours share lines that costs
 * little; where each has a line of its own (ell_scattered) it doubles the
 * lines, beyond what the caches of a few CUs hold.  Rows of a cube shuffled in
 * blocks, us of 60 PCG iterations resident / kernels: blocks of 2,048 (54
 * lines) 64^3 1,070 / 1,145, 101^3 2,162 / 2,630; blocks of 8,192 (61) 1,434 /
 * 1,275 and 3,392 / 3,069; all rows (63) 1,921 / 1,664 and 11,086 / 5,860, and
 * 40^3 968 / 925, but 32^3 834 / 882.  BiCGSTAB alike.  The mixed loop's two
 * words lie in one line and it keeps its gain (101^3 4,325 / 8,368). */
sfr_res sfr_pcg_res(const sfr_context *ctx, const sfr_matrix *A)
{
  if (A->rpt_set || A->rpt_pcg || A->scattered) return (sfr_res){0, 0};
  return shape_of(ctx, A, 4, 8);
}

sfr_res sfr_mx_res(const sfr_context *ctx, const sfr_matrix *A)
{
  if (A->rpt_set) return (sfr_res){0, 0};
  return shape_of(ctx, A, 1, 8);
}

sfr_res sfr_bicg_res(const sfr_context *ctx, const sfr_matrix *A)
{
  if (A->rpt_set || A->scattered) return (sfr_res){0, 0};
  return shape_of(ctx, A, 1, 4);
}
