// Grid-resident solver loops: every workgroup of the launch stays on its CU
// for many iterations, keeps its rows' vectors in registers and LDS, and
// meets the others at grid-wide sums instead of at kernel boundaries.
//
// Why: a kernel boundary with its launch, its scalar and partial loads and
// its ramp costs 3-4 us, and a loop of three kernels re-reads every vector
// from memory between them.  A grid-wide sum here costs (MI355X, measured,
// 1,024 threads a workgroup) 1.35 us over 8 workgroups, 1.9 us over 64 or
// 128 and 2.8 us over 256; only what other workgroups gather crosses memory.
//
// One grid-wide sum (grid_total): each workgroup adds its rows' values and
// posts the sum in its slot, two 64-bit words of half a double and the sum's
// number each, so that a slot is its own arrival flag.  The first four waves
// of every workgroup read all slots, one a lane, until each carries the
// number, and add them in one fixed order: all workgroups get bitwise the
// same total, and so take the same decisions.  Slots alternate between two sets: a workgroup
// posts sum k + 2 only after sum k + 1, that is after every workgroup has
// finished reading sum k.
//
// Visibility between XCDs (each has its own L2):
//  - what others gather, and the slots, is written by agent-scope atomic
//    stores, which go through to memory; a wave waits for its stores before
//    its workgroup posts the slot that announces them;
//  - the sum that precedes a gathering phase (ACQ) invalidates this CU's L1
//    and this XCD's L2 by an agent-scope acquire.  No workgroup gathers
//    between the sum before and this one, so an invalidation anywhere in
//    between removes every stale line; the last wave issues it while the
//    first ones poll (after the poll it cost 1.5 us more at 256 workgroups).
//
// Every wait ends: a wave that has polled for `patience` clock ticks (0: once)
// marks the launch stalled and leaves, the others see the mark and leave too, and
// the host then runs the loop of kernels instead.  That happens only if
// some workgroup cannot get a CU for that long: the host never has more
// resident workgroups of this process on a device than it has CUs, but another
// process's resident launches may hold some.  A workgroup may give up on a
// sum that the others see complete, so what they record of a marked launch
// does not count.
#pragma once

#include "dev_common.hpp"

#define SFR_RT 1024                      // threads of a resident workgroup
#define SFR_RWV (SFR_RT / 64)            // its waves: 16, a row of lanes
static_assert(SFR_RWV == 16, "a workgroup's wave sums fill one row of lanes");
#define SFR_RES_POLL (SFR_RES_WG / 64)   // waves that poll, a slot a lane

// What the G workgroups that sum together share, and this one's place among
// them: the slots (2 x 4 x G x 2 words, zero before the first sum of a
// solve) and the stall mark.
struct GridSync {
  unsigned long long *slot;
  unsigned *stall;
  unsigned long long patience;
  int G, id;
};

__device__ __forceinline__ unsigned long long bits_of(double v)
{
  unsigned long long u;
  __builtin_memcpy(&u, &v, sizeof u);
  return u;
}
__device__ __forceinline__ double of_bits(unsigned long long u)
{
  double v;
  __builtin_memcpy(&v, &u, sizeof v);
  return v;
}

__device__ __forceinline__ void agent_store(double *p, double v)
{
  __hip_atomic_store((unsigned long long *)p, bits_of(v), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

// Sum over the wave, the same bits in every lane, by data-parallel-primitive
// moves inside the rows of 16 lanes and lane reads across them: a step costs
// an add's latency, where a shuffle goes through the LDS pipe (0.05 us a step;
// an iteration of the resident loops has 30 of them in one chain).
#ifdef __HIP_DEVICE_COMPILE__
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v)
{
  const unsigned long long u = bits_of(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)u, CTRL, 0xf, 0xf, true);
  const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, 0xf, 0xf, true);
  return v + of_bits((unsigned long long)hi << 32 | lo);
}
__device__ __forceinline__ double lane_of(double v, int l)
{
  const unsigned long long u = bits_of(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(u >> 32), l);
  return of_bits((unsigned long long)hi << 32 | lo);
}
// sum over each row of 16 lanes
__device__ __forceinline__ double row_sum(double v)
{
  v = dpp_add<0xb1>(v);                  // quad_perm 1,0,3,2
  v = dpp_add<0x4e>(v);                  // quad_perm 2,3,0,1
  v = dpp_add<0x141>(v);                 // row_half_mirror
  return dpp_add<0x140>(v);              // row_mirror
}
__device__ __forceinline__ double wave_total(double v)
{
  v = row_sum(v);
  return (lane_of(v, 0) + lane_of(v, 16)) + (lane_of(v, 32) + lane_of(v, 48));
}
#else
__device__ inline double row_sum(double v)
{
  for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
__device__ inline double wave_total(double v) { return wave_sum(v); }
#endif

// {r, p} of a row in one 64-bit word
__device__ __forceinline__ unsigned long long pair_bits(float r, float p)
{
  unsigned a, b;
  __builtin_memcpy(&a, &r, 4);
  __builtin_memcpy(&b, &p, 4);
  return (unsigned long long)b << 32 | a;
}
__device__ __forceinline__ float comb(unsigned long long u, float beta)
{
  const unsigned a = (unsigned)u, b = (unsigned)(u >> 32);
  float r, p;
  __builtin_memcpy(&r, &a, 4);
  __builtin_memcpy(&p, &b, 4);
  return fmad(beta, p, r);
}

// this wave's stores are complete at the scope they were made for
__device__ __forceinline__ void stores_done()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0x0f70);    // vmcnt(0)
}

// Add v over all threads of the G workgroups; every thread gets the totals.
// ep: the sum's number, the same in every workgroup, ascending from 1.
// Returns false when the launch has stalled (the caller leaves the loop).
// Other workgroups may set the stall mark at any time, so a workgroup whose
// waves each looked at it before a barrier could leave in part; only here does
// it look, for all of its threads.  LOOK: before it waits, too (the first sum of
// a launch queued behind one that may have stalled).
template <int NV, bool ACQ, bool LOOK = false>
__device__ __forceinline__ bool grid_total(double (&v)[NV], const GridSync &g, unsigned ep)
{
  __shared__ double sh[NV][SFR_RWV];
  __shared__ double tot[NV][SFR_RES_POLL];
  __shared__ int ok[SFR_RES_POLL];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, G = g.G;
#pragma unroll
  for (int k = 0; k < NV; k++) {
    v[k] = wave_total(v[k]);
    if (lane == 0) sh[k][w] = v[k];
  }
  stores_done();
  __syncthreads();
  if (ACQ && w == SFR_RWV - 1) {
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    __builtin_amdgcn_s_waitcnt(0x0f70);
  }
  unsigned long long *set = g.slot + (size_t)(ep & 1) * (8 * (size_t)G);
  const unsigned long long tag = (unsigned long long)ep << 32;
  if (w == 0) {
#pragma unroll
    for (int k = 0; k < NV; k++) {
      const double s = row_sum(sh[k][lane & (SFR_RWV - 1)]);
      if (lane == 0) {
        unsigned long long *my = set + ((size_t)k * G + g.id) * 2;
        __hip_atomic_store(my, tag | (bits_of(s) & 0xffffffffull), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(my + 1, tag | (bits_of(s) >> 32), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  if (w < SFR_RES_POLL) {
    // lane's slot: workgroup threadIdx.x's
    const bool mine = (int)threadIdx.x < G;
    unsigned long long lo[NV], hi[NV], t0 = 0;
    bool fine = true;
#pragma unroll
    for (int k = 0; k < NV; k++) lo[k] = hi[k] = 0;
    if (LOOK) fine = !__hip_atomic_load(g.stall, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (unsigned spin = 0; mine && (!LOOK || fine); spin++) {
      bool all = true;
#pragma unroll
      for (int k = 0; k < NV; k++) {
        const unsigned long long *at = set + ((size_t)k * G + threadIdx.x) * 2;
        lo[k] = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        hi[k] = __hip_atomic_load(at + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
#pragma unroll
      for (int k = 0; k < NV; k++)
        all &= (unsigned)(lo[k] >> 32) == ep && (unsigned)(hi[k] >> 32) == ep;
      if (all) break;
      if ((spin & 255) == 255 || !g.patience) {
        const unsigned long long now = wall_clock64();
        if (!t0) t0 = now;
        if (!g.patience || now - t0 > g.patience ||
            __hip_atomic_load(g.stall, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
          __hip_atomic_store(g.stall, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          fine = false;
          break;
        }
      }
    }
#pragma unroll
    for (int k = 0; k < NV; k++) {
      const double s = wave_total(of_bits((hi[k] << 32) | (lo[k] & 0xffffffffull)));
      if (lane == 0) tot[k][w] = s;
    }
    fine = __all(fine);
    if (lane == 0) ok[w] = fine;
  }
  __syncthreads();
  bool fine = true;
#pragma unroll
  for (int j = 0; j < SFR_RES_POLL; j++) fine &= ok[j] != 0;
#pragma unroll
  for (int k = 0; k < NV; k++) {
    double s = tot[k][0];
#pragma unroll
    for (int j = 1; j < SFR_RES_POLL; j++) s += tot[k][j];
    v[k] = s;
  }
  return fine;
}

// Keep what follows from recomputing x in every iteration instead of holding
// it in registers across the loop (the addresses of eight passes of gathers
// are twice the registers a thread has), and keep one pass's loads from
// being moved into the next's.
#ifdef __HIP_DEVICE_COMPILE__
#define SFR_OPAQUE(x) asm volatile("" : "+v"(x))
#define SFR_SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)
#else
#define SFR_OPAQUE(x) (void)(x)
#define SFR_SCHED_FENCE()
#endif

// Rows of a resident workgroup: RPT passes of SFR_RT consecutive rows.  The
// grid is a multiple of 8 workgroups (or 1), handed to the XCDs round-robin:
// XCD x owns one contiguous eighth of the rows, and in each pass its
// workgroups lie next to one another, so what they gather in a pass is a
// compact piece of that XCD's L2.
template <int RPT>
__device__ __forceinline__ int res_row(int r, int t)
{
  const int G = gridDim.x;
  const int x = G >= 8 ? (blockIdx.x & 7) : 0, per = G >= 8 ? G >> 3 : 1;
  const int b = G >= 8 ? blockIdx.x >> 3 : 0;
  return ((x * RPT + r) * per + b) * SFR_RT + t;
}

__device__ __forceinline__ int clamp_row(int i, int n) { return i < n ? i : n - 1; }

// a 32-bit byte offset from a uniform base: one address register a gather
template <class T>
__device__ __forceinline__ T at_row(const T *base, int i)
{
  return *(const T *)((const char *)base + (unsigned)i * (unsigned)sizeof(T));
}

// ---- row operators of a resident loop ---------------------------------------
// State<RPT> holds what a thread keeps of its rows, filled by load(); row()
// forms (A c)_i of its pass r with ci = c_i, c_j = cj(ld(j)) and ld(j) the
// word neighbour j has published: acc = a_ii c_i, then the slots in ascending
// order, the products of dev_common.hpp bit for bit.

// Rows kept in registers: S slots, PK = column offsets packed as 16 bits, else
// one 32-bit column each.  ESC: an escaped offset is kept as the row itself
// and the few rows that have one (bit r of esc) are fixed up as EllOp does (a
// variant of its own: the test costs the others 3-6 % an iteration).
// T = float: the Jacobi-scaled copy, whose diagonal is 1.
template <typename T, int S, bool PK, bool ESC = false>
struct KeptRows {
  static constexpr bool UNIT = sizeof(T) == 4;
  const T *val;
  const double *ad;
  const int32_t *col;
  const int16_t *dcol;
  int n;
  const int64_t *xk;
  const int32_t *xc;
  int nx;
  __device__ __forceinline__ int rows() const { return n; }
  template <int RPT>
  struct State {
    unsigned esc;
    T v[RPT][S];
    double d[UNIT ? 1 : RPT];
    int c[RPT][PK ? (S + 1) / 2 : S];
  };
  template <int RPT>
  __device__ __forceinline__ void load(State<RPT> &st, int r, int i, bool valid) const
  {
#pragma unroll
    for (int f = 0; f < S; f++) st.v[r][f] = valid ? val[(size_t)f * n + i] : T(0);
    if constexpr (!UNIT) st.d[r] = valid ? ad[i] : 0.0;
    if (r == 0) st.esc = 0;
    if constexpr (PK) {
      const auto off = [&](int f) {
        const int d = valid && f < S ? dcol[(size_t)f * n + i] : 0;
        st.esc |= d == SFR_D16_ESC ? 1u << r : 0u;
        return d == SFR_D16_ESC ? 0 : d;
      };
#pragma unroll
      for (int f = 0; f < (S + 1) / 2; f++) {
        const int a = off(2 * f), b = off(2 * f + 1);
        st.c[r][f] = (a & 0xffff) | (int)((unsigned)b << 16);
      }
    } else {
#pragma unroll
      for (int f = 0; f < S; f++) st.c[r][f] = valid ? col[(size_t)f * n + i] : n - 1;
    }
  }
  template <int RPT, class L, class C>
  __device__ __forceinline__ T row(const State<RPT> &st, int r, int i, T ci, L ld, C cj) const
  {
    const auto at = [&](int f) {
      int c = st.c[r][PK ? f / 2 : f];
      SFR_OPAQUE(c);
      if constexpr (PK) return i + (f & 1 ? c >> 16 : (int)(int16_t)c);
      else return c;
    };
    T acc = ci;
    if constexpr (UNIT) {
      // all words before the first product: left to itself the compiler
      // spread the loads out between the products (20.4 against 17.5 us an
      // iteration of the 128^3 mixed loop; FP64, short of registers for
      // them, is 4 % slower this way)
      decltype(ld(0)) w[S];
#pragma unroll
      for (int f = 0; f < S; f++) w[f] = ld(at(f));
      SFR_SCHED_FENCE();
#pragma unroll
      for (int f = 0; f < S; f++) acc = fmad(st.v[r][f], cj(w[f]), acc);
    } else {
      acc = st.d[r] * ci;
#pragma unroll
      for (int f = 0; f < S; f++) acc = fmad(st.v[r][f], cj(ld(at(f))), acc);
    }
    if constexpr (ESC)
      if (st.esc >> r & 1) acc += escaped(i, ci, ld, cj);
    return acc;
  }
  // sum over the escaped entries of row i of a_k (c_col - c_i)
  template <class L, class C>
  __device__ T escaped(int i, T ci, L ld, C cj) const
  {
    T fix = T(0);
    for (int e = 0; e < nx; e++)
      if (xk[e] % n == i) fix += val[xk[e]] * (cj(ld(xc[e])) - ci);
    return fix;
  }
};

// Rows streamed from memory in every iteration, S slots (0: read at run
// time).  IDX: how the columns are read -- 32-bit columns, 16-bit offsets
// (escapes fixed up as EllOp does), or 16-bit offsets with the second slot
// of a face pair taken from the neighbour's first-slot plane (PairOp).
enum { IDX_COL = 0, IDX_D16 = 1, IDX_PAIR = 2 };

template <typename T, int S, int IDX>
struct StreamedRows {
  static constexpr bool UNIT = sizeof(T) == 4;
  const T *val;
  const double *ad;
  const int32_t *col;
  const int16_t *dcol;
  int n, s;
  const int64_t *xk;
  const int32_t *xc;
  int nx;
  __device__ __forceinline__ int rows() const { return n; }
  template <int RPT> struct State {};
  template <int RPT>
  __device__ __forceinline__ void load(State<RPT> &, int, int, bool) const {}
  template <int RPT, class L, class C>
  __device__ __forceinline__ T row(const State<RPT> &, int, int i, T ci, L ld, C cj) const
  {
    T acc = ci;
    if constexpr (!UNIT) acc = at_row(ad, i) * ci;
    if constexpr (IDX == IDX_COL) {
      const int slots = S > 0 ? S : s;
#pragma unroll
      for (int f = 0; f < slots; f++)
        acc = fmad(at_row(val + (size_t)f * n, i), cj(ld(at_row(col + (size_t)f * n, i))), acc);
    } else {
      bool esc = false;
#pragma unroll
      for (int f = 0; f < S; f++) {
        int d = at_row(dcol + (size_t)f * n, i);
        if constexpr (IDX == IDX_PAIR) {
          const int g = pair_src<S>(f);
          const T v = g == f ? at_row(val + (size_t)f * n, i)
                             : (d == 0 ? T(0) : at_row(val + (size_t)g * n, i + d));
          acc = fmad(v, cj(ld(i + d)), acc);
        } else {
          const bool e = d == SFR_D16_ESC;
          esc |= e;
          d = e ? 0 : d;
          acc = fmad(at_row(val + (size_t)f * n, i), cj(ld(i + d)), acc);
        }
      }
      if (IDX == IDX_D16 && esc) {
        T fix = T(0);
        for (int e = 0; e < nx; e++)
          if (xk[e] % n == i) fix += val[xk[e]] * (cj(ld(xc[e])) - ci);
        acc += fix;
      }
    }
    return acc;
  }
};

// Add v over the one workgroup of a launch; every thread gets the totals.
// One barrier: the two sets of sh alternate from sum to sum.
template <int NV>
__device__ __forceinline__ void one_total(double (&v)[NV], unsigned par)
{
  __shared__ double sh[2][NV][SFR_RWV];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < NV; k++) {
    v[k] = wave_total(v[k]);
    if (lane == 0) sh[par & 1][k][w] = v[k];
  }
  __syncthreads();
  // 16 partial sums: one a lane, summed in every row of 16
#pragma unroll
  for (int k = 0; k < NV; k++) v[k] = row_sum(sh[par & 1][k][lane & (SFR_RWV - 1)]);
}

// Call f(rows) with the row operator of a resident loop at rpt passes: kept
// in registers where 128 a thread allow it, else streamed (FP64 through face
// pairs where the view has them).
template <typename T, int RPT, typename F>
__host__ inline void with_rows(const sfr_mat_view *A, const T *val, F &&f)
{
  // passes the registers hold: of six slots an FP64 row takes 17 (packed) or 20,
  // beside 6 to 8 of the loop's vectors, an FP32 row 9 or 12
  constexpr int KEEP_PK = sizeof(T) == 8 ? 4 : 8, KEEP_COL = sizeof(T) == 8 ? 2 : 4;
  const bool pk = A->col16 != nullptr;
  const int n = (int)A->n;
#define KEEP(S, ...)                                                            \
  do {                                                                          \
    f(KeptRows<T, S, __VA_ARGS__>{val, A->ad, A->col, A->col16, n, A->exc_k, A->exc_col, \
                         A->nexc});                                             \
    return;                                                                     \
  } while (0)
#define STREAM(S, IDX)                                                          \
  do {                                                                          \
    f(StreamedRows<T, S, IDX>{val, A->ad, A->col, A->col16, n, A->slots,        \
                              A->exc_k, A->exc_col, A->nexc});                  \
    return;                                                                     \
  } while (0)
  if constexpr (RPT <= KEEP_PK) {
    if (pk && A->nexc == 0 && A->slots == 6) KEEP(6, true);
    if (pk && A->nexc == 0 && A->slots == 4) KEEP(4, true);
    if (pk && A->slots == 6) KEEP(6, true, true);
    if (pk && A->slots == 4) KEEP(4, true, true);
  }
  if constexpr (RPT <= KEEP_COL) {
    if (A->slots == 6) KEEP(6, false);
    if (A->slots == 4) KEEP(4, false);
    if (A->slots == 3) KEEP(3, false);
  }
  if constexpr (RPT > KEEP_PK) {
    if (pk && A->nexc == 0 && A->pair == SFR_PAIR_HEX && A->slots == 6) STREAM(6, IDX_PAIR);
    if (pk && A->nexc == 0 && A->pair == SFR_PAIR_QUAD && A->slots == 4) STREAM(4, IDX_PAIR);
  }
  if constexpr (RPT > KEEP_COL) {
    if (A->col16 && A->slots == 6) STREAM(6, IDX_D16);
    if (A->col16 && A->slots == 4) STREAM(4, IDX_D16);
    if (A->slots == 6) STREAM(6, IDX_COL);
    if (A->slots == 4) STREAM(4, IDX_COL);
    if (A->slots == 3) STREAM(3, IDX_COL);
  }
  STREAM(0, IDX_COL);
#undef STREAM
#undef KEEP
}
