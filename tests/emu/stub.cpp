// TEST INFRASTRUCTURE -- host stand-ins for the HIP runtime calls the
// library makes, for the CPU emulation build (see emu.hpp), and the fiber
// scheduler that runs emulated workgroups.  "Device" memory is host memory
// filled with 0x7f bytes (garbage, like fresh device memory, so a read of
// memory never written shows up); copies are memcpy; a device with 4 CUs, or
// SFR_EMU_CUS.
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>
#if defined(__SANITIZE_ADDRESS__)
#include <sanitizer/common_interface_defs.h>
#else
static inline void __sanitizer_start_switch_fiber(void **, const void *, size_t) {}
static inline void __sanitizer_finish_switch_fiber(void *, const void **, size_t *) {}
#endif
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <thread>
#include <vector>
#include "emu.hpp"
#include "sfr_internal.h"

namespace emu {
thread_local Idx tIdx, bIdx;
Idx gDim, bDim;
thread_local int lane;

// Switch stacks: the registers a callee keeps go to the old one.  (swapcontext
// makes two system calls a switch, most of an emulated run's time.)
#ifndef __x86_64__
#error "the emulation's fibers are written for x86-64"
#endif
extern "C" void emu_switch(void **from, void *to);
asm(R"(
.text
.globl emu_switch
.type emu_switch, @function
emu_switch:
  pushq %rbp
  pushq %rbx
  pushq %r12
  pushq %r13
  pushq %r14
  pushq %r15
  movq %rsp, (%rdi)
  movq %rsi, %rsp
  popq %r15
  popq %r14
  popq %r13
  popq %r12
  popq %rbx
  popq %rbp
  ret
.size emu_switch, .-emu_switch
)");

// One workgroup: its work-items are fibers on the thread that runs it, which
// switch back to the scheduler below at a barrier (the workgroup waits for
// all its items) and at a wave exchange (the wave waits for its lanes).
enum { MAXT = 1024, STACK = 256 * 1024 };
enum { RUN, AT_BARRIER, AT_WAVE, GONE };
struct Group {
  void *sched, *item[MAXT];                  // stack pointers
  unsigned char at[MAXT];
  double buf[MAXT];
  char *stacks;
  int cur, n;
  const std::function<void()> *job;
};
static thread_local Group *G;
struct Pool {                                // a thread's Group, kept for its next workgroup
  Group g;
  Pool()
  {
    g.stacks = (char *)mmap(nullptr, (size_t)MAXT * STACK, PROT_READ | PROT_WRITE,
                            MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (g.stacks == MAP_FAILED) { perror("emu: stacks"); abort(); }
  }
  ~Pool() { munmap(g.stacks, (size_t)MAXT * STACK); }
};

static void yield_at(int where)
{
  Group *g = G;
  g->at[g->cur] = (unsigned char)where;
  void *fs = nullptr;
  __sanitizer_start_switch_fiber(&fs, nullptr, 0);   // back to the scheduler's stack
  emu_switch(&g->item[g->cur], g->sched);
  __sanitizer_finish_switch_fiber(fs, nullptr, nullptr);
}

static void item_main()
{
  __sanitizer_finish_switch_fiber(nullptr, nullptr, nullptr);
  (*G->job)();
  G->at[G->cur] = GONE;
  __sanitizer_start_switch_fiber(nullptr, nullptr, 0);
  emu_switch(&G->item[G->cur], G->sched);
}

void sync_block() { yield_at(AT_BARRIER); }

double shfl(double v, int src)
{
  G->buf[G->cur] = v;
  yield_at(AT_WAVE);
  const double r = G->buf[(G->cur & ~63) + src];
  yield_at(AT_WAVE);
  return r;
}

// the lanes of the wave that are still there agree on v
int all(int v)
{
  G->buf[G->cur] = v != 0;
  yield_at(AT_WAVE);
  int r = 1;
  for (int t = G->cur & ~63, e = t + 64; t < e; t++)
    if (G->at[t] != GONE && G->buf[t] == 0.0) r = 0;
  yield_at(AT_WAVE);
  return r;
}

extern "C" {
// Tests of what a workgroup does that waits in vain (grid-resident loops):
// workgroup emu_late_wg never sees the others' sum number emu_late_sum, as if
// its waves had been suspended past its wait; and the items of workgroup
// emu_split_wg from the 512th on enter a kernel only after workgroup 0 has
// left it, workgroup 0 only after the items before have.
int emu_late_wg = -1, emu_split_wg = -1;
unsigned emu_late_sum = 0;
int emu_wide = 0;                            // launches of 1,024-item workgroups
}
static std::atomic<int> split_in, first_out;

bool late(unsigned long long slot)
{
  return emu_late_wg == (int)bIdx.x && (unsigned)(slot >> 32) == emu_late_sum;
}

static void bad(const char *what, unsigned b)
{
  fprintf(stderr, "emu: workgroup %u: %s\n", b, what);
  abort();
}

static void run_block(unsigned b, unsigned block, const std::function<void()> &f)
{
  thread_local Pool pool;
  Group *g = G = &pool.g;
  g->n = (int)block;
  g->job = &f;
  for (int t = 0; t < g->n; t++) {
    // six registers and the entry, which finds its stack as after a call
    void **top = (void **)(g->stacks + (size_t)(t + 1) * STACK) - 1;
    *--top = (void *)item_main;
    for (int k = 0; k < 6; k++) *--top = nullptr;
    g->item[t] = top;
    g->at[t] = RUN;
  }
  bIdx = {b, 0, 0};
  for (bool first = true;; first = false) {
    int live = 0, ran = 0;
    for (int t = 0; t < g->n; t++) {
      if (first && (int)b == emu_split_wg && t == 512) {
        split_in = 1;
        while (!first_out) std::this_thread::yield();
      }
      if (g->at[t] == GONE) continue;
      live++;
      if (g->at[t] != RUN) continue;
      ran++;
      g->cur = t;
      tIdx = {(unsigned)t, 0, 0};
      lane = t & 63;
      void *fs = nullptr;
      __sanitizer_start_switch_fiber(&fs, g->stacks + (size_t)t * STACK, STACK);
      emu_switch(&g->sched, g->item[t]);
      __sanitizer_finish_switch_fiber(fs, nullptr, nullptr);
    }
    if (!live) break;
    int barrier = 0, gone = 0, freed = 0;
    for (int w = 0; w < g->n; w += 64) {
      int here = 0, left = 0;
      for (int t = w; t < w + 64; t++) {
        here += g->at[t] == AT_WAVE;
        left += g->at[t] != AT_WAVE && g->at[t] != GONE;
        barrier += g->at[t] == AT_BARRIER;
        gone += g->at[t] == GONE;
      }
      if (here && !left) {
        for (int t = w; t < w + 64; t++)
          if (g->at[t] == AT_WAVE) g->at[t] = RUN;
        freed++;
      }
    }
    if (barrier && barrier + gone == g->n) {
      if (gone) bad("some items left before a barrier that others wait at", b);
      for (int t = 0; t < g->n; t++) g->at[t] = RUN;
      freed++;
    }
    if (!ran && !freed) bad("items wait for one another", b);
  }
}

// Workgroups of 1,024 items may wait for one another (grid-resident loops):
// up to 64 of them run side by side, a thread each.  Others run in turn.
static void run_grid(const std::function<void()> &f, unsigned grid, unsigned block)
{
  if (block > MAXT || block % 64) { fprintf(stderr, "emu: bad block %u\n", block); abort(); }
  gDim = {grid, 1, 1};
  bDim = {block, 1, 1};
  emu_wide += block == MAXT;
  if (block < MAXT || grid == 1 || grid > 64) {
    for (unsigned b = 0; b < grid; b++) run_block(b, block, f);
    return;
  }
  split_in = first_out = 0;
  std::vector<std::thread> ts;
  for (unsigned b = 0; b < grid; b++)
    ts.emplace_back([&f, b, block, grid]() {
      if (b == 0 && emu_split_wg > 0 && emu_split_wg < (int)grid)
        while (!split_in) std::this_thread::yield();
      run_block(b, block, f);
      if (b == 0) first_out = 1;
    });
  for (auto &t : ts) t.join();
}

static bool capturing = false;
static std::vector<std::function<void()>> *cap = nullptr;

void launch_fn(std::function<void()> f, unsigned grid, unsigned block)
{
  if (grid == 0) { fprintf(stderr, "emu: empty grid\n"); abort(); }
  if (capturing) {
    cap->push_back([f, grid, block]() { run_grid(f, grid, block); });
    return;
  }
  run_grid(f, grid, block);
}

// 100 MHz, as hipDeviceAttributeWallClockRate says below
unsigned long long clock()
{
  return 1000 + (unsigned long long)(std::chrono::steady_clock::now().time_since_epoch() /
                                     std::chrono::nanoseconds(10));
}
}  // namespace emu

struct ihipStream_t { int dummy; };
struct ihipEvent_t { double t; };
struct ihipGraph { std::vector<std::function<void()>> ops; };
struct hipGraphExec { std::vector<std::function<void()>> ops; };

static double now_ms()
{
  return std::chrono::duration<double, std::milli>(
             std::chrono::steady_clock::now().time_since_epoch()).count();
}

// Device allocations, so that copies can be checked the way the runtime
// checks them: a device-side range must lie inside one allocation.
static std::map<uintptr_t, size_t> g_dev;

static bool dev_range(const void *p, size_t n)
{
  const uintptr_t a = (uintptr_t)p;
  auto it = g_dev.upper_bound(a);
  if (it == g_dev.begin()) return false;
  --it;
  return a >= it->first && a + n <= it->first + it->second;
}

static hipError_t check_copy(void *d, const void *s, size_t n, hipMemcpyKind k)
{
  const bool dd = k == hipMemcpyHostToDevice || k == hipMemcpyDeviceToDevice;
  const bool sd = k == hipMemcpyDeviceToHost || k == hipMemcpyDeviceToDevice;
  if (!d || !s || (dd && !dev_range(d, n)) || (sd && !dev_range(s, n))) {
    fprintf(stderr, "emu: invalid copy d=%p s=%p n=%zu kind=%d\n", d, s, n, (int)k);
    return hipErrorInvalidValue;
  }
  return hipSuccess;
}

extern "C" {
hipError_t hipMalloc(void **p, size_t n)
{
  *p = malloc(n ? n : 1);
  memset(*p, 0x7f, n);
  g_dev[(uintptr_t)*p] = n ? n : 1;
  return hipSuccess;
}
hipError_t hipFree(void *p)
{
  if (p) g_dev.erase((uintptr_t)p);
  free(p);
  return hipSuccess;
}
// A __device__ variable is host memory here; the library's one such
// variable is its static scratch, registered as a device range of its size.
hipError_t hipGetSymbolAddress(void **p, const void *sym)
{
  *p = (void *)sym;
  g_dev[(uintptr_t)sym] = SFR_SCRATCH_BYTES;
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned int)
{
  *p = malloc(n ? n : 1);
  return hipSuccess;
}
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k)
{
  const hipError_t e = check_copy(d, s, n, k);
  if (e != hipSuccess) return e;
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t)
{
  if (emu::capturing) { fprintf(stderr, "emu: memcpy in capture\n"); abort(); }
  const hipError_t e = check_copy(d, s, n, k);
  if (e != hipSuccess) return e;
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t)
{
  if (emu::capturing) { fprintf(stderr, "emu: memset in capture\n"); abort(); }
  memset(d, v, n);
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int)
{
  const char *cus = getenv("SFR_EMU_CUS");
  *v = a == hipDeviceAttributeMultiprocessorCount ? (cus ? atoi(cus) : 4) : 100000;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned int) { *s = new ihipStream_t; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { delete s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = new ihipEvent_t{0}; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { e->t = now_ms(); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) { *ms = (float)(b->t - a->t); return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode)
{
  emu::capturing = true;
  emu::cap = new std::vector<std::function<void()>>();
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g)
{
  emu::capturing = false;
  *g = new ihipGraph{*emu::cap};
  delete emu::cap;
  emu::cap = nullptr;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *, char *, size_t)
{
  *e = new hipGraphExec{g->ops};
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { delete g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { delete e; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t)
{
  for (auto &f : e->ops) f();
  return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "hipSuccess" : "hipError"; }
hipError_t hipGetLastError(void) { return hipSuccess; }
}
