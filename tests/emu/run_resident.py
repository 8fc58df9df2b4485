"""TEST INFRASTRUCTURE -- runs the grid-resident loops of the emulated library
(argv[1]) in a process of its own, on an emulated device of 256 CUs, and
compares them with the loops of kernels on the same matrices.  argv[2] names
the group of checks.  Prints PASS/FAIL lines and exits non-zero on any
failure."""
import ctypes as C
import os
import sys
import threading
import time

os.environ["SFR_EMU_CUS"] = "256"
ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path.insert(0, ROOT)
EMU = sys.argv[1]
_cdll = C.CDLL
C.CDLL = lambda path, *a, **k: _cdll(EMU if str(path).endswith("libsfr3d.so") else path, *a, **k)
import numpy as np  # noqa: E402
import sfr3d_amd as S  # noqa: E402
from sfr3d_amd import systems  # noqa: E402
from sfr3d_amd._lib import lib  # noqa: E402
from tests.test_gpu_resident import chain, rel  # noqa: E402
C.CDLL = _cdll

fails = 0


def check(tag, ok):
    global fails
    print(("PASS " if ok else "FAIL ") + tag, flush=True)
    fails += not ok


def emu(name, kind=C.c_int):
    return kind.in_dll(lib, "emu_" + name)


def counted(ctx, f):
    """f(), and what it added to the context's (resident solves, stalls)."""
    a = ctx.resident_info()
    out = f()
    b = ctx.resident_info()
    return out, (b[0] - a[0], b[1] - a[1])


def solve(ctx, A, b, solver, tol, maxit, prec=S.PREC_FP64, x0=None):
    db, dx = ctx.array(b), ctx.array(np.zeros(len(b)) if x0 is None else x0)
    st = ctx.solve_device(A, solver, tol, maxit, db, dx, newX=x0 is None, precision=prec)
    x = dx.get()
    db.free()
    dx.free()
    return x, st


def by(ctx, wait, f):
    ctx.set_option("resident_wait", wait)
    try:
        return counted(ctx, f)
    finally:
        ctx.set_option("resident_wait", 2)


def routes():
    """Every resident kernel at one and at several workgroups, odd row counts,
    each way the rows are read; the emulated loops add in the same order
    on every run, so a repeated solve has the same bits."""
    ctx = S.Context(0)
    boxes = [((1, 1, 1), S.CSRD), ((7, 5, 3), S.CSRC), ((10, 10, 10), S.ELLPACK),
             ((11, 11, 11), S.CSRD), ((17, 17, 17), S.ELLPACK)]
    cases = []
    for box, st in boxes:
        B = systems.poisson3d(box[0], ny=box[1], nz=box[2], seed=3, storage=st)
        cases.append(("x".join(map(str, box)), B.system, B.b[:B.system.neq]))
    B = systems.poisson2d(33, 31, storage=S.ELLPACK)
    cases.append(("33x31", B.system, B.b[:B.system.neq]))
    for n, hops in ((1025, (1,)), (1500, (1, 2, 3, 4)), (33001, (1, 7, 90))):
        cases.append((f"chain {n} {hops}", *chain(n, hops)))
    for tag, system, b in cases:
        A = ctx.matrix(system)
        n = system.neq
        its = 2 if n > 10000 else 6
        x0 = np.random.default_rng(1).uniform(-1.0, 1.0, n)
        for name, solver, prec, bar in (("pcg", S.PCG, 0, 1e-11), ("mixed", S.PCG, 1, 1e-5),
                                        ("bicg", S.PBICGSTAB, 0, 1e-10)):
            k = its if solver == S.PCG else 2
            f = lambda: solve(ctx, A, b, solver, 0.0, k, prec, x0)  # noqa: E731
            (x, sx), nx = by(ctx, 2, f)
            (x2, _), _ = by(ctx, 2, f)
            (y, sy), ny = by(ctx, -1, f)
            check(f"{tag} {name} it {sx['iters']}/{sy['iters']} rel {rel(x, y):.1e} {nx} {ny}",
                  sx["status"] == sy["status"] and sx["iters"] == sy["iters"]
                  and (n < 200 or rel(x, y) < bar) and np.array_equal(x, x2)
                  and nx == (1, 0) and ny == (0, 0))
        A.destroy()
    # batches: u/v/w, species (values of their own), uneven
    M = systems.momentum3d(11)
    ads = [M.system.ad[:M.system.neq] * (1.0 + 0.05 * c) for c in range(3)]
    sysm, sp = systems.species3d(6, 5, seed=3)
    built = systems.uneven_batch(3, seed=3, kmin=1e-2, sides=np.array([4, 11, 6]))
    Bt = ctx.batch([B.system for B in built], tune=False)
    for name, nsys, f in (
            ("uvw", 3, lambda: ctx.solve_shared(M.system, S.PBICGSTAB, 1e-6, 1000,
                                                list(M.extra["b_all"]), ads)),
            ("species", 5, lambda: ctx.solve_batched(sysm, S.PBICGSTAB, 1e-6, 1000,
                                                     [a for a, _, _ in sp], [d for _, d, _ in sp],
                                                     [b for _, _, b in sp])),
            ("uneven", 3, lambda: Bt.solve([B.b[:B.system.neq] for B in built], 1e-3, 1000))):
        (xs, st), n = by(ctx, 2, f)
        (ys, su), m = by(ctx, -1, f)
        worst = max(rel(x, y) for x, y in zip(xs, ys))
        check(f"{name} it {[v['iters'] for v in st]} {[v['iters'] for v in su]} rel {worst:.1e} {n} {m}",
              all(v["status"] == 0 for v in st + su) and worst < (1e-2 if name == "uneven" else 4e-6)
              and n == (nsys, 0) and m == (0, 0))
    Bt.destroy()
    ctx.close()


def late():
    """Workgroup 3 gives up on the last sum of a solve, which the others see
    complete: the call may answer OK only with all of x solved."""
    ctx = S.Context(0)
    B = systems.poisson3d(17, seed=3)
    M = systems.momentum3d(17)
    n = M.system.neq
    ads = [M.system.ad[:n] * (1.0 + 0.05 * c) for c in range(3)]
    sysm, sp = systems.species3d(17, 3, seed=3)
    AB, AM = ctx.matrix(B.system), ctx.matrix(M.system)
    dn = [ctx.array(B.b[:B.system.neq]), ctx.empty(B.system.neq)]

    def noalloc():
        st = S._lib.SfrStats()
        rc = lib.sfr_solve_device_noalloc(ctx.h, AB.h, S.PCG, 1e-3, 1000, dn[0].ptr, dn[1].ptr,
                                          1, C.byref(st))
        assert rc == st.status
        return [dn[1].get()], [st.as_dict()]

    def one(A, b, solver):
        x, st = solve(ctx, A, b, solver, 1e-3, 1000)
        return [x], [st]
    for name, sums, f in (
            ("pcg", 2, lambda: one(AB, B.b[:B.system.neq], S.PCG)),
            ("noalloc", 2, noalloc),
            ("bicg", 3, lambda: one(AM, M.b[:n], S.PBICGSTAB)),
            ("uvw", 3, lambda: ctx.solve_shared(M.system, S.PBICGSTAB, 1e-3, 1000,
                                                list(M.extra["b_all"]), ads)),
            ("species", 3, lambda: ctx.solve_batched(sysm, S.PBICGSTAB, 1e-3, 1000,
                                                     [a for a, _, _ in sp], [d for _, d, _ in sp],
                                                     [b for _, _, b in sp]))):
        ys, su = f()
        k = max(v["iters"] for v in su)
        gave_up = 0
        # a BiCGSTAB solve ends at the half-step test or at the full one
        for last in range(sums * k - (sums == 3), sums * k + 1):
            emu("late_wg").value, emu("late_sum", C.c_uint).value = 3, last
            (xs, st), (_, stalls) = by(ctx, 1.5, f)
            emu("late_wg").value = -1
            gave_up += stalls
            worst = max(rel(x, y) for x, y in zip(xs, ys))
            check(f"late {name} sum {last} status {[v['status'] for v in st]} rel {worst:.1e}",
                  all(v["status"] == 0 for v in st) and worst < 2e-2)
        check(f"late {name} gave up {gave_up}", gave_up >= 1)
    ctx.close()


def split():
    """Half of workgroup 2's items enter a resident kernel after workgroup 0,
    which had no patience, has given up and left: all of them or none may
    go on (the emulation ends the process at a barrier that some have left)."""
    ctx = S.Context(0)
    B = systems.poisson3d(17, seed=3)
    M = systems.momentum3d(17)
    AB, AM = ctx.matrix(B.system), ctx.matrix(M.system)
    for name, A, b, solver, prec in (("pcg", AB, B.b, S.PCG, S.PREC_FP64),
                                     ("mixed", AB, B.b, S.PCG, S.PREC_MIXED),
                                     ("bicg", AM, M.b, S.PBICGSTAB, S.PREC_FP64)):
        f = lambda: solve(ctx, A, b[:A.system.neq], solver, 1e-3, 1000, prec)  # noqa: E731
        (y, _), _ = by(ctx, -1, f)
        emu("split_wg").value = 2
        (x, st), n = by(ctx, 0, f)
        emu("split_wg").value = -1
        check(f"split {name} status {st['status']} rel {rel(x, y):.1e} {n}",
              st["status"] == 0 and rel(x, y) < 2e-2 and n == (0, 1))
    ctx.close()


def away():
    """What a stall costs: one wait for a whole batch, and none for the
    context's next solves until 64 such waits have passed."""
    ctx = S.Context(0)
    M = systems.momentum3d(17)
    n = M.system.neq
    ads = [M.system.ad[:n] * (1.0 + 0.05 * c) for c in range(3)]
    sysm, sp = systems.species3d(17, 4, seed=3)
    built = systems.uneven_batch(2, seed=3, kmin=1e-2, sides=np.array([17, 4]))
    Bt = ctx.batch([B.system for B in built], tune=False)
    small = systems.poisson3d(6, seed=3)
    A = ctx.matrix(small.system)

    def alone():
        return counted(ctx, lambda: solve(ctx, A, small.b, S.PCG, 1e-3, 1000))[1]
    def stalled(wait, f):
        ctx.set_option("resident_wait", wait)
        emu("late_wg").value, emu("late_sum", C.c_uint).value = 3, 1
        out = counted(ctx, f)
        emu("late_wg").value = -1
        return out
    for name, f in (
            ("uvw", lambda: ctx.solve_shared(M.system, S.PBICGSTAB, 1e-3, 1000,
                                             list(M.extra["b_all"]), ads)),
            ("uneven", lambda: Bt.solve([B.b[:B.system.neq] for B in built], 1e-2, 1000)),
            ("species", lambda: ctx.solve_batched(sysm, S.PBICGSTAB, 1e-3, 1000,
                                                  [a for a, _, _ in sp], [d for _, d, _ in sp],
                                                  [b for _, _, b in sp]))):
        (ys, _), _ = by(ctx, -1, f)
        (xs, st), k = stalled(1.0, f)
        worst = max(rel(x, y) for x, y in zip(xs, ys))
        check(f"away {name} status {[v['status'] for v in st]} rel {worst:.1e} {k}",
              all(v["status"] == 0 for v in st) and worst < 2e-2 and k == (0, 1))
        k = alone()
        check(f"away {name} next solve {k}", k == (0, 0))
    B = systems.poisson3d(17, seed=3)
    A17, wait = ctx.matrix(B.system), 0.1
    t0 = time.monotonic()
    _, k = stalled(wait, lambda: solve(ctx, A17, B.b, S.PCG, 0.0, 2))
    t1 = time.monotonic()
    while alone() == (0, 0) and time.monotonic() - t0 < 200 * wait:
        time.sleep(0.1)
    t2 = time.monotonic()
    check(f"away {t2 - t1:.1f} to {t2 - t0:.1f} s {k}",
          k == (0, 1) and t2 - t1 < 150 * wait and t2 - t0 > 64 * wait)
    stalled(1.0, lambda: solve(ctx, A17, B.b, S.PCG, 0.0, 2))
    ctx.set_option("resident_wait", 1.0)    # the option starts afresh
    k = alone()
    check(f"away no more {k}", k == (1, 0))
    ctx.close()


def slices():
    """A solve's launches are of at most 16 iterations here (RES_LIMIT), batches'
    too: the CUs are given back in between, and the solve goes on as if they
    had not been."""
    ctx = S.Context(0)
    system, b = chain(1500, (1,))
    rng = np.random.default_rng(5)
    bs = [b] + [rng.uniform(-1.0, 1.0, system.neq) for _ in range(2)]
    ads = [system.ad * (1.0 + 1e-4 * c) for c in range(3)]
    built = systems.uneven_batch(3, seed=3, kmin=1e-2, sides=np.array([4, 11, 8]))
    Bt = ctx.batch([B.system for B in built], tune=False)
    A = ctx.matrix(system)
    for name, its, launches, bar, f in (
            ("pcg", 40, 3, 1e-11, lambda: [[v] for v in solve(ctx, A, b, S.PCG, 0.0, 40)]),
            ("bicg", 20, 2, 1e-9, lambda: [[v] for v in solve(ctx, A, b, S.PBICGSTAB, 0.0, 20)]),
            ("uvw", 20, 6, 1e-9, lambda: ctx.solve_shared(system, S.PBICGSTAB, 0.0, 20, bs, ads)),
            ("species", 20, 6, 1e-9, lambda: ctx.solve_batched(
                system, S.PBICGSTAB, 0.0, 20, [system.al * (1.0 - 1e-4 * c) for c in range(3)], ads, bs)),
            ("uneven", 40, None, 1e-2, lambda: Bt.solve([B.b[:B.system.neq] for B in built], 1e-3, 1000))):
        (ys, su), _ = by(ctx, -1, f)
        emu("wide").value = 0
        (xs, st), n = by(ctx, 2, f)
        w = emu("wide").value
        worst = max(rel(x, y) for x, y in zip(xs, ys))
        longest = max(v["iters"] for v in st)
        check(f"slices {name} it {[v['iters'] for v in st]} {[v['iters'] for v in su]} "
              f"launches {w} rel {worst:.1e} {n}",
              worst < bar and n == (len(xs), 0) and [v["status"] for v in st] == [v["status"] for v in su]
              and (w == launches and longest == its if launches else 2 <= w <= longest / 16 + 1))
    Bt.destroy()
    ctx.close()


def count():
    """Launches that together want more CUs of one XCD than it has wait for one
    another in the host's count: workgroup i goes to XCD i % 8, so 130 and 126
    put 17 and 16 on the first of them."""
    def enters(wgs):
        t = threading.Thread(target=lib.sfr_res_enter, args=(0, 256, wgs), daemon=True)
        t.start()
        t.join(0.5)
        return t
    for first, second, together in ((130, 126, False), (129, 127, False), (128, 128, True),
                                    (200, 56, True), (248, 1, True), (256, 1, False)):
        assert not enters(first).is_alive()
        t = enters(second)
        check(f"count {first} and {second} together {not t.is_alive()}",
              t.is_alive() != together)
        lib.sfr_res_leave(0, first)
        t.join(5)
        check(f"count {second} after {first}", not t.is_alive())
        lib.sfr_res_leave(0, second)
    t = enters(256)
    check("count given back", not t.is_alive())


{"routes": routes, "late": late, "split": split, "away": away,
 "slices": slices, "count": count}[sys.argv[2]]()
print("RESIDENT OK" if not fails else f"RESIDENT FAILED {fails}", flush=True)
sys.exit(1 if fails else 0)
