"""Grid-resident PCG and BiCGSTAB loops (device/resident.hpp) against the loops of kernels
they stand in for, on the same resident matrix (an explicit rows-per-thread
choice keeps the loop of kernels), at the edges of their launch shapes: one
workgroup and its 1,024-row passes, the first sizes of several workgroups,
ragged last workgroups, each number of passes, and every way the rows are
read (16-bit offsets, escapes, 32-bit columns, an odd slot count).

Bars.  Both sides run the same recurrences on the same products; only the
order of the dot products' sums differs, a relative 1e-16 n^(1/2) each that
the solve carries along.  After a fixed 40 iterations that leaves x within
1e-10; converged solves agree as their stop tests do (tol 1e-10, side s:
s tol).  In mixed precision the sums enter through FP32 scalars, so the
fixed-count bar is 1e-5.  Iteration counts agree to within 2."""
import numpy as np
import pytest

import oracle
import sfr3d_amd as S
from sfr3d_amd import systems

pytestmark = pytest.mark.gpu

BOXES = [(2, 2, 2), (31, 33, 1), (32, 32, 1), (25, 41, 1), (16, 16, 16), (17, 241, 1),
         (13, 19, 33), (51, 51, 51), (64, 64, 33), (71, 63, 59), (81, 80, 81), (101, 100, 99)]


def rel(x, y):
    return np.linalg.norm(x - y) / np.linalg.norm(y)


def counted(ctx, f):
    """f(), and what it added to the context's (resident solves, stalls)."""
    a = ctx.resident_info()
    out = f()
    b = ctx.resident_info()
    return out, (b[0] - a[0], b[1] - a[1])


def both(ctx, system, b, tol, maxit, prec, x0=None, solver=S.PCG):
    """(x, stats) of the resident loop and of the loop of kernels, and that each
    is the one that ran."""
    out = []
    for tuned in (False, True):
        A = ctx.matrix(system)
        if tuned:
            A.tune(A.info()["rows_per_thread"])
        db, dx = ctx.array(b), ctx.array(np.zeros(system.neq) if x0 is None else x0)
        st, ran = counted(ctx, lambda: ctx.solve_device(A, solver, tol, maxit, db, dx,
                                                        newX=x0 is None, precision=prec))
        assert ran == (0 if tuned else 1, 0)
        out.append((dx.get(), st))
        A.destroy(); db.free(); dx.free()
    return out


@pytest.mark.parametrize("box", BOXES, ids=["x".join(map(str, b)) for b in BOXES])
@pytest.mark.parametrize("prec", [S.PREC_FP64, S.PREC_MIXED], ids=["fp64", "mixed"])
def test_matches_the_loop_of_kernels(ctx, box, prec):
    B = systems.poisson3d(box[0], ny=box[1], nz=box[2], seed=3, storage=S.CSRD,
                          reorder=box[0] % 2 == 0)
    n = B.system.neq
    print(f"resident {box} n={n} prec={prec}", flush=True)
    (x, st), (y, sk) = both(ctx, B.system, B.b[:n], 1e-10, 100000, prec)
    assert st["status"] == sk["status"] == 0 and abs(st["iters"] - sk["iters"]) <= 2
    assert rel(x, y) < (max(box) * 1e-10 if prec == S.PREC_FP64 else 1e-6)
    # a fixed count, from a given guess
    x0 = np.random.default_rng(1).uniform(-1.0, 1.0, n)
    (x, st), (y, sk) = both(ctx, B.system, B.b[:n], 0.0, 40, prec, x0)
    assert st["status"] == sk["status"] and st["iters"] == sk["iters"]
    if n > 200:                              # smaller ones are solved to rounding by then
        assert rel(x, y) < (1e-10 if prec == S.PREC_FP64 else 1e-5)


def chain(n, hops):
    """Symmetric CSRD system whose row i couples to i +- h for h in hops,
    periodically for the hops that wrap (long-range entries)."""
    rows = [set() for _ in range(n)]
    for i in range(n):
        for h in hops:
            j = (i + h) % n
            if j != i:
                rows[max(i, j)].add(min(i, j))
    ia = np.zeros(n + 1, np.int32)
    np.cumsum([len(r) for r in rows], out=ia[1:])
    ja = np.array([j for r in rows for j in sorted(r)], np.int32)
    rng = np.random.default_rng(n)
    al = -rng.uniform(0.1, 1.0, len(ja))
    i = np.repeat(np.arange(n), np.diff(ia))
    ad = np.full(n, 1e-2)
    np.add.at(ad, i, -al)
    np.add.at(ad, ja, -al)
    return S.System(n, len(ja), ia, ja, al, ad, S.CSRD, False), rng.uniform(-1.0, 1.0, n)


@pytest.mark.parametrize("n,hops", [
    (1500, (1,)), (5000, (1, 40)), (40000, (1, 7)), (40000, (1, 9, 300)), (9000, (1, 2, 3, 4)),
    (150000, (1, 40, 900)), (300000, (1, 40, 900)), (600000, (1, 900)),
], ids=lambda v: str(v).replace(" ", ""))
@pytest.mark.parametrize("prec", [S.PREC_FP64, S.PREC_MIXED], ids=["fp64", "mixed"])
def test_row_operators(ctx, n, hops, prec):
    """Other slot counts (2, 4, 6, 8) and wrapped hops: beyond 32,767 rows
    their offsets leave 16 bits (escapes)."""
    system, b = chain(n, hops)
    print(f"resident chain n={n} hops={hops} prec={prec}", flush=True)
    (x, st), (y, sk) = both(ctx, system, b, 0.0, 40, prec)
    assert st["iters"] == sk["iters"]
    assert rel(x, y) < (1e-10 if prec == S.PREC_FP64 else 1e-5)


@pytest.mark.parametrize("n", [12, 40])
def test_zero_rhs_and_exact_guess(ctx, n):
    B = systems.poisson3d(n, seed=2)
    for b, x0 in ((np.zeros(B.system.neq), None), (np.zeros(B.system.neq), np.zeros(B.system.neq))):
        (x, st), (y, sk) = both(ctx, B.system, b, 1e-8, 100, S.PREC_FP64, x0)
        assert st["status"] == sk["status"] == 0 and st["iters"] == sk["iters"] == 0
        assert np.array_equal(x, np.zeros_like(x)) and np.array_equal(x, y)


def test_long_solve_takes_several_launches(ctx):
    """More iterations than one launch runs (1,024), and the maxit status."""
    B = systems.poisson2d(160, 90, storage=S.ELLPACK)
    n = B.system.neq
    (x, st), (y, sk) = both(ctx, B.system, B.b[:n], 1e-13, 100000, S.PREC_FP64)
    assert st["status"] == sk["status"] == 0 and sk["iters"] > 1100
    assert abs(st["iters"] - sk["iters"]) <= 2 and rel(x, y) < 1e-9
    (x, st), (y, sk) = both(ctx, B.system, B.b[:n], 0.0, 1025, S.PREC_FP64)
    assert st["status"] == sk["status"] == S._lib.MAXIT and st["iters"] == sk["iters"] == 1025


@pytest.mark.parametrize("prec", [S.PREC_FP64, S.PREC_MIXED], ids=["fp64", "mixed"])
def test_falls_back_when_a_workgroup_has_to_wait(ctx, prec):
    """No patience at all: the first sum that is not complete when polled
    stalls the launch, and the call answers through the loop of kernels."""
    B = systems.poisson3d(48, seed=4)
    db, dx = ctx.array(B.b), ctx.empty(B.system.neq)
    A = ctx.matrix(B.system)
    try:
        ctx.set_option("resident_wait", 0)
        st, ran = counted(ctx, lambda: ctx.solve_device(A, S.PCG, 1e-9, 10000, db, dx,
                                                        precision=prec))
    finally:
        ctx.set_option("resident_wait", 2)
    assert ran == (0, 1)
    xo, so = oracle.pcg(B.system, B.b, 1e-9, 10000)
    assert st["status"] == 0 and rel(dx.get(), xo) < 1e-6
    with pytest.raises(S.SolverError):
        ctx.set_option("resident_wait", 100)
    A.destroy(); db.free(); dx.free()


@pytest.mark.parametrize("n", [2, 10, 11, 16, 45, 51, 64, 80, 82, 101])
def test_bicgstab_matches_the_loop_of_kernels(ctx, n):
    """Momentum systems, a fixed 4 iterations from a guess (bar: the sums'
    rounding, relative to the guess where the solution is smaller: 2^3's
    right-hand side cancels to 1e-17) and to tol 1e-10."""
    M = systems.momentum3d(n, storage=S.CSRC if n % 2 else S.CSRD)
    print(f"resident BiCGSTAB {n}^3", flush=True)
    x0 = np.random.default_rng(2).uniform(-1.0, 1.0, M.system.neq)
    (x, st), (y, sk) = both(ctx, M.system, M.b, 0.0, 4, S.PREC_FP64, x0, S.PBICGSTAB)
    assert st["iters"] == sk["iters"] == 4 and st["status"] == sk["status"]
    assert np.linalg.norm(x - y) < 1e-12 * max(np.linalg.norm(y), np.linalg.norm(x0))
    (x, st), (y, sk) = both(ctx, M.system, M.b, 1e-10, 1000, S.PREC_FP64, None, S.PBICGSTAB)
    assert st["status"] == sk["status"] == 0 and abs(st["iters"] - sk["iters"]) <= 1
    assert rel(x, y) < 4e-10


@pytest.mark.parametrize("n,hops", [(1500, (1,)), (40000, (1, 7)), (9000, (1, 2, 3, 4)),
                                    (150000, (1, 40, 900)), (600000, (1, 900))],
                         ids=lambda v: str(v).replace(" ", ""))
def test_bicgstab_row_operators(ctx, n, hops):
    system, b = chain(n, hops)
    (x, st), (y, sk) = both(ctx, system, b, 0.0, 6, S.PREC_FP64, None, S.PBICGSTAB)
    assert st["iters"] == sk["iters"] == 6 and rel(x, y) < 1e-10


@pytest.mark.parametrize("wait", [2, 0, -1], ids=["resident", "stalled", "kernels"])
def test_batches_by_every_route(ctx, wait):
    """u/v/w and species batches through the resident loop, through its
    fallback and through the batched kernels: the same answers as single
    solves by the oracle."""
    M = systems.momentum3d(24)
    n = M.system.neq
    ads = [M.system.ad[:n] * (1.0 + 0.05 * c) for c in range(3)]
    sysm, sp = systems.species3d(20, 5, seed=3)
    try:
        ctx.set_option("resident_wait", wait)
        before = ctx.resident_info()
        xs, st = ctx.solve_shared(M.system, S.PBICGSTAB, 1e-10, 1000, list(M.extra["b_all"]), ads)
        ys, sy = ctx.solve_batched(sysm, S.PBICGSTAB, 1e-10, 1000, [a for a, _, _ in sp],
                                   [d for _, d, _ in sp], [b for _, _, b in sp])
        after = ctx.resident_info()
    finally:
        ctx.set_option("resident_wait", 2)
    assert (after[0] - before[0], after[1] - before[1]) == {2: (8, 0), 0: (0, 2), -1: (0, 0)}[wait]
    s0 = M.system
    for c in range(3):
        s = S.System(n, s0.nad, s0.ia, s0.ja, s0.al, ads[c], s0.storage, s0.unsym)
        xo, so = oracle.pbicgstab(s, M.extra["b_all"][c], 1e-10, 1000)
        assert st[c]["status"] == 0 and rel(xs[c], xo) < 1e-9
        assert wait == 0 or abs(st[c]["iters"] - so["iters"]) <= 1
    for c, (al, ad, b) in enumerate(sp):
        s = S.System(sysm.neq, sysm.nad, sysm.ia, sysm.ja, al, ad, sysm.storage, sysm.unsym)
        xo, so = oracle.pbicgstab(s, b, 1e-10, 1000)
        assert sy[c]["status"] == 0 and rel(ys[c], xo) < 1e-9
        assert wait == 0 or abs(sy[c]["iters"] - so["iters"]) <= 1


@pytest.mark.parametrize("sides", [[2], [10, 11], [16, 3, 40, 7, 25], [12] * 40 + [39],
                                   [64, 50, 33, 20, 9], [80, 60, 45, 30], [101, 70, 48]],
                         ids=lambda v: f"{len(v)}x{v[0]}")
def test_uneven_batch_matches_the_batch_kernels(ctx, sides):
    """Each number of passes, systems of one and of many workgroups; every
    system meets its own test by the resident launch, by its fallback and by
    the batch's kernels, with solutions that agree (mixed precision to
    tol 1e-9: 1e-6 apart at most)."""
    built = systems.uneven_batch(len(sides), seed=3, kmin=1e-2, sides=np.array(sides))
    got = {}
    for wait in (2, 0, -1):
        print(f"uneven {sides[:5]} wait={wait}", flush=True)
        try:
            ctx.set_option("resident_wait", wait)
            Bt = ctx.batch([B.system for B in built], tune=False)
            got[wait], ran = counted(ctx, lambda: Bt.solve([B.b[:B.system.neq] for B in built],
                                                           1e-9, 20000))
            Bt.destroy()
            waits = wait == 0 and max(sides) > 10        # a system of several workgroups
            assert ran == ((0, 0) if wait < 0 else (0, 1) if waits else (len(sides), 0))
        finally:
            ctx.set_option("resident_wait", 2)
    for k, B in enumerate(built):
        for wait in (2, 0, -1):
            st = got[wait][1][k]
            assert st["status"] == 0 and st["norm_r_m"] < st["conv"] * (1 + 1e-12)
            assert rel(got[wait][0][k], got[-1][0][k]) < 1e-6
        assert abs(got[2][1][k]["iters"] - got[-1][1][k]["iters"]) <= max(
            3, 0.05 * got[-1][1][k]["iters"])


@pytest.mark.parametrize("wait", [0, 2e-6, 1e-5])
def test_short_waits_leave_no_part_unsolved(ctx, wait):
    """Waits of a sum's own length, at which workgroups give up on any sum, the
    last one included: whatever answers OK has all of x."""
    B, M = systems.poisson3d(24, seed=4), systems.momentum3d(40)
    n = M.system.neq
    ads = [M.system.ad[:n] * (1.0 + 0.05 * c) for c in range(3)]
    sysm, sp = systems.species3d(24, 4, seed=3)
    want = {"pcg": [oracle.pcg(B.system, B.b, 1e-9, 10000)[0]],
            "bicg": [oracle.pbicgstab(M.system, M.b, 1e-9, 1000)[0]], "uvw": [], "species": []}
    for c in range(3):
        s = S.System(n, M.system.nad, M.system.ia, M.system.ja, M.system.al, ads[c],
                     M.system.storage, M.system.unsym)
        want["uvw"].append(oracle.pbicgstab(s, M.extra["b_all"][c], 1e-9, 1000)[0])
    for al, ad, b in sp:
        s = S.System(sysm.neq, sysm.nad, sysm.ia, sysm.ja, al, ad, sysm.storage, sysm.unsym)
        want["species"].append(oracle.pbicgstab(s, b, 1e-9, 1000)[0])

    def one(A, b, solver):
        db, dx = ctx.array(b), ctx.empty(len(b))
        st = ctx.solve_device(A, solver, 1e-9, 10000, db, dx)
        x = dx.get()
        db.free(); dx.free()
        return [x], [st]
    AB, AM = ctx.matrix(B.system), ctx.matrix(M.system)
    calls = {"pcg": lambda: one(AB, B.b, S.PCG), "bicg": lambda: one(AM, M.b, S.PBICGSTAB),
             "uvw": lambda: ctx.solve_shared(M.system, S.PBICGSTAB, 1e-9, 1000,
                                             list(M.extra["b_all"]), ads),
             "species": lambda: ctx.solve_batched(sysm, S.PBICGSTAB, 1e-9, 1000,
                                                  [a for a, _, _ in sp], [d for _, d, _ in sp],
                                                  [b for _, _, b in sp])}
    try:
        for _ in range(4):
            for name, call in calls.items():
                ctx.set_option("resident_wait", wait)
                (xs, st), ran = counted(ctx, call)
                print(f"wait {wait} {name} {ran}", flush=True)
                for x, s, xo in zip(xs, st, want[name]):
                    assert s["status"] == 0 and rel(x, xo) < 1e-6
    finally:
        ctx.set_option("resident_wait", 2)
    AB.destroy(); AM.destroy()


def shuffled(B, block, seed=0):
    """The rows of a symmetric CSRD system in random order inside blocks."""
    s, n = B.system, B.system.neq
    p, rng = np.arange(n), np.random.default_rng(seed)
    for a in range(0, n, block):
        p[a:a + block] = a + rng.permutation(min(block, n - a))
    i = p[np.repeat(np.arange(n), np.diff(s.ia[:n + 1]))]
    j = p[s.ja[:s.ia[n]]]
    hi, lo = np.maximum(i, j), np.minimum(i, j)
    o = np.lexsort((lo, hi))
    ia = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(hi, minlength=n), out=ia[1:])
    ad, b = np.empty(n), np.empty(n)
    ad[p], b[p] = s.ad[:n], B.b[:n]
    return S.System(n, s.nad, ia, lo[o].astype(np.int32), s.al[:len(o)][o], ad, S.CSRD, False), b


@pytest.mark.parametrize("n,block,resident", [(51, 512, True), (51, 2048, True), (51, 1 << 20, False),
                                              (32, 1 << 20, True)])
def test_scattered_rows_keep_the_loop_of_kernels(ctx, n, block, resident):
    """FP64 loops whose gathers share no lines were slower resident (101^3 in
    random order: half the speed); the mixed loop was not."""
    system, b = shuffled(systems.poisson3d(n, seed=3, storage=S.CSRD, reorder=False), block)
    A, db, dx = ctx.matrix(system), ctx.array(b), ctx.empty(system.neq)
    for solver, prec in ((S.PCG, S.PREC_FP64), (S.PBICGSTAB, S.PREC_FP64), (S.PCG, S.PREC_MIXED)):
        before = ctx.resident_info()[0]
        ctx.solve_device(A, solver, 0.0, 3, db, dx, precision=prec)
        went = ctx.resident_info()[0] - before
        assert went == (resident or prec == S.PREC_MIXED)
    A.destroy(); db.free(); dx.free()


def test_contexts_side_by_side(ctx):
    """Two threads' resident solves share the device: each waits for its
    turn's workgroups, both answer as alone."""
    import threading
    B = systems.poisson3d(72, seed=6)
    db = ctx.array(B.b)
    A, dx = ctx.matrix(B.system), ctx.empty(B.system.neq)
    ctx.solve_device(A, S.PCG, 1e-8, 10000, db, dx)
    alone = dx.get()
    got = [None, None]

    def work(k):
        with S.Context(0) as c:
            M, b, x = c.matrix(B.system), c.array(B.b), c.empty(B.system.neq)
            for _ in range(5):
                c.solve_device(M, S.PCG, 1e-8, 10000, b, x)
            got[k] = x.get()
            M.destroy(); b.free(); x.free()
    ts = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert np.array_equal(got[0], alone) and np.array_equal(got[1], alone)
    A.destroy(); db.free(); dx.free()
