"""The work that programs have the solver do, as cases that can be timed and
compared: Jacobi-PCG on pressure-type systems from a small 2-D cavity to the
128^3 Poisson system (FP64 and mixed precision), BiCGSTAB on momentum systems
(one component, the u/v/w batch, a species batch on host arrays), GMRES, the
adjoint of a diffusion solve, an uneven batch of independent systems, and the
SIMPLE cell loops with the device assembly behind them.

A case is a dict of plain values; prepare() makes what a program holds before
the call (matrix, vectors, plan), run() is one call through the public entry
points, exact() the same outputs in 64 bits from plain torch.
"""
import ctypes as C
import functools
import math

import numpy as np
import torch

import sfr3d_amd as S
from sfr3d_amd import structure, systems
from sfr3d_amd._lib import SfrStats, lib

STORAGE = {"CSRD": S.CSRD, "CSRC": S.CSRC, "ELLPACK": S.ELLPACK}
MAXIT = 100000


def listed():
    return [
        # the pressure correction of a small 2-D cavity: a few rows, bound by
        # what one iteration costs, not by what it moves
        dict(name="pcg_cavity_32", kind="pcg2d", nx=32, ny=32, storage="CSRD", tol=1e-11),
        # the 2-D cavity of the tests and benchmark configurations, 16,383 rows
        dict(name="pcg_cavity_128", kind="pcg2d", nx=128, ny=128, storage="ELLPACK", tol=1e-11),
        # a box of odd sides with a pinned cell, natural order, the storage and
        # tolerance of the shipped solver decks (an everyday 3-D mesh)
        dict(name="pcg_box_odd", kind="pcg3d", nx=61, ny=47, nz=38, storage="CSRC",
             reorder=False, pinned=True, prec="fp64", tol=1e-11),
        # the benchmark's system, FP64: the largest call
        dict(name="pcg_128", kind="pcg3d", nx=128, ny=128, nz=128, storage="ELLPACK",
             reorder=True, pinned=False, prec="fp64", tol=1e-8),
        # the benchmark's headline: the same system in mixed precision
        dict(name="mixed_128", kind="pcg3d", nx=128, ny=128, nz=128, storage="ELLPACK",
             reorder=True, pinned=False, prec="mixed", tol=1e-8),
        # one momentum component, unsymmetric CSRC as in the shipped decks
        dict(name="bicg_45", kind="bicg", n=45, storage="CSRC", tol=1e-11),
        # u, v and w of a SIMPLE step on one pattern, vectors on the device
        dict(name="uvw_96", kind="uvw", n=96, storage="CSRD", tol=1e-8),
        # ten transported species, host arrays in and out, uploads included
        dict(name="species_48", kind="species", n=48, count=10, storage="CSRD", tol=1e-8),
        # GMRES(15) on a momentum component
        dict(name="gmres_64", kind="gmres", n=64, storage="CSRD", tol=1e-10),
        # a differentiable solve: forward PCG, adjoint PCG, value gradients
        dict(name="adjoint_64", kind="adjoint", nx=64, ny=64, nz=64, storage="ELLPACK",
             tol=1e-10),
        # many independent systems of uneven sizes in one batch
        dict(name="uneven_48", kind="uneven", count=48, smin=12, smax=40, tol=1e-8),
        # one SIMPLE outer iteration's coefficients: momentum and pressure cell
        # loops and both matrices assembled on the device
        dict(name="simple_cells", kind="cells", nx=80, ny=64, nz=56),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pcg2d", "pcg3d", "pcg3d", "mixed", "bicg", "uvw", "species", "gmres",
                       "adjoint", "uneven", "cells"])
    if kind == "pcg2d":
        return dict(kind=kind, nx=_log(rng, 24, 200), ny=_log(rng, 24, 200),
                    storage=rng.choice(["CSRD", "CSRC", "ELLPACK"]), tol=1e-11)
    if kind in ("pcg3d", "mixed"):
        side = _log(rng, 8, 110)
        box = [max(5, round(side * rng.uniform(0.7, 1.3))) for _ in range(3)]
        return dict(kind="pcg3d", nx=box[0], ny=box[1], nz=box[2],
                    storage=rng.choice(["CSRD", "CSRC", "ELLPACK"]),
                    reorder=rng.random() < 0.5, pinned=rng.random() < 0.5,
                    prec="mixed" if kind == "mixed" else "fp64",
                    tol=1e-8 if kind == "mixed" else rng.choice([1e-8, 1e-11]))
    if kind in ("bicg", "gmres"):
        return dict(kind=kind, n=_log(rng, 10, 100), storage=rng.choice(["CSRD", "CSRC"]),
                    tol=rng.choice([1e-8, 1e-10]))
    if kind == "uvw":
        return dict(kind=kind, n=_log(rng, 14, 96), storage=rng.choice(["CSRD", "CSRC"]),
                    tol=rng.choice([1e-8, 1e-10]))
    if kind == "species":
        return dict(kind=kind, n=_log(rng, 10, 48), count=rng.randint(2, 10), storage="CSRD",
                    tol=1e-8)
    if kind == "adjoint":
        side = _log(rng, 10, 64)
        box = [max(5, round(side * rng.uniform(0.7, 1.2))) for _ in range(3)]
        return dict(kind=kind, nx=box[0], ny=box[1], nz=box[2],
                    storage=rng.choice(["CSRD", "ELLPACK"]), tol=1e-10)
    if kind == "uneven":
        return dict(kind=kind, count=rng.randint(5, 48), smin=8, smax=rng.randint(16, 40),
                    tol=1e-8)
    side = _log(rng, 12, 66)
    box = [max(5, round(side * rng.uniform(0.7, 1.3))) for _ in range(3)]
    return dict(kind="cells", nx=box[0], ny=box[1], nz=box[2])


# ---- what a program keeps ------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _context():
    return S.Context(0)


class _Dev:
    """A torch tensor as the device array the entry points take."""

    def __init__(self, t):
        self.t, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


def _put(a):
    return _Dev(torch.from_numpy(np.ascontiguousarray(a)).cuda())


def _zeros(n):
    return _Dev(torch.zeros(int(n), dtype=torch.float64, device="cuda"))


class _State(dict):
    """Inputs, outputs and handles of one case; the handles go with it."""

    def __del__(self):
        for h in self.get("handles", ()):
            h.destroy()


def _box(case):
    """The pressure-type system of a pcg2d, pcg3d or adjoint case."""
    st = STORAGE[case["storage"]]

    def make(seed):
        if case["kind"] == "pcg2d":
            return systems.poisson2d(case["nx"], case["ny"], seed=seed, storage=st)
        pin = case["nx"] * case["ny"] * case["nz"] // 2 if case.get("pinned") else None
        return systems.poisson3d(case["nx"], seed=seed, ny=case["ny"], nz=case["nz"],
                                 storage=st, reorder=bool(case.get("reorder", True)),
                                 pinned_cell=pin)
    return make


def _with(s, al=None, ad=None):
    return S.System(s.neq, s.nad, s.ia, s.ja, s.al if al is None else al,
                    s.ad if ad is None else ad, s.storage, s.unsym)


@functools.lru_cache(maxsize=2)
def _momentum(n, storage):
    return systems.momentum3d(n, storage=STORAGE[storage])


def _momentum_rhs(case, seed):
    """The momentum system and its three right-hand sides, the old velocity
    disturbed by the seed."""
    M = _momentum(case["n"], case["storage"])
    rng = np.random.default_rng(seed)
    h = 2.0 * math.pi / case["n"]
    bs = M.extra["b_all"] + 2.0 * h * h * 0.3 * rng.uniform(-1.0, 1.0, M.extra["b_all"].shape)
    return M.system, bs


@functools.lru_cache(maxsize=2)
def _species_pattern(n, storage):
    return systems.species3d(n, 1, storage=STORAGE[storage])[0]


def _species(case, seed):
    s, sp = systems.species3d(case["n"], case["count"], seed=seed, storage=STORAGE[case["storage"]])
    p = _species_pattern(case["n"], case["storage"])   # one mesh: the same ia/ja every time
    return S.System(s.neq, s.nad, p.ia, p.ja, s.al, s.ad, s.storage, s.unsym), sp


def _sides(case):
    """Cube sides, log-uniform between smin and smax in a mixed order."""
    ratio = case["smax"] / case["smin"]
    return [round(case["smin"] * ratio ** ((0.6180339887 * k + 0.5) % 1.0)) for k in range(case["count"])]


def _uneven(case, seed):
    return systems.uneven_batch(case["count"], seed=seed, kmin=1e-2, sides=np.array(_sides(case)))


@functools.lru_cache(maxsize=2)
def _mesh(nx, ny, nz):
    """The mesh with its momentum and pressure patterns (CSRD)."""
    m = systems.hex_mesh(nx, ny, nz, ratio=(1.01, 0.99, 1.0), shear=(0.05, 0.02, -0.03), warp=0.02)
    nel = m["nelcon"].reshape(-1, m["maxViz"])
    num = np.arange(1, m["numel"] + 1, dtype=np.int32)
    pats = []
    for ids, unsym in ((systems.simple_vel_case(m, seed=1)["id"], True),
                       (systems.simple_pres_case(m, seed=1)["id"], False)):
        pats.append(structure.datastruct(S.CSRD, unsym, ids, num, nel, m["nFace"], int(ids.max())))
    return m, nel, pats


def _zero_system(pat):
    n = pat.neq
    return S.System(n, pat.nad, pat.ia, pat.ja, np.zeros(max(1, int(pat.ia[n]))), np.ones(n),
                    pat.storage, bool(pat.unsym))


def prepare(case, seed):
    ctx, kind = _context(), case["kind"]
    if kind in ("pcg2d", "pcg3d", "adjoint"):
        B = _box(case)(seed)
        n = B.system.neq
        A = ctx.matrix(B.system)
        s = _State(case=case, A=A, handles=[A], b=_put(B.b[:n]), x=_zeros(n))
        if kind == "adjoint":
            g = np.random.default_rng(seed).uniform(-1.0, 1.0, n)
            s.update(g=_put(g), lam=_zeros(n), gal=_zeros(len(B.system.al)), gad=_zeros(n))
        return s
    if kind in ("bicg", "gmres"):
        sysm, bs = _momentum_rhs(case, seed)
        A = ctx.matrix(sysm)
        return _State(case=case, A=A, handles=[A], b=_put(bs[0]), x=_zeros(sysm.neq))
    if kind == "uvw":
        sysm, bs = _momentum_rhs(case, seed)
        ads = np.stack([sysm.ad[:sysm.neq] * (1.0 + 0.05 * c) for c in range(3)])
        A = ctx.matrix(_with(sysm, ad=ads[0]))
        return _State(case=case, A=A, handles=[A], ad=_put(ads.reshape(-1)),
                      b=_put(bs.reshape(-1)), x=_zeros(3 * sysm.neq))
    if kind == "species":
        sysm, sp = _species(case, seed)
        return _State(case=case, system=sysm, al=[a for a, _, _ in sp], ad=[d for _, d, _ in sp],
                      b=[b for _, _, b in sp])
    if kind == "uneven":
        built = _uneven(case, seed)
        Bt = ctx.batch([B.system for B in built], tune=False)
        hb, x, parts = np.zeros(Bt.rows), _zeros(Bt.rows), []
        for k, B in enumerate(built):
            r0 = Bt.info(k)["row0"]
            hb[r0:r0 + B.system.neq] = B.b[:B.system.neq]
            parts.append(x.t[r0:r0 + B.system.neq])
        return _State(case=case, batch=Bt, handles=[Bt], b=_put(hb), x=x, parts=parts)
    m, nel, pats = _mesh(case["nx"], case["ny"], case["nz"])
    numel = m["numel"]
    cv, cp = systems.simple_vel_case(m, seed=seed), systems.simple_pres_case(m, seed=seed, diffusion=4)
    vel, pres = ctx.cells(m, dict(cv, loadsPres=[])), ctx.cells(m, cp)
    Av, Ap = (ctx.matrix(_zero_system(p)) for p in pats)
    pv, pp = (ctx.assembly(A, p, c["id"], nel, m["nFace"]) for A, p, c in zip((Av, Ap), pats, (cv, cp)))
    neq = pats[0].neq
    s = _State(case=case, vel=vel, pres=pres, pv=pv, pp=pp, handles=[pv, pp, vel, pres, Av, Ap],
               opts=cv["opts"], neq=neq, id=_put(cv["id"]), lav=_zeros(7 * numel), advel=_zeros(3 * neq),
               bvel=_zeros(3 * neq), rcv=_zeros(3 * numel), dout=_zeros(3 * numel),
               lap=_zeros(7 * numel), lbp=_zeros(numel), rcp=_zeros(numel), bp=_zeros(pats[1].neq))
    for k in ("pres", "gradPres", "vel", "gradVel", "dField", "eddyVisc"):
        s["v_" + k] = _put(cv[k])
    for k in ("pres", "gradPres", "vel", "dField"):
        s["p_" + k] = _put(cp[k])
    return s


def run(s):
    ctx, case = _context(), s["case"]
    kind = case["kind"]
    if kind in ("pcg2d", "pcg3d"):
        prec = S.PREC_MIXED if case.get("prec") == "mixed" else S.PREC_FP64
        st = ctx.solve_device(s["A"], S.PCG, case["tol"], MAXIT, s["b"], s["x"], precision=prec)
        return {"x": s["x"].t, "xKx": st["xKx"], "norm_x": st["norm_x"], "status": st["status"]}
    if kind in ("bicg", "gmres"):
        sid = S.PBICGSTAB if kind == "bicg" else S.GMRES
        st = ctx.solve_device(s["A"], sid, case["tol"], MAXIT, s["b"], s["x"])
        return {"x": s["x"].t, "xKx": st["xKx"], "norm_x": st["norm_x"], "status": st["status"]}
    if kind == "uvw":
        st = (SfrStats * 3)()
        rc = lib.sfr_solve_shared_device(ctx.h, s["A"].h, 3, s["ad"].ptr, s["b"].ptr, s["x"].ptr,
                                         S.PBICGSTAB, case["tol"], MAXIT, 1, st)
        return {"x": s["x"].t, "norm_x": [v.norm_x for v in st], "status": rc}
    if kind == "species":
        xs, st = ctx.solve_batched(s["system"], S.PBICGSTAB, case["tol"], MAXIT, s["al"], s["ad"], s["b"])
        return {"x": xs, "status": [v["status"] for v in st]}
    if kind == "adjoint":
        st = ctx.solve_device(s["A"], S.PCG, case["tol"], MAXIT, s["b"], s["x"])
        sa = ctx.solve_adjoint(s["A"], S.PCG, case["tol"], MAXIT, s["x"], s["g"], s["lam"], s["gal"], s["gad"])
        return {"x": s["x"].t, "lambda": s["lam"].t, "grad_al": s["gal"].t, "grad_ad": s["gad"].t,
                "status": [st["status"], sa["status"]]}
    if kind == "uneven":
        st = s["batch"].solve_device(s["b"], s["x"], case["tol"], MAXIT)
        return {"x": s["parts"], "status": max(v["status"] for v in st)}
    s["vel"].vel(s["opts"], s["id"], s["neq"], s["v_pres"], s["v_gradPres"], s["v_vel"], s["v_gradVel"],
                 s["v_eddyVisc"], None, s["v_dField"], s["dout"], s["lav"], s["advel"], s["bvel"], s["rcv"])
    s["pv"].assemble(s["lav"])
    s["pres"].pres(4, s["p_pres"], s["p_gradPres"], s["p_vel"], s["p_dField"], s["lap"], s["lbp"], s["rcp"])
    s["pp"].assemble(s["lap"], s["lbp"], s["bp"])
    return {k: s[k].t for k in ("lav", "advel", "bvel", "rcv", "dout", "lap", "lbp", "rcp", "bp")}


# ---- what a pass cannot do without ---------------------------------------------

def _rows(case):
    """(rows, off-diagonal entries a row, longest side) of one system."""
    kind = case["kind"]
    if kind == "pcg2d":
        return case["nx"] * case["ny"], 4, max(case["nx"], case["ny"])
    if kind in ("bicg", "gmres", "uvw", "species"):
        return case["n"] ** 3, 6, case["n"]
    return case["nx"] * case["ny"] * case["nz"], 6, max(case["nx"], case["ny"], case["nz"])


def work(case):
    """Bytes: matrix (values, 2-byte column offsets, diagonal), right-hand
    side and solution once.  Operations: the iterations such a system takes
    to its tolerance, each a product and the solver's vector updates."""
    kind = case["kind"]
    if kind == "cells":
        # face geometry (15 planes and 2 indices a slot) and fields in,
        # coefficients, right-hand sides and residuals out, of both loops;
        # the assembled values once
        n = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": n * (1109 + 641 + 2 * 7 * 8 + 8), "flops": n * 2500}
    digits = -math.log10(case["tol"])
    if kind == "uneven":
        sides = _sides(case)
        return {"bytes": sum(v ** 3 for v in sides) * (6 * 10 + 24),
                "flops": sum(v ** 3 * 9.5 * v * digits / 8 * 24 for v in sides)}
    n, s, side = _rows(case)
    if kind in ("bicg", "uvw", "species"):
        k = {"bicg": 1, "uvw": 3, "species": case.get("count", 1)}[kind]
        mats = 1 if kind == "uvw" else k
        return {"bytes": mats * n * s * 8 + n * s * 2 + k * n * 24,
                "flops": k * n * digits * 0.9 * (4 * (s + 1) + 20)}
    if kind == "gmres":
        return {"bytes": n * (s * 10 + 24), "flops": n * 15 * math.ceil(digits / 9) * (2 * (s + 1) + 32)}
    its = 9.5 * side * digits / 8
    if kind == "adjoint":
        return {"bytes": n * (s * 10 + 24) + n * (s * 8 + 32), "flops": 2 * n * its * 24}
    return {"bytes": n * (s * 10 + 24), "flops": n * its * (2 * (s + 1) + 10)}


def tolerance(case):
    """A solve stops at a residual of tol, so two correct ones differ by what
    that leaves in the solution (an error that grows with the system's side,
    and with the FP32 iterations in mixed precision): about four times the
    error that the solves show.  Cell coefficients are the same bits by
    contract."""
    kind = case["kind"]
    if kind == "cells":
        return "exact"
    if kind == "uneven":
        return {"rel": 8e-6}
    if kind in ("pcg2d", "pcg3d", "adjoint"):
        side = _rows(case)[2]
        if case.get("prec") == "mixed":
            return {"rel": 4e-6 * max(side, 16) / 128}
        return {"rel": max(side * case["tol"], 2e-11)}
    return {"rel": max(4.0 * case["tol"], 2e-11)}


# ---- the same in 64 bits ---------------------------------------------------------

def _torch_matrix(s):
    """(off-diagonal entries as row, column and value, the diagonal)."""
    n, st = s.neq, s.storage
    if st == S.ELLPACK:
        w = int(s.ia[0])
        i = np.repeat(np.arange(n), w)
        j, a = s.ja[:n * w].astype(np.int64), s.al[:n * w]
    else:
        i = np.repeat(np.arange(n), np.diff(s.ia[:n + 1]))
        k = int(s.ia[n])
        j, a = s.ja[:k].astype(np.int64), s.al[:k]
        if st == S.CSRC and s.unsym:
            up = s.al[s.nad:s.nad + k]
            i, j, a = np.r_[i, j], np.r_[j, i], np.r_[a, up]
        elif not s.unsym:
            i, j, a = np.r_[i, j], np.r_[j, i], np.r_[a, a]
    keep = a != 0.0
    return i[keep], j[keep], a[keep], s.ad[:n]


def _csr(i, j, a, n):
    order = np.argsort(i, kind="stable")
    ptr = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(i, minlength=n), out=ptr[1:])
    t = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()  # noqa: E731
    return torch.sparse_csr_tensor(t(ptr), t(j[order]), t(a[order]), (n, n), dtype=torch.float64)


def _solve(i, j, a, ad, b, symmetric):
    """A^-1 b in 64 bits: Jacobi-preconditioned CG or BiCGSTAB to rounding."""
    n = len(ad)
    M, d = _csr(i, j, a, n), torch.from_numpy(np.ascontiguousarray(ad)).cuda()
    mul = lambda v: M.matmul(v) + d * v  # noqa: E731
    b = torch.from_numpy(np.ascontiguousarray(b)).cuda()
    x, r = torch.zeros_like(b), b.clone()
    stop = 1e-14 * float(b.norm())
    if symmetric:
        p = r / d
        rz = torch.dot(r, p)
        for k in range(6000):
            q = mul(p)
            al = rz / torch.dot(p, q)
            x += al * p
            r -= al * q
            z = r / d
            new = torch.dot(r, z)
            p = z + (new / rz) * p
            rz = new
            if k % 25 == 24 and float(r.norm()) < stop:
                break
        return x
    for _ in range(3):          # restarted on the true residual
        r = b - mul(x)
        r0, p, rho = r.clone(), r.clone(), torch.dot(r, r)
        for k in range(200):
            if float(r.norm()) < stop:
                break
            z = p / d
            v = mul(z)
            al = rho / torch.dot(v, r0)
            q = r - al * v
            y = q / d
            t = mul(y)
            w = torch.dot(t, q) / torch.dot(t, t)
            x += al * z + w * y
            r = q - w * t
            new = torch.dot(r, r0)
            p = r + (new / rho) * (al / w) * (p - w * v)
            rho = new
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind == "cells":
        return None             # the reference's cell loops: bit-exact by their own tests
    if kind in ("pcg2d", "pcg3d", "adjoint"):
        B = _box(case)(seed)
        n = B.system.neq
        i, j, a, ad = _torch_matrix(B.system)
        x = _solve(i, j, a, ad, B.b[:n], True)
        if kind == "adjoint":
            g = np.random.default_rng(seed).uniform(-1.0, 1.0, n)
            lam = _solve(i, j, a, ad, g, True)
            return {"x": x, "lambda": lam, "grad_al": None, "grad_ad": -lam * x, "status": [0, 0]}
        nx = float(x.norm())
        xKx = float(torch.dot(x, torch.from_numpy(np.ascontiguousarray(B.b[:n])).cuda()))
        return {"x": x, "xKx": xKx, "norm_x": nx, "status": 0}
    if kind in ("bicg", "gmres", "uvw"):
        sysm, bs = _momentum_rhs(case, seed)
        i, j, a, ad = _torch_matrix(sysm)
        if kind == "uvw":
            xs = [_solve(i, j, a, ad * (1.0 + 0.05 * c), bs[c], False) for c in range(3)]
            return {"x": torch.cat(xs), "norm_x": [float(x.norm()) for x in xs], "status": 0}
        x = _solve(i, j, a, ad, bs[0], False)
        xKx = float(torch.dot(x, torch.from_numpy(bs[0]).cuda()))
        return {"x": x, "xKx": xKx, "norm_x": float(x.norm()), "status": 0}
    if kind == "species":
        sysm, sp = _species(case, seed)
        xs = [_solve(*_torch_matrix(_with(sysm, al, ad)), b, False) for al, ad, b in sp]
        return {"x": xs, "status": [0] * len(xs)}
    built = _uneven(case, seed)
    parts = [_torch_matrix(B.system) for B in built]
    at = np.cumsum([0] + [B.system.neq for B in built])
    x = _solve(np.concatenate([p[0] + o for p, o in zip(parts, at)]),
               np.concatenate([p[1] + o for p, o in zip(parts, at)]),
               np.concatenate([p[2] for p in parts]), np.concatenate([p[3] for p in parts]),
               np.concatenate([B.b[:B.system.neq] for B in built]), True)
    return {"x": [x[i:j] for i, j in zip(at[:-1], at[1:])], "status": 0}
