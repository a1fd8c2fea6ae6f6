"""The work that a user of this library has it do, case by case.

Every case is one pass through a public entry point of ``mfix_amd`` on
seeded inputs: single solves (FP64 and mixed precision, LINE and DIAG, 2-D
and 3-D), the batched stage of a SIMPLE sweep, a batch of independent
systems, the assembled gas pressure correction and scalar transport chains,
the residual norms, the host-array drop-in and the serving loop.  Sizes and
solver settings are MFIX's defaults (LINE/RSRS, TOL 1e-4, ITMAX 5 for
momentum, 15 for scalars, 20 for the pressure correction) or those of the
library's own benchmark workloads (1e-10 solves).

``listed()`` names the cases, ``draw(rng)`` gives one more of the same
ranges, ``prepare(case, seed)`` makes what a program holds before the call,
``run(state)`` is the pass, ``work(case)`` its least bytes and flops and
``exact(case, seed)`` what 64-bit arithmetic gives for its outputs where
they have such a value (a solve that stops at ITMAX or at a loose TOL has
none for VAR: the iterate depends on where it stops).
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from mfix_amd import leq
from mfix_amd.serve import Server

DEV = "cuda"
RESID_FIELDS = ("num", "den", "resid", "max_resid", "ijk_resid", "ncells")


# ---- cases -------------------------------------------------------------------

def listed():
    return [
        # a 2-D run's pressure correction (MFIX's tutorials are 2-D grids of
        # this size): the smallest call, launches and their latency count
        dict(name="line_2d_30x90", path="solve", kind="pressure", imax=30, jmax=90, kmax=0, pc="LINE", mixed=False,
             tol=1e-4, itmax=20),
        # the parity configuration: 32^3 pressure correction to 1e-10
        dict(name="diag_32", path="solve", kind="pressure", imax=32, jmax=32, kmax=32, pc="DIAG", mixed=False,
             tol=1e-10, itmax=500),
        # upwind momentum 128^3, LINE, FP64 to 1e-10
        dict(name="line_128", path="solve", kind="momentum", imax=128, jmax=128, kmax=128, pc="LINE", mixed=False,
             tol=1e-10, itmax=500),
        # the mixed-precision counterpart on a ragged mid-size grid
        dict(name="line_mixed_90x117x101", path="solve", kind="momentum", imax=90, jmax=117, kmax=101, pc="LINE",
             mixed=True, tol=1e-10, itmax=500),
        # the headline: void-fraction pressure correction 256^3, mixed precision
        dict(name="void_256_mixed", path="solve", kind="void", imax=256, jmax=256, kmax=256, pc="DIAG", mixed=True,
             tol=1e-10, itmax=4000),
        # independent systems of one batched solve, DIAG or LINE each
        dict(name="batch_16_mixed", path="batch", nsys=16, lo=16, hi=96, spec=3, mixed=True, tol=1e-10, itmax=2000),
        # SOLVE_VEL_STAR of three phases: nine momentum equations in one flush
        dict(name="sweep_9x64", path="sweep", nsys=9, imax=64, jmax=64, kmax=64, tol=1e-4, itmax=5),
        # SOLVE_PP_G of one SIMPLE iteration, assembled and solved on the device
        dict(name="pp_g_256", path="pp_g", imax=256, jmax=256, kmax=256, tol=1e-4, itmax=20),
        # a scalar equation: CONV_DIF_PHI, SOURCE_PHI, then the residual, the
        # under-relaxation and the solve
        dict(name="phi_150x201x180", path="phi", imax=150, jmax=201, kmax=180, tol=1e-4, itmax=15),
        # CALC_RESID_C of an assembled equation
        dict(name="resid_200x230x170", path="resid", kind="C", imax=200, jmax=230, kmax=170),
        # the drop-in LEQ_BICGS on host arrays, as the Fortran program calls it
        dict(name="host_64", path="host", kind="momentum", imax=64, jmax=64, kmax=64, pc="LINE", tol=1e-4, itmax=5),
        # a burst of requests to the serving loop
        dict(name="serve_16", path="serve", nsys=16, lo=24, hi=100, spec=4, mixed=True, itmax=2000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["solve", "solve", "solve", "solve", "batch", "sweep", "pp_g", "phi", "resid", "host", "serve"])
    if path == "solve":
        if rng.random() < 0.25:
            imax, jmax, kmax = _log_int(rng, 10, 300), _log_int(rng, 10, 300), 0
        else:
            imax, jmax, kmax = (_log_int(rng, 10, 150) for _ in range(3))
        pc = rng.choice(["LINE", "LINE", "DIAG"])
        kind = rng.choice(["momentum", "pressure", "void"]) if kmax else rng.choice(["momentum", "pressure"])
        tol = rng.choice([1e-4, 1e-10])
        return dict(path=path, kind=kind, imax=imax, jmax=jmax, kmax=kmax, pc=pc, mixed=rng.random() < 0.4, tol=tol,
                    itmax=rng.choice([5, 15, 20]) if tol == 1e-4 else 2000)
    if path == "batch":
        return dict(path=path, nsys=rng.randint(2, 16), lo=16, hi=rng.randint(40, 96), spec=rng.randrange(1000),
                    mixed=rng.random() < 0.5, tol=1e-10, itmax=2000)
    if path == "sweep":
        imax, jmax, kmax = (_log_int(rng, 12, 100) for _ in range(3))
        return dict(path=path, nsys=rng.choice([3, 6, 9]), imax=imax, jmax=jmax, kmax=kmax, tol=1e-4, itmax=5)
    if path == "serve":
        return dict(path=path, nsys=rng.randint(4, 16), lo=24, hi=rng.randint(48, 100), spec=rng.randrange(1000),
                    mixed=rng.random() < 0.5, itmax=2000)
    if path == "host":
        imax, jmax, kmax = (_log_int(rng, 12, 96) for _ in range(3))
        return dict(path=path, kind=rng.choice(["momentum", "pressure"]), imax=imax, jmax=jmax, kmax=kmax, pc="LINE",
                    tol=1e-4, itmax=rng.choice([5, 20]))
    imax, jmax, kmax = (_log_int(rng, 20, 250) for _ in range(3))
    if path == "pp_g":
        return dict(path=path, imax=imax, jmax=jmax, kmax=kmax, tol=1e-4, itmax=20)
    if path == "phi":
        return dict(path=path, imax=imax, jmax=jmax, kmax=kmax, tol=1e-4, itmax=15)
    return dict(path="resid", kind=rng.choice(["C", "S", "PP"]), imax=imax, jmax=jmax, kmax=kmax)


# ---- seeded inputs, made on the GPU --------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) % (1 << 62))


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, dtype=torch.float64, device=DEV)


def _between(g, lo, hi, *shape):
    return lo + (hi - lo) * _rand(g, *shape)


def _dims(case):
    """Array shape (nk, ni, nj) with the ghost layers; one K plane in 2-D."""
    return (case["kmax"] + 2 if case["kmax"] else 1, case["imax"] + 2, case["jmax"] + 2)


def _interior(shape):
    m = torch.zeros(shape, dtype=torch.float64, device=DEV)
    (m[0] if shape[0] == 1 else m[1:-1])[..., 1:-1, 1:-1] = 1.0
    return m


def _put_faces(a, fw, axis, lo, hi):
    """Off-diagonals of the faces along `axis`: lo is the plane of the minus
    neighbour, hi of the plus one; fw = (coefficient seen from the plus cell,
    from the minus cell)."""
    n = a.shape[1 + axis]
    a[lo].narrow(axis, 1, n - 1).copy_(fw[0])
    a[hi].narrow(axis, 0, n - 1).copy_(fw[1])


def _inner_faces(m, axis):
    n = m.shape[axis]
    return m.narrow(axis, 0, n - 1) * m.narrow(axis, 1, n - 1)


PLANES = {0: (0, 6), 1: (2, 4), 2: (1, 5)}   # array axis (K, I, J) -> planes of its minus and plus neighbour


def _pressure(g, shape, void):
    """Symmetric pressure-correction system: faces 10^U[-1,1], times the
    face-averaged void fraction of a bed of spheres, and a small diagonal shift."""
    m = _interior(shape)
    eps = None
    if void:
        nk, ni, nj = shape
        eps = torch.ones(shape, dtype=torch.float64, device=DEV)
        ns = max(1, int(2000 * m.numel() / 258 ** 3))
        for cx, cy, cz, u in _rand(g, ns, 4).cpu().tolist():
            r = 3.0 + 9.0 * u
            c = [1 + cz * (nk - 2), 1 + cx * (ni - 2), 1 + cy * (nj - 2)]
            lo = [max(1, int(x - r)) for x in c]
            hi = [min(n - 1, int(x + r) + 2) for x, n in zip(c, shape)]
            if any(l >= h for l, h in zip(lo, hi)):
                continue
            ax = [(torch.arange(l, h, device=DEV, dtype=torch.float64) + 0.5 - x) ** 2 for l, h, x in zip(lo, hi, c)]
            box = eps[lo[0]:hi[0], lo[1]:hi[1], lo[2]:hi[2]]
            box[ax[0][:, None, None] + ax[1][None, :, None] + ax[2][None, None, :] <= r * r] = 0.4
    a = torch.zeros((7,) + shape, dtype=torch.float64, device=DEV)
    for axis, (lo, hi) in PLANES.items():
        n = shape[axis]
        if n == 1:
            continue
        im = _inner_faces(m, axis)
        f = im * 10.0 ** (2.0 * _rand(g, *im.shape) - 1.0)
        if eps is not None:
            f *= 0.5 * (eps.narrow(axis, 0, n - 1) + eps.narrow(axis, 1, n - 1))
        _put_faces(a, (f, f), axis, lo, hi)
    a[3] = torch.where(m > 0, -a.sum(0) - 1e-3 * _rand(g, *shape), torch.full_like(m, -1.0))
    return a, (1e-3 if void else 1.0) * m * (2.0 * _rand(g, *shape) - 1.0)


def _momentum(g, shape):
    """Nonsymmetric first-order-upwind system: diffusion 0.5*4^U, a
    divergence-free flux of eight modes with cell Peclet number up to 10, and
    the transient term of a CFL 0.5 step."""
    nk, ni, nj = shape
    n = (max(nk - 2, 1), ni - 2, nj - 2)          # interior cells along K, I, J
    modes = [(1 + (4.0 * _rand(g, 3)).floor(), 2.0 * _rand(g, 3) - 1.0) for _ in range(8)]

    def sines(length, p, half):
        x = torch.arange(length + (0 if half else 1), device=DEV, dtype=torch.float64) + (0.5 if half else 0.0)
        return torch.sin(math.pi * p * x / length)

    def psi(comp):
        """Component `comp` (K, I, J) of the vector potential on the grid edges along it."""
        out = 0.0
        for p, amp in modes:
            t = [sines(n[q], p[q], q == comp) for q in range(3)]
            if nk == 1:
                t[0] = torch.ones(1, device=DEV, dtype=torch.float64)
            out = out + amp[comp] * t[0][:, None, None] * t[1][None, :, None] * t[2][None, None, :]
        return out
    two_d = nk == 1
    pk = psi(0)
    fi, fj = pk.diff(dim=2), -pk.diff(dim=1)      # flux through the I faces and the J faces
    fk = None
    if not two_d:
        pi, pj = psi(1), psi(2)
        fi = fi - pj.diff(dim=0)
        fj = fj + pi.diff(dim=0)
        fk = pj.diff(dim=1) - pi.diff(dim=2)
    m = _interior(shape)
    flux, dif = {}, {}
    for axis, f in ((0, fk), (1, fi), (2, fj)):
        if f is None:
            continue
        f = f.narrow(axis, 1, n[axis] - 1)        # interior faces only: walls carry no flux
        flux[axis], dif[axis] = f, 0.5 * 4.0 ** _rand(g, *f.shape)
    pe = max(float((f.abs() / dif[q]).max()) if f.numel() else 0.0 for q, f in flux.items())
    scale = 10.0 / pe if pe > 0.0 else 0.0
    fmax = max(float(f.abs().max()) * scale if f.numel() else 0.0 for f in flux.values())
    transient = 2.0 * fmax if fmax > 0.0 else 1.0
    a = torch.zeros((7,) + shape, dtype=torch.float64, device=DEV)
    for axis, f in flux.items():
        lo, hi = PLANES[axis]
        f = f * scale
        whole = [0, 0]
        for side, v in enumerate((dif[axis] + f.clamp(min=0.0), dif[axis] + (-f).clamp(min=0.0))):
            w = torch.zeros(_inner_faces(m, axis).shape, dtype=torch.float64, device=DEV)
            inner = w if two_d else w.narrow(0, 1, w.shape[0] - 2)
            for q in (1, 2):
                inner = inner.narrow(q, 1, inner.shape[q] - 2)
            inner.copy_(v)
            whole[side] = w
        _put_faces(a, whole, axis, lo, hi)
    a[3] = torch.where(m > 0, -(a.sum(0) + transient), torch.full_like(m, -1.0))
    return a, m * (2.0 * _rand(g, *shape) - 1.0)


def _system(kind, shape, seed):
    g = _gen(seed)
    return _momentum(g, shape) if kind == "momentum" else _pressure(g, shape, kind == "void")


class Resident(leq.DeviceArray):
    """A torch tensor's memory handed to the library's *_dev entries."""

    def __init__(self, t):
        assert t.is_contiguous()
        self.t, self.n = t, t.numel()
        self.dtype = np.dtype(str(t.dtype).removeprefix("torch."))
        self.nbytes, self.ptr = self.n * self.dtype.itemsize, t.data_ptr()

    def free(self):
        self.ptr = None


class System:
    """A_M, B_M and VAR of one equation side by side in one block, as work
    arrays are: an assembly fills all of them before each solve, and a device
    copy of the assembled block stands for it here."""

    def __init__(self, a, b, block=None):
        n3 = b.numel()
        self.t = torch.empty(9 * n3, dtype=torch.float64, device=DEV) if block is None else block
        self.t[:7 * n3], self.t[7 * n3:8 * n3] = a.reshape(-1), b.reshape(-1)
        self.t[8 * n3:] = 0.0
        self.views = (self.t[8 * n3:], self.t[:7 * n3], self.t[7 * n3:8 * n3])
        self.var, self.a, self.b = (Resident(v) for v in self.views)

    def outputs(self):
        return dict(zip(("var", "a_m", "b_m"), self.views))


def _grid(case):
    leq.grid_init(case["imax"], case["jmax"], max(case["kmax"], 1), no_k=not case["kmax"])


def _specs(case):
    """The systems of a batch or of a burst of requests: sides, kinds and
    preconditioners, the same for every seed of the inputs."""
    rng = random.Random(case["spec"])
    out = []
    for q in range(case["nsys"]):
        if case["path"] == "batch":       # sides log-uniform, half of each kind, DIAG or LINE
            side, kind = _log_int(rng, case["lo"], case["hi"]), ("pressure", "momentum")[q % 2]
            pc, tol = rng.choice(["DIAG", "LINE"]), case["tol"]
        else:                             # sides lognormal around 64, 60 % momentum by LINE
            side = int(min(max(round(64.0 * math.exp(0.5 * rng.gauss(0.0, 1.0))), case["lo"]), case["hi"]))
            kind = "momentum" if rng.random() < 0.6 else "pressure"
            pc, tol = ("LINE" if kind == "momentum" else "DIAG"), rng.choice([1e-8, 1e-10])
        out.append(dict(kind=kind, imax=side, jmax=side, kmax=side, pc=pc, tol=tol))
    return out


def _flag(shape):
    """Ghost walls, an inflow face and a pressure-outflow face, fluid inside."""
    f = torch.full(shape, 100, dtype=torch.int32, device=DEV)
    f[1:-1, 1:-1, 1:-1] = 1
    f[1:-1, 0, 1:-1] = 20
    f[1:-1, -1, 1:-1] = 11
    return f


def _pp_fields(g, shape):
    dx = 0.01
    f = {k: _between(g, 0.5, 1.5, *shape) for k in ("rop_ge", "rop_gn", "rop_gt")}
    f |= {k: torch.full(shape, dx * dx, dtype=torch.float64, device=DEV) for k in ("ayz", "axz", "axy")}
    f["vol"] = torch.full(shape, dx ** 3, dtype=torch.float64, device=DEV)
    f["rop_g"] = _between(g, 0.9, 1.1, *shape)
    f |= {k: _between(g, -1.0, 1.0, *shape) for k in ("u_g", "v_g", "w_g")}
    f["sum_r_g"] = _between(g, -1e-3, 1e-3, *shape)
    f |= {k: _between(g, 0.1, 1.0, *shape) for k in ("d_e", "d_n", "d_t")}
    f["rop_go"] = f["rop_g"] * _between(g, 0.99, 1.01, *shape)
    return f


def _phi_fields(g, shape):
    nk, ni, nj = shape
    dx = 0.01
    f = {k: _between(g, -1.0, 1.0, *shape) for k in ("u", "v", "w")}
    rop = _between(g, 0.9, 1.1, *shape)
    area = torch.full(shape, dx * dx, dtype=torch.float64, device=DEV)
    f |= {"flux_e": rop * f["u"] * area, "flux_n": rop * f["v"] * area, "flux_t": rop * f["w"] * area}
    f |= {"ayz": area, "axz": area.clone(), "axy": area.clone(), "dif": _between(g, 0.5e-5, 2e-5, *shape)}
    f["s_p"] = rop * dx ** 3 * 100.0
    f["phi"] = _rand(g, *shape)
    f["s_c"] = f["s_p"] * f["phi"]
    f["ep"] = _between(g, 0.4, 1.0, *shape)

    def line(n, v):
        return torch.full((n,), v, dtype=torch.float64, device=DEV)
    f |= {"odx_e": line(ni, 1 / dx), "ody_n": line(nj, 1 / dx), "odz_t": line(nk, 1 / dx), "ox": line(ni, 1.0)}
    for name, n in (("fx_e", ni), ("fy_n", nj), ("fz_t", nk)):
        f |= {name: line(n, 0.5), name + "_bar": line(n, 0.5)}
    return f


class Requests:
    """Host arrays of a burst of requests and the server that takes them."""

    def __init__(self, case, seed):
        self.specs, self.mixed, self.itmax = _specs(case), case["mixed"], case["itmax"]
        self.arrays = []
        for q, s in enumerate(self.specs):
            a, b = (t.cpu().numpy().reshape(-1) for t in _system(s["kind"], _dims(s), seed * 64 + q))
            self.arrays.append((a, b, np.zeros_like(b)))
        self.server = Server(6 << 30, 64)

    def __del__(self):
        if getattr(self, "server", None) is not None:
            self.server.close()


# ---- prepare and run -----------------------------------------------------------

def prepare(case, seed):
    leq.init(0)
    path = case["path"]
    st = {"case": dict(case)}
    if path == "serve":
        return st | {"burst": Requests(case, seed)}
    if path == "batch":
        specs = _specs(case)
        sizes = [9 * math.prod(_dims(s)) for s in specs]
        block = torch.empty(sum(sizes), dtype=torch.float64, device=DEV)
        parts = torch.split(block, sizes)
        systems = [System(*_system(s["kind"], _dims(s), seed * 64 + q), block=p)
                   for q, (s, p) in enumerate(zip(specs, parts))]
        items = [leq.BatchSystem(s["imax"], s["jmax"], s["kmax"], y.var, y.a, y.b, pc=s["pc"], tol=s["tol"],
                                 itmax=case["itmax"], mixed=case["mixed"], seed=q)
                 for q, (s, y) in enumerate(zip(specs, systems))]
        return st | {"systems": systems, "items": items, "work": Resident(block), "fresh": Resident(block.clone())}
    _grid(case)
    shape = _dims(case)
    if path == "sweep":
        n = 9 * math.prod(shape)
        block = torch.empty(case["nsys"] * n, dtype=torch.float64, device=DEV)
        systems = [System(*_system("momentum", shape, seed * 64 + q), block=p)
                   for q, p in enumerate(torch.split(block, n))]
        return st | {"systems": systems, "work": Resident(block), "fresh": Resident(block.clone())}
    if path in ("pp_g", "phi"):
        g = _gen(seed)
        fields = _pp_fields(g, shape) if path == "pp_g" else _phi_fields(g, shape)
        st["fields"] = {k: Resident(v) for k, v in fields.items()}
        st["flag"] = Resident(_flag(shape))
        names = ("a", "b", "b_mmax", "pp_g") if path == "pp_g" else ("a", "b", "phi")
        st |= {k: Resident(torch.zeros((7,) * (k == "a") + shape, dtype=torch.float64, device=DEV)) for k in names}
        return st
    a, b = _system(case["kind"] if path in ("solve", "host") else "void", shape, seed)
    if path == "solve":
        y = System(a, b)
        return st | {"system": y, "work": Resident(y.t), "fresh": Resident(y.t.clone())}
    if path == "resid":
        var = _between(_gen(seed + 1), -1.0, 1.0, *shape)
        return st | {"a": Resident(a), "b": Resident(b), "var": Resident(var), "flag": Resident(_flag(shape))}
    a, b = (t.cpu().numpy().reshape(-1) for t in (a, b))
    return st | {"a": a, "b": b, "var": np.zeros_like(b)}


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "solve":
        state["work"].copy_from(state["fresh"])
        y = state["system"]
        r = leq.bicgs_dev(y.var, y.a, y.b, pc=case["pc"], cmethod="RSRS", tol=case["tol"], itmax=case["itmax"],
                          mixed=case["mixed"])
        return y.outputs() | {"ier": r.ier}
    if path == "batch":
        state["work"].copy_from(state["fresh"])
        res = leq.batch_solve(state["items"])
        return {"systems": [y.outputs() for y in state["systems"]], "ier": np.array([r.ier for r in res])}
    if path == "sweep":
        state["work"].copy_from(state["fresh"])
        for q, y in enumerate(state["systems"]):
            leq.solve_lin_eq_deferred("UVW"[q % 3], 3 + q % 3, y.var, y.a, y.b, case["itmax"], "RSRS", case["tol"],
                                      "LINE")
        done = leq.sweep_flush()
        return {"systems": [y.outputs() for y in state["systems"]], "ier": np.array([d.ier for d in done])}
    if path == "pp_g":
        r = leq.solve_pp_g_dev(state["fields"], state["flag"], 100.0, 0, 0.0, state["pp_g"], state["a"], state["b"],
                               state["b_mmax"], itmax=case["itmax"], tol=case["tol"], pc="LINE")
        return {k: state[k].t for k in ("pp_g", "a", "b", "b_mmax")} | {"resg": r["resg"], "ier": r["ier"]}
    if path == "phi":
        f, flag, a, b, phi = state["fields"], state["flag"], state["a"], state["b"], state["phi"]
        phi.copy_from(f["phi"])
        leq.conv_dif_phi_dev(f, flag, a, b, sync=False)
        leq.source_phi_dev(f["s_p"], f["s_c"], f["ep"], phi, flag, a, b, sync=False)
        resid, r = leq.resid_relax_bicgs_dev("S", phi, a, b, flag, 0.8, pc="LINE", tol=case["tol"],
                                             itmax=case["itmax"])
        return {"phi": phi.t, "a": a.t, "b": b.t, "ier": r.ier} | {k: resid[k] for k in RESID_FIELDS}
    if path == "resid":
        if case["kind"] == "PP":
            r = leq.calc_resid_dev("PP", b=state["b"], flag=state["flag"], norm=1.0)
        else:
            r = leq.calc_resid_dev(case["kind"], b=state["b"], flag=state["flag"], var=state["var"], a=state["a"])
        return {k: r[k] for k in RESID_FIELDS}
    if path == "host":
        # A_M and B_M come back row-scaled, as the reference leaves them: a
        # later pass is given the same equations in that form
        state["var"].fill(0.0)
        ier = leq.leq_bicgs("U_g", 3, state["var"], state["a"], state["b"], "RSRS", case["tol"], case["pc"],
                            case["itmax"])
        return {"var": state["var"], "a_m": state["a"], "b_m": state["b"], "ier": ier}
    burst = state["burst"]
    ids = []
    for q, (s, (a, b, x)) in enumerate(zip(burst.specs, burst.arrays)):
        x.fill(0.0)
        ids.append(burst.server.submit(a, b, x, s["imax"], s["jmax"], s["kmax"], pc=s["pc"], tol=s["tol"],
                                       itmax=burst.itmax, mixed=burst.mixed, seed=q))
    burst.server.run_until_done()
    done = [burst.server.poll(i) for i in ids]
    return {"var": [d.var for d in done], "ier": np.array([d.ier for d in done])}


# ---- work ------------------------------------------------------------------------

def _iterations(kind, pc, side, tol, itmax):
    """Iterations such a solve takes (measured on these systems, to a few per cent)."""
    if kind == "momentum":
        n = 4 if pc == "LINE" else 13
    else:
        n = (300 if pc == "DIAG" else 95) * (side / 32.0) ** 0.75
    return max(1.0, min(itmax, n * (0.4 if tol > 1e-6 else 1.0)))


def _solve_work(cells, kind, pc, mixed, tol, itmax, host=False):
    """The system read once and left scaled, and per iteration the least an
    iteration moves: the coefficients and the Krylov vectors of the fused
    schedule (DIAG 15 coefficients and 15 vectors a cell, LINE 42 and 30)."""
    its = _iterations(kind, pc, cells ** (1 / 3), tol, itmax)
    s = 4 if mixed else 8
    per = (15 * s + 15 * s if pc == "DIAG" else 42 * s + 30 * s) + 16
    flops = 60 if pc == "DIAG" else 180
    return {"bytes": cells * (2.0 * 9 * 8 + its * per), "flops": cells * its * flops}


def work(case):
    path = case["path"]
    if path in ("batch", "serve"):
        each = [_solve_work(math.prod(_dims(s)), s["kind"], s["pc"], case["mixed"], s["tol"], case["itmax"])
                for s in _specs(case)]
        return {k: sum(e[k] for e in each) for k in ("bytes", "flops")}
    cells = math.prod(_dims(case))
    if path == "resid":
        return {"bytes": cells * (12.0 if case["kind"] == "PP" else 76.0), "flops": cells * 16.0}
    if path == "sweep":
        one = _solve_work(cells, "momentum", "LINE", False, case["tol"], case["itmax"])
        return {k: case["nsys"] * v for k, v in one.items()}
    if path == "pp_g":
        w = _solve_work(cells, "pressure", "LINE", False, case["tol"], case["itmax"])
        return {"bytes": w["bytes"] + cells * 204.0, "flops": w["flops"] + cells * 50.0}
    if path == "phi":
        # (the accumulation term lets LINE converge in one iteration)
        w = _solve_work(cells, "momentum", "LINE", False, case["tol"], 1)
        return {"bytes": w["bytes"] + cells * (148.0 + 48.0), "flops": w["flops"] + cells * 100.0}
    return _solve_work(cells, case["kind"], case["pc"], case.get("mixed", False), case["tol"], case["itmax"])


# ---- the outputs in plain 64-bit arithmetic -----------------------------------------

def _neighbour(x, axis, step):
    """x at the neighbour along `axis`, the cell itself past the array's end."""
    n = x.shape[axis]
    if n == 1:
        return x
    if step < 0:
        return torch.cat([x.narrow(axis, 0, 1), x.narrow(axis, 0, n - 1)], axis)
    return torch.cat([x.narrow(axis, 1, n - 1), x.narrow(axis, n - 1, 1)], axis)


def _matvec(a, x):
    y = a[3] * x
    for axis, (lo, hi) in PLANES.items():
        n = x.shape[axis]
        if n == 1:
            continue
        y.narrow(axis, 1, n - 1).addcmul_(a[lo].narrow(axis, 1, n - 1), x.narrow(axis, 0, n - 1))
        y.narrow(axis, 0, n - 1).addcmul_(a[hi].narrow(axis, 0, n - 1), x.narrow(axis, 1, n - 1))
    return y


def _scaled(a, b):
    s = 1.0 / a.abs().amax(0)
    return a * s, b * s


def _solution(a, b, limit=3000):
    """A x = b for a row-scaled system by BiCGSTAB to 1e-14 of ||b||; None if it does not get to 1e-12."""
    d = 1.0 / a[3]
    x, r = torch.zeros_like(b), b.clone()
    top = float(b.norm())
    if top == 0.0:
        return x
    q, p, v = r.clone(), r.clone(), None
    rho = float((q * r).sum())
    for it in range(limit):
        v = _matvec(a, p * d)
        alpha = rho / float((q * v).sum())
        s = r - alpha * v
        t = _matvec(a, s * d)
        omega = float((t * s).sum()) / max(float((t * t).sum()), 1e-300)
        x += (alpha * p + omega * s) * d
        r = s - omega * t
        new = float((q * r).sum())
        size = float(r.norm())
        if size <= 1e-14 * top or rho == 0.0 or omega == 0.0:
            break
        if it % 100 == 99:                # start again from the true residual
            r = b - _matvec(a, x)
            q, p = r.clone(), r.clone()
            rho = float((q * r).sum())
            continue
        p = r + (new / rho) * (alpha / omega) * (p - omega * v)
        rho = new
    return x if float((b - _matvec(a, x)).norm()) <= 1e-12 * top else None


def _exact_solve(a, b, tol, var):
    a, b = _scaled(a, b)
    x = _solution(a, b) if var and tol <= 1e-8 else None
    return {"var": None if x is None else x.reshape(-1), "a_m": a.reshape(-1), "b_m": b.reshape(-1)}


def exact(case, seed):
    path = case["path"]
    if path in ("solve", "host"):
        a, b = _system(case["kind"], _dims(case), seed)
        r = _exact_solve(a, b, case["tol"], a[0].numel() < 1 << 22)
        return ({k: None if v is None else v.cpu().numpy() for k, v in r.items()} if path == "host" else r) | {"ier": None}
    if path in ("batch", "sweep", "serve"):
        specs = _specs(case) if path != "sweep" else [dict(case, kind="momentum")] * case["nsys"]
        each = [_exact_solve(*_system(s["kind"], _dims(s), seed * 64 + q), s["tol"], True) for q, s in enumerate(specs)]
        if path == "serve":
            return {"var": [None if e["var"] is None else e["var"].cpu().numpy() for e in each], "ier": None}
        return {"systems": each, "ier": None}
    shape = _dims(case)
    flag = _flag(shape)
    fluid = flag == 1
    if path == "resid":
        a, b = _system("void", shape, seed)
        v = _between(_gen(seed + 1), -1.0, 1.0, *shape)
        r = b - a[3] * v
        for axis, planes in PLANES.items():
            for plane, step in zip(planes, (-1, 1)):
                vn = _neighbour(v, axis, step)
                if case["kind"] == "C":   # a wall neighbour stands for the cell itself
                    vn = torch.where(_neighbour(flag, axis, step) >= 100, v, vn)
                r = r - a[plane] * vn
        if case["kind"] == "PP":
            r, den1 = b, torch.ones_like(b)
        else:
            den1 = (a[3] * v).abs()
        r = torch.where(fluid, r.abs(), torch.zeros_like(r))
        num, den, cells = float(r.sum()), float(den1[fluid].sum()), int(fluid.sum())
        return {"num": num, "den": den, "resid": num / den, "max_resid": cells * float(r.max()) / den,
                "ijk_resid": None, "ncells": None}
    g = _gen(seed)
    low = {0: "t", 1: "e", 2: "n"}
    zero = torch.zeros(shape, dtype=torch.float64, device=DEV)
    a = torch.zeros((7,) + shape, dtype=torch.float64, device=DEV)
    if path == "pp_g":
        f = _pp_fields(g, shape)
        area, vel = {0: "axy", 1: "ayz", 2: "axz"}, {0: "w_g", 1: "u_g", 2: "v_g"}
        src = (f["rop_g"] - f["rop_go"]) * f["vol"] * 100.0
        react = f["sum_r_g"] * f["vol"]
        net, top = src.clone(), torch.maximum(src.abs(), react.abs())
        for axis, (lo, hi) in PLANES.items():
            plus = f["rop_g" + low[axis]] * f[area[axis]]
            through = plus * f[vel[axis]]
            net = net + through - _neighbour(through, axis, -1)
            top = torch.maximum(top, torch.maximum(through.abs(), _neighbour(through, axis, -1).abs()))
            a[hi] = plus * f["d_" + low[axis]]
            a[lo] = _neighbour(a[hi], axis, -1)
        b = torch.where(fluid, net - react, zero)
        a[3] = torch.where(fluid, -a.sum(0), zero - 1.0)
        for axis, planes in PLANES.items():
            for plane, step in zip(planes, (-1, 1)):
                nb = _neighbour(flag, axis, step)
                a[plane] = torch.where(fluid & (nb != 10) & (nb != 11), a[plane], zero)
        bm = torch.where(fluid, top, zero)
        cells = float(fluid.sum())
        resg = (float(b.abs().sum()) / cells) / (float(bm.sum()) / cells / 10.0)
        a, b = _scaled(a, b)
        return {"pp_g": None, "a": a, "b": b, "b_mmax": bm, "resg": resg, "ier": None}
    f = _phi_fields(g, shape)
    area, vel = {0: "axy", 1: "ayz", 2: "axz"}, {0: "w", 1: "u", 2: "v"}
    wall = flag >= 100
    for axis, (lo, hi) in PLANES.items():
        dm, dp = f["dif"], _neighbour(f["dif"], axis, 1)
        wm, wp = wall, _neighbour(wall.to(torch.int32), axis, 1) > 0
        dm, dp = torch.where(wm, dp, dm), torch.where(wp, dm, dp)
        d = dm * dp / torch.clamp(0.5 * dm + 0.5 * dp, min=1e-15) * (100.0 * f[area[axis]])   # 1 cm cells
        flow, up = f["flux_" + low[axis]], f[vel[axis]] >= 0.0
        touches = fluid | (_neighbour(fluid.to(torch.int32), axis, 1) > 0)
        a[hi] = torch.where(fluid, torch.where(up, d, d - flow), zero)
        plus = torch.where(touches, torch.where(up, d + flow, d), zero)
        n = shape[axis]
        a[lo].narrow(axis, 1, n - 1).copy_(plus.narrow(axis, 0, n - 1))
    nb = a.sum(0)
    a[3] = torch.where(fluid, -(nb + f["s_p"]), zero - 1.0)
    b = torch.where(fluid, -f["s_c"], zero)
    r = b - a[3] * f["phi"]
    for axis, planes in PLANES.items():
        for plane, step in zip(planes, (-1, 1)):
            r = r - a[plane] * _neighbour(f["phi"], axis, step)
    r = torch.where(fluid, r.abs(), zero)
    num, den, cells = float(r.sum()), float((a[3] * f["phi"]).abs()[fluid].sum()), int(fluid.sum())
    b = torch.where(fluid, b + a[3] * f["phi"] * (1.0 / 0.8 - 1.0), b)
    a[3] = torch.where(fluid, a[3] / 0.8, a[3])
    a, b = _scaled(a, b)
    return {"phi": None, "a": a, "b": b, "ier": None, "num": num, "den": den, "resid": num / den,
            "max_resid": cells * float(r.max()) / den, "ijk_resid": None, "ncells": None}
