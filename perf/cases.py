"""Performance cases of the HDG Newton-GMRES framework: the solves, time steps, batches and single
stages that a program runs through exasim_amd.hdg, over the sizes its workloads use.

A case's "kind" names the call that is timed:

* ``solve``    reset() and solve() of one steady problem: the residual, assembly and condensation,
               the preconditioner's set-up, GMRES, the update and, in the mixed form, refinement;
* ``batch``    the same for a batch of independent problems in one handle;
* ``step``     reset() and solve() of a time-dependent problem: DIRK stages, each a Newton solve;
* ``assemble`` assemble() alone, for programs that solve the condensed system themselves;
* ``matvec``   the condensed matvec alone, the same programs' operator;
* ``gmres``    gmres() on the assembled system with a right-hand side of the caller's.

"problem" names the workload the package's own benchmark and examples are made of: ``poisson``
(the steady Poisson examples in 2D and 3D), ``cd2d`` (the served and batched 2D convection-diffusion
requests), ``cd3d`` (the two-component 3D convection-diffusion problem and its batch) and ``ns2d``
(compressible Navier-Stokes).  "precision" is the solver's option: 0 FP64, 1 mixed.
"""
import os
import tempfile

import numpy as np
import torch

from exasim_amd import cases as builders
from exasim_amd import datain as dw
from exasim_amd.hdg import HDGSolver

_CD2D_SIZES = (8, 16, 24, 32, 48, 64)     # the 2D batch workload's grids
_CD3D_SIZES = (4, 6, 8)                   # the 3D batch workload's grids, without its largest


def listed():
    return [
        # The smallest call: the reference's 2D Poisson example (16 x 16 quads, p = 3, block-Jacobi,
        # MGS), 2176 trace unknowns; launches and latency count.
        dict(name="poisson2d_16_p3", kind="solve", problem="poisson", nd=2, n=16, p=3, precond="bjacobi",
             ortho=0, precision=0),
        # The 3D Poisson example on an odd grid (m = 96).
        dict(name="poisson3d_11_p3", kind="solve", problem="poisson", nd=3, n=11, p=3, precond="bjacobi",
             ortho=0, precision=0),
        # One served request at the highest order, on an odd grid: Schwarz, CGS, mixed form.
        dict(name="cd2d_61_p5_mixed", kind="solve", problem="cd2d", nd=2, n=61, p=5, precond="eas", ortho=1,
             precision=1),
        # The headline workload (3D convection-diffusion, p = 4, superelement block-ILU(0)) in FP64 and
        # in the mixed form with BF16 factors, on the largest grid of which three states fit the card.
        dict(name="cd3d_20_p4", kind="solve", problem="cd3d", nd=3, n=20, p=4, precond="bilu0", ortho=1,
             precision=0),
        dict(name="cd3d_20_p4_mixed", kind="solve", problem="cd3d", nd=3, n=20, p=4, precond="bilu0", ortho=1,
             precision=1),
        # The parametrized 2D batch (FP64) and the 3D batch (mixed, BF16 Schwarz blocks), one order each.
        dict(name="batch_cd2d_24_p4", kind="batch", problem="cd2d", nd=2, count=24, p=4, precond="eas", ortho=1,
             precision=0),
        dict(name="batch_cd3d_8_p3_mixed", kind="batch", problem="cd3d", nd=3, count=8, p=3, precond="eas",
             ortho=1, precision=1),
        # Navier-Stokes time steps: DIRK(3,3) with block-ILU(0) on the channel grid in the mixed form,
        # and a served request's DIRK(2,2) step with Schwarz on an odd square grid in FP64.
        dict(name="ns2d_128x32_p4_mixed", kind="step", problem="ns2d", nd=2, n=128, ny=32, p=4, precond="bilu0",
             ortho=0, stages=3, precision=1),
        dict(name="ns2d_45_p5", kind="step", problem="ns2d", nd=2, n=45, ny=45, p=5, precond="eas", ortho=1,
             stages=2, precision=0),
        # Single stages: assembly and condensation, the operator, and the Krylov solve.
        dict(name="assemble_cd3d_13_p3", kind="assemble", problem="cd3d", nd=3, n=13, p=3, precond="eas", ortho=1,
             precision=0),
        dict(name="matvec_cd3d_22_p3_mixed", kind="matvec", problem="cd3d", nd=3, n=22, p=3, precond="bjacobi",
             ortho=1, precision=1),
        dict(name="gmres_cd3d_15_p2", kind="gmres", problem="cd3d", nd=3, n=15, p=2, precond="bjacobi", ortho=1,
             precision=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "batch", "step", "assemble", "matvec", "gmres"])
    precision = rng.choice([0, 1])
    if kind == "step":
        p = rng.choice([2, 3, 4, 5])
        precond = rng.choice(["bilu0", "eas"])
        n = _log_int(rng, 12, 128 if p < 5 else 64)
        ny = _log_int(rng, 12, 48 if p < 5 else 32)
        if precond == "bilu0":                     # 2 x 2 superelements
            n, ny = n + n % 2, ny + ny % 2
        return dict(kind=kind, problem="ns2d", nd=2, n=n, ny=ny, p=p, precond=precond,
                    ortho=0 if precond == "bilu0" else 1, stages=rng.choice([2, 3]), precision=precision)
    if kind == "batch":
        if rng.random() < 0.5:
            return dict(kind=kind, problem="cd2d", nd=2, count=_log_int(rng, 2, 32), p=rng.choice([2, 3, 4, 5]),
                        precond="eas", ortho=1, precision=precision)
        return dict(kind=kind, problem="cd3d", nd=3, count=_log_int(rng, 2, 12), p=rng.choice([2, 3, 4]),
                    precond="eas", ortho=1, precision=precision)
    problem = rng.choice(["poisson", "cd2d", "cd3d"])
    if problem == "cd2d":
        return dict(kind=kind, problem=problem, nd=2, n=_log_int(rng, 8 if kind != "matvec" else 24, 128), p=rng.choice([2, 3, 4, 5]),
                    precond="eas", ortho=1, precision=precision)
    nd = 3 if problem == "cd3d" else rng.choice([2, 3])
    p = rng.choice([1, 2, 3, 4, 5] if nd == 2 else [2, 3, 4])
    n = _log_int(rng, 6, 64) if nd == 2 else _log_int(rng, 4, {2: 24, 3: 20, 4: 18}[p])
    if kind == "matvec":                           # single matvecs of grids that take over a few microseconds
        n, p = max(n, 12), max(p, 2)
    precond = rng.choice(["bjacobi", "eas", "bilu0"])
    if precond == "bilu0":                         # 2 x 2 (x 2) superelements
        n += n % 2
    return dict(kind=kind, problem=problem, nd=nd, n=n, p=p, precond=precond, ortho=rng.choice([0, 1]),
                precision=precision)


# ---- the inputs of a case, from the seed ------------------------------------------------------

def _instances(case, seed):
    """The problems of a case as plain parameters, one per instance (one for all but batches)."""
    rng = np.random.default_rng(seed)
    prob, out = case["problem"], []
    for i in range(case.get("count", 1)):
        d = dict(seed=int(rng.integers(1 << 30)))
        batch = case["kind"] == "batch"
        if prob == "poisson":
            d.update(n=case["n"], kappa=float(rng.uniform(0.5, 2.0)), vel=(0.0,) * case["nd"])
        elif prob == "cd2d":                       # kappa log-uniform in [1e-3, 1], any direction
            n = int(_CD2D_SIZES[(5 * i + 3) % 6]) if batch else case["n"]
            lo = -3.0 if batch else -2.0
            d.update(n=n, kappa=float(10.0 ** rng.uniform(lo, 0.0)), angle=float(rng.uniform(0, 2 * np.pi)),
                     k=int(rng.integers(1, 5)))
            d["vel"] = (float(np.cos(d["angle"])), float(np.sin(d["angle"])))
        elif prob == "cd3d" and batch:
            v = rng.normal(size=3)
            v /= np.linalg.norm(v)
            d.update(n=int(_CD3D_SIZES[i % 3]), kappa=float(10.0 ** rng.uniform(-2.0, -1.0)),
                     vel=tuple(float(x) for x in v))
        elif prob == "cd3d":
            d.update(n=case["n"], kappa=1e-2, vel=(1.0, 0.5, 0.25))
        else:
            d.update(mach=float(rng.uniform(0.3, 0.5)), re=float(10.0 ** rng.uniform(2.5, 3.0)))
        out.append(d)
    return out


def _write(case, d, path):
    nd, p, pre = case["nd"], case["p"], case["precond"]
    cart = [] if pre != "bilu0" or "n" not in d else [nd] + [d["n"]] * nd + [2] * nd + [0]
    if case["problem"] == "poisson":
        builders.poisson2d(path, n=d["n"], porder=p, pgauss=2 * p, kappa=d["kappa"], precond=pre, nd=nd,
                           ortho=case["ortho"], cartgridpart=cart, gmres_maxit=2000)
        return "poisson"
    if case["problem"] == "cd2d":
        builders.convdiff2d_param(path, n=d["n"], porder=p, kappa=d["kappa"], angle=d["angle"], k=d["k"],
                                  precond=pre, restart=100, ortho=case["ortho"])
        return "cd2d"
    if case["problem"] == "cd3d":
        builders.convdiff3d(path, n=d["n"], porder=p, kappa=d["kappa"], vel=d["vel"], seed=d["seed"], precond=pre,
                            ortho=case["ortho"], cartgridpart=cart, inflow_dirichlet=case["kind"] == "batch")
        return "convdiff"
    S = case["stages"]
    served = pre == "eas"                          # a served request, or the channel with bumps
    builders.navierstokes2d(path, nx=case["n"], ny=case["ny"], porder=p, mach=d["mach"], re=d["re"], seed=d["seed"],
                            length=(1.0, 1.0) if served else (5.0, 1.0), stretch=1.0 if served else 1.05,
                            nbumps=8, dt=5e-3 if served else 1e-2, nsteps=1, torder=S, nstage=S, precond=pre,
                            tau=1.0 + 1.0 / d["mach"], gmres_tol=1e-10, newton_tol=1e-10, ortho=case["ortho"],
                            restart=50 if served else 100, cartgridpart=not served)
    return "ns2d"


class _Device:
    """A library device array as something torch can view without a copy."""

    def __init__(self, solver, name):
        ptr, n = solver.device_ptr(name)
        self.solver = solver                       # the array lives as long as its handle
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<f8", data=(ptr, False), version=2, strides=None)


def _view(solver, name):
    t = torch.as_tensor(_Device(solver, name), device="cuda")
    t.solver = solver
    return t


def prepare(case, seed):
    inst = _instances(case, seed)
    with tempfile.TemporaryDirectory() as tmp:
        paths, model = [], None
        for i, d in enumerate(inst):
            paths.append(os.path.join(tmp, "%03d" % i))
            model = _write(case, d, paths[-1])
        S = HDGSolver.batch(paths, model) if case["kind"] == "batch" else HDGSolver(paths[0], model)
    if case["precision"]:
        # the benchmark's refinement settings and BF16 preconditioner blocks
        cycles = case["kind"] == "batch" and case["nd"] == 2
        S.set_option("precision", 1)
        for k, v in (dict(refine_first_tol=1e-7, refine_tol=1e-7, refine_cycles=1, refine_maxit=40) if cycles
                     else dict(refine_first_tol=1e-5, refine_tol=1e-5)).items():
            S.set_option(k, v)
        S.set_option("precond_bf16", 0 if cycles else 1)
    state = dict(kind=case["kind"], solver=S)
    if case["kind"] in ("solve", "batch", "step"):
        state["out"] = [_view(S, "udg"), _view(S, "uh")]
    elif case["kind"] == "assemble":
        S.get_q()
        state["out"] = [_view(S, "b")] + ([] if case["precision"] else [_view(S, "H"), _view(S, "DinvF")])
    else:
        S.get_q()
        S.assemble()
        state["v"] = torch.from_numpy(_vector(S.sizes["N"], seed)).cuda()
        state["w"] = torch.empty_like(state["v"])
    S.sync()
    torch.cuda.synchronize()
    return state


def _vector(N, seed):
    return np.random.default_rng(seed + 1).standard_normal(N)


def run(state):
    S, kind = state["solver"], state["kind"]
    if kind == "assemble":
        S.assemble()
        return state["out"]
    if kind == "matvec":
        S.matvec(state["v"].data_ptr(), state["w"].data_ptr())
        return state["w"]
    if kind == "gmres":
        S.gmres(state["v"].data_ptr(), state["w"].data_ptr())
        return state["w"]
    S.reset()
    S.solve()
    return state["out"]


# ---- what a pass cannot do without, and how exact its results are ------------------------------

def _sizes(case, n, ny=None):
    nd, p = case["nd"], case["p"]
    ncu = {"poisson": 1, "cd2d": 1, "cd3d": 2, "ns2d": 4}[case["problem"]]
    npe, npf = (p + 1) ** nd, (p + 1) ** (nd - 1)
    ne = n * (ny or n) * (n if nd == 3 else 1)
    return dict(nd=nd, ncu=ncu, ne=ne, npe=npe, npf=npf, n=npe * ncu, m=2 * nd * npf * ncu,
                N=(nd * ne + nd * n ** (nd - 1)) * npf * ncu)


def work(case):
    """Bytes: the fields of the state, the geometry and the coefficients read once and the results
    written once; for a stage on the assembled system, the condensed operator read once.  Flops: the
    elimination of q and u, and two per entry of the operator for each GMRES iteration (the counts are
    round figures of the workloads, whose solves stop at a tolerance)."""
    size, flops, moved = (4 if case["precision"] else 8), 0.0, 0.0
    iters = {"bjacobi": 150, "eas": 80, "bilu0": 60}[case["precond"]]
    for d in _instances(case, 1):
        z = _sizes(case, d.get("n", case.get("n")), case.get("ny"))
        n, m, ne, ncu, q = z["n"], z["m"], z["ne"], z["ncu"], z["npe"] * z["nd"]
        op, vec = float(m) * m * ne, z["N"] * 8.0
        eliminate = ne * (2.0 * q * ncu * (n + m) * (z["npe"] + m / ncu)
                          + 2.0 / 3.0 * n ** 3 + 2.0 * n * n * (m + 1) + 2.0 * m * m * n)
        fields = ne * z["npe"] * (z["nd"] + ncu * (z["nd"] + 2)) * 8.0
        if case["kind"] in ("solve", "batch", "step"):
            k = case.get("stages", 1) * (2 if case["problem"] == "ns2d" else 1)
            flops += k * (eliminate + iters * 2.0 * op)
            moved += fields + ne * z["npe"] * ncu * (z["nd"] + 1) * 8.0 + vec
        elif case["kind"] == "assemble":
            flops += eliminate
            moved += fields + vec + (ne * float(n) * m + op) * size
        else:
            flops += (iters if case["kind"] == "gmres" else 1) * 2.0 * op
            moved += op * size + 2 * vec
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    # About four times the largest error against exact() over the ranges.  Solves stop at 1e-10 of
    # the right-hand side and the mixed form refines to 1e-10 of its first residual: 4e-10 seen on the
    # fields, 1e-9 between the two forms of a Navier-Stokes step; a random right-hand side 6e-9, and
    # 1e-4 with the FP32 operator.  Stages carry their type's rounding: 5e-12 (D^-1 F at p = 5) and
    # 5e-7 for the assembly, 1e-13 and 8e-7 for the matvec.
    mixed = bool(case["precision"])
    if case["kind"] in ("solve", "batch", "step"):
        return {"rel": 4e-9, "max": 1e-6}
    rel = {"gmres": (2.5e-8, 4e-4), "assemble": (2e-11, 2e-6), "matvec": (1e-12, 3e-6)}[case["kind"]][mixed]
    return {"rel": rel, "max": 100 * rel}


# ---- the same discretisation in plain torch, in 64 bits ------------------------------------------
# On a uniform grid with constant coefficients every element has the same local matrices, except
# for its boundary rows, and the components do not couple.

_FACES = {2: ((0, 1), (1, 2), (2, 3), (3, 0)),
          3: ((0, 3, 2, 1), (4, 5, 6, 7), (0, 1, 5, 4), (2, 3, 7, 6), (1, 2, 6, 5), (3, 0, 4, 7))}


class _Exact:
    """One linear problem (poisson, cd2d, cd3d) on its grid: local matrices by boundary type,
    face numbering and the condensed system of one component."""

    def __init__(self, case, d):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        T = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=self.dev)  # noqa: E731
        nd, p, self.case, self.d = case["nd"], case["p"], case, d
        m = dw.make_master(nd, p, 2 * p)
        pts, t = dw.structured_grid([d["n"]] * nd)
        self.xdg = xdg = dw.compute_dgnodes(m, pts, t)
        self.nd, self.ne, self.npe, self.npf = nd, t.shape[0], m["npe"], m["npf"]
        nfe = 2 * nd
        self.ndf = nfe * self.npf
        perm = np.asarray(m["perm"]).reshape(nfe, self.npf)
        kappa, vel, tau = d["kappa"], d["vel"], 1.0

        # faces: interior ones in the order their second side is met, then boundary ones by condition
        fv = np.sort(t[:, np.array(_FACES[nd])], axis=2).reshape(self.ne * nfe, -1)
        _, first, inv, cnt = np.unique(fv, axis=0, return_index=True, return_inverse=True, return_counts=True)
        inv = inv.reshape(-1)
        side = np.arange(self.ne * nfe)
        second = side[(side != first[inv]) & (cnt[inv] == 2)]
        bnd = side[cnt[inv] == 1]
        x0 = pts[t[:, np.array(_FACES[nd])]].reshape(self.ne * nfe, -1, nd)
        bc = self._conditions(x0[bnd])
        o = np.argsort(bc, kind="stable")
        bnd, bc = bnd[o], bc[o]
        self.nf = len(second) + len(bnd)
        s1 = np.concatenate([first[inv[second]], bnd])
        xf = xdg[:, perm].reshape(self.ne * nfe, self.npf, nd)          # trace node coordinates
        con = np.empty((self.ne * nfe, self.npf), dtype=np.int64)
        con[s1] = np.arange(self.nf)[:, None] * self.npf + np.arange(self.npf)
        a, b = xf[s1[:len(second)]], xf[second]
        key = lambda x: np.lexsort([np.round(x[..., k] * 1e6) for k in range(nd)], axis=-1)  # noqa: E731
        ia, ib = key(a), key(b)
        rows = np.arange(len(second))[:, None]
        tmp = np.empty_like(ia)
        tmp[rows, ib] = np.arange(len(second))[:, None] * self.npf + ia
        con[second] = tmp
        self.con = T(con.reshape(self.ne, self.ndf))
        side_bc = np.zeros(self.ne * nfe, dtype=np.int64)
        side_bc[bnd] = bc
        types, self.type_of = np.unique(side_bc.reshape(self.ne, nfe), axis=0, return_inverse=True)
        self.type_of = T(self.type_of.reshape(-1))

        # local matrices of an element
        phi, dphi = T(m["shapeg"][0]), [T(g) for g in m["shapeg"][1:]]
        e0 = T(xdg[0])
        J = torch.stack([g @ e0 for g in dphi], 1)                      # [g, a, b] = dx_b / dxi_a
        w = T(m["gwe"]) * torch.linalg.det(J)
        Ji = torch.linalg.inv(J)
        grad = [sum(Ji[:, b_, a_, None] * dphi[a_] for a_ in range(nd)) for b_ in range(nd)]
        M = phi.T @ (w[:, None] * phi)
        C = [g.T @ (w[:, None] * phi) for g in grad]
        P = torch.zeros(self.ndf, self.npe, dtype=torch.float64, device=self.dev)
        P[torch.arange(self.ndf, device=self.dev), T(perm.reshape(-1))] = 1.0
        F0, Fd, gwf = T(m["shapfg"][0]), [T(g) for g in m["shapfg"][1:]], T(m["gwf"])
        Tm = torch.zeros(self.ndf, self.ndf, dtype=torch.float64, device=self.dev)
        nrm = torch.zeros(nd, self.ndf, dtype=torch.float64, device=self.dev)
        for l in range(nfe):
            xl = e0[T(perm[l])]
            tan = [(g @ xl) for g in Fd]
            n_ = torch.stack([tan[0][:, 1], -tan[0][:, 0]], 1) if nd == 2 else torch.linalg.cross(tan[0], tan[1])
            jac = n_.norm(dim=1)
            r = slice(l * self.npf, (l + 1) * self.npf)
            Tm[r, r] = F0.T @ ((gwf * jac)[:, None] * F0)
            nrm[:, r] = (n_[0] / jac[0])[:, None]
        E = [P.T @ (nrm[k][:, None] * Tm) for k in range(nd)]
        MC, ME = [torch.linalg.solve(M, c) for c in C], [torch.linalg.solve(M, e) for e in E]
        cn = sum(vel[k] * nrm[k] for k in range(nd))
        face = [kappa * (P.T @ (nrm[k][:, None] * (Tm @ P)) - C[k]) for k in range(nd)]
        D = sum(-vel[k] * C[k] + face[k] @ MC[k] for k in range(nd)) + tau * P.T @ Tm @ P
        F = P.T @ ((cn - tau)[:, None] * Tm) - sum(face[k] @ ME[k] for k in range(nd))
        qn = [kappa * nrm[k][:, None] * (Tm @ P) for k in range(nd)]
        K0 = sum(qn[k] @ MC[k] for k in range(nd)) + tau * Tm @ P
        H0 = -sum(qn[k] @ ME[k] for k in range(nd)) - tau * Tm
        self.DF, self.D, self.MC, self.ME, self.w, self.phi = torch.linalg.solve(D, F), D, MC, ME, w, phi
        rowbc = T(np.repeat(types, self.npf, axis=1))                   # [types, ndf]
        self.K, self.H = [], []
        for k in range(types.shape[0]):
            wall = (rowbc[k] == 1)[:, None]
            K = torch.where(wall, torch.zeros_like(K0), K0)
            conv = torch.where((rowbc[k] == 0)[:, None], cn[:, None] * Tm, torch.zeros_like(Tm))
            Hk = torch.where(wall, -tau * Tm, H0 + conv)
            self.K.append(K)
            self.H.append(Hk - K @ self.DF)
        self.N = self.nf * self.npf
        self.groups = [torch.nonzero(self.type_of == k)[:, 0] for k in range(types.shape[0])]

    def _conditions(self, x):
        """Boundary condition of each boundary face, from its vertices x[face, vertex, nd]."""
        if self.case["problem"] != "cd3d":
            return np.ones(len(x), dtype=np.int64)
        planes = [(0, 0.0)]
        if self.case["kind"] == "batch":                                # u = 0 on every inflow face
            planes = [(i, 0.0 if self.d["vel"][i] > 0 else 1.0) for i in range(3)]
        on = np.zeros(len(x), dtype=bool)
        for i, c in planes:
            on |= np.all(np.abs(x[:, :, i] - c) < 1e-8, axis=1)
        return np.where(on, 1, 2)

    def sources(self):
        """The load vectors (s, w) of each component: [components][ne, npe]."""
        T = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=self.dev)  # noqa: E731
        wphi = self.w[:, None] * self.phi
        if self.case["problem"] == "cd3d":
            odg = np.random.default_rng(self.d["seed"]).uniform(-1.0, 1.0, size=(self.ne, self.npe, 2))
            return [(T(odg[:, :, c]) @ self.phi.T) @ wphi for c in range(2)]
        xg = torch.einsum("gi,eid->egd", self.phi, T(self.xdg))
        if self.case["problem"] == "poisson":
            s = self.nd * np.pi ** 2 * torch.sin(np.pi * xg).prod(dim=2)
        else:
            s = torch.sin(self.d["k"] * np.pi * xg[..., 0]) * torch.cos(self.d["k"] * np.pi * xg[..., 1])
        return [s @ wphi]

    def gather(self, we):
        out = torch.zeros(self.N, dtype=torch.float64, device=self.dev)
        return out.index_add_(0, self.con.reshape(-1), we.reshape(-1))

    def matvec(self, v):
        ve, we = v[self.con], torch.empty(self.ne, self.ndf, dtype=torch.float64, device=self.dev)
        for g, H in zip(self.groups, self.H):
            we[g] = ve[g] @ H.T
        return self.gather(we)

    def load(self, s):
        u = torch.linalg.solve(self.D, s.T).T
        we = torch.empty(self.ne, self.ndf, dtype=torch.float64, device=self.dev)
        for g, K in zip(self.groups, self.K):
            we[g] = u[g] @ K.T
        return u, -self.gather(we)

    def solve(self, b, tol=1e-13, cycle=300, cycles=20):
        """GMRES with the face blocks' inverses, restarted until the residual is at rounding."""
        npf, f = self.npf, self.con.reshape(self.ne, -1, self.npf)
        B = torch.zeros(self.nf, npf * npf, dtype=torch.float64, device=self.dev)
        for g, H in zip(self.groups, self.H):
            for l in range(f.shape[1]):
                fc = f[g, l]
                at = fc % npf
                blk = H[l * npf:(l + 1) * npf, l * npf:(l + 1) * npf]
                B.scatter_add_(0, (fc[:, :1] // npf).expand(-1, npf * npf),
                               torch.zeros(len(g), npf * npf, dtype=torch.float64, device=self.dev).scatter_(
                                   1, (at[:, :, None] * npf + at[:, None, :]).reshape(len(g), -1),
                                   blk.reshape(1, -1).expand(len(g), -1).contiguous()))
        Bi = torch.linalg.inv(B.reshape(self.nf, npf, npf))
        pre = lambda r: (Bi * r.reshape(self.nf, 1, npf)).sum(2).reshape(-1)  # noqa: E731
        x, nb = torch.zeros_like(b), float(b.norm())
        V = torch.empty(cycle + 1, self.N, dtype=torch.float64, device=self.dev)
        for _ in range(cycles):
            r = b - self.matvec(x)
            if float(r.norm()) <= tol * nb:
                break
            r = pre(r)
            beta = float(r.norm())
            V[0] = r / beta
            h = torch.zeros(cycle + 1, cycle, dtype=torch.float64, device=self.dev)
            k = 0
            for k in range(cycle):
                w = pre(self.matvec(V[k]))
                for _pass in range(2):
                    c = V[:k + 1] @ w
                    w -= c @ V[:k + 1]
                    h[:k + 1, k] += c
                h[k + 1, k] = w.norm()
                V[k + 1] = w / h[k + 1, k]
                if k % 25 == 24 or k + 1 == cycle:
                    y, res = _least(h[:k + 2, :k + 1], beta)
                    if res < 1e-2 * tol * beta or k + 1 == cycle or not np.isfinite(res):
                        break
            y, _ = _least(h[:k + 2, :k + 1], beta)
            x = x + y @ V[:k + 1]
        return x

    def fields(self, u0, uh):
        """u and q = -grad u of a trace, as the framework stores them: [ne, 1 + nd, npe]."""
        e = uh[self.con]
        u = u0 - e @ self.DF.T
        return torch.stack([u] + [u @ c.T - e @ f.T for c, f in zip(self.MC, self.ME)], 1)


def _least(h, beta):
    H = h.cpu().numpy()
    rhs = np.zeros(H.shape[0])
    rhs[0] = beta
    y = np.linalg.lstsq(H, rhs, rcond=None)[0]
    return torch.as_tensor(y, device=h.device), float(np.linalg.norm(H @ y - rhs))


def _interleave(parts):
    """Component c of node i at c + ncu*i."""
    return torch.stack(parts, -1).reshape(-1)


def exact(case, seed):
    if case["problem"] == "ns2d":          # a nonlinear system: its Newton solves take minutes in plain torch
        return None
    inst = _instances(case, seed)
    if case["kind"] in ("matvec", "gmres", "assemble"):
        X = _Exact(case, inst[0])
        ncu = 2 if case["problem"] == "cd3d" else 1
        if case["kind"] == "assemble":
            b = _interleave([X.load(s)[1] for s in X.sources()])
            if case["precision"]:
                return [b]
            eye = torch.eye(ncu, dtype=torch.float64, device=X.dev)
            # H[t', t] column-major with t = c + ncu*node; DinvF[r, t] with r = i + npe*c
            H = [torch.einsum("ts,cd->sdtc", h, eye).reshape(-1) for h in X.H]
            F = torch.einsum("it,cd->tdci", -X.DF, eye).reshape(-1)
            return [b, torch.stack(H)[X.type_of].reshape(-1), F.repeat(X.ne)]
        v = torch.as_tensor(_vector(ncu * X.N, seed), device=X.dev).reshape(-1, ncu)
        f = X.matvec if case["kind"] == "matvec" else X.solve
        return _interleave([f(v[:, c].contiguous()) for c in range(ncu)])
    udg, uh = [], []
    for d in inst:
        X = _Exact(case, d)
        parts = []
        for s in X.sources():
            u0, b = X.load(s)
            x = X.solve(b)
            parts.append((X.fields(u0, x), x))
        # udg [npe, nc, ne] with the components of u, then of q_x, q_y, ..
        udg.append(torch.stack([f for f, _ in parts], 2).reshape(-1))
        uh.append(_interleave([x for _, x in parts]))
    return [torch.cat(udg), torch.cat(uh)]
