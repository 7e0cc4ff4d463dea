"""The one-wave LU of matrices below 64 rows (lu.hip, k_lu_small): rows that are one, few and all but one of the lanes,
each register width (augmented columns up to 16, 32, 48, 64 and 96), right-hand sides split over several waves
with a narrow last one, and blocks whose pivots are off the diagonal.  Assembled matrices, their solves against the
oracle through D^{-1} F, and the inverted face blocks against their inverses."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # builder, arguments, n, m, ncf
    ("poisson2d", dict(n=3, porder=1, pgauss=2, elemtype=0), 3, 6, 2),
    ("poisson2d", dict(n=3, porder=2, pgauss=4), 9, 12, 3),
    ("poisson2d", dict(n=3, porder=3, pgauss=6, elemtype=0), 10, 12, 4),
    ("poisson2d", dict(n=3, porder=4, pgauss=8), 25, 20, 5),
    ("poisson2d", dict(n=3, porder=5, pgauss=10), 36, 24, 6),
    ("poisson2d", dict(n=2, porder=6, pgauss=12), 49, 28, 7),
    ("poisson2d", dict(n=2, porder=2, pgauss=4, nd=3), 27, 54, 9),
    ("convdiff3d", dict(n=2, porder=2), 54, 108, 18),
    ("navierstokes2d", dict(nx=3, ny=2, porder=2, nsteps=1, cartgridpart=False), 36, 48, 12),
]


@pytest.mark.parametrize("builder,kw,n,m,ncf", CASES)
def test_solves(tmp_path, builder, kw, n, m, ncf):
    from exasim_amd import cases
    from exasim_amd.hdg import HDGSolver
    from oracle import hdg as ora
    info = getattr(cases, builder)(str(tmp_path), precond="bjacobi", **kw)
    P = ora.HDGProblem(str(tmp_path), info["model"])
    P.get_q(P.udg, P.uh)
    _, S, _ = P.assemble()
    F = S["DinvF"].transpose(0, 2, 1).reshape(-1)
    cond = max(np.linalg.cond(d) for d in S["D"])
    eps = 2.0 ** -53
    print(builder, kw, "cond", cond, flush=True)
    with HDGSolver(str(tmp_path), info["model"]) as G:
        assert (G.sizes["n"], G.sizes["m"], info["npf"] * info["ncu"]) == (n, m, ncf)
        G.get_q()
        G.assemble()
        # backward stability with partial pivoting (growth n at worst here) and the assembly's own rounding
        assert np.abs(G.get("DinvF") - F).max() < 10 * n * cond * eps * np.abs(F).max()
        B = G.get("BE").reshape(-1, ncf, ncf).transpose(0, 2, 1)
        # the face blocks: H's face parts summed over each face's elements, in the face's own node order
        con = G.get("elemcon").astype(int).reshape(-1, m // info["ncu"])
        H = G.get("H").reshape(-1, m, m).transpose(0, 2, 1)
        K = np.zeros_like(B)
        for e in range(H.shape[0]):
            for l in range(m // ncf):
                nodes = con[e, l * info["npf"]:(l + 1) * info["npf"]]
                f, j = nodes[0] // info["npf"], nodes % info["npf"]
                idx = (j[:, None] * info["ncu"] + np.arange(info["ncu"])).reshape(-1)
                K[f][np.ix_(idx, idx)] += H[e, l * ncf:(l + 1) * ncf, l * ncf:(l + 1) * ncf]
        for f in range(len(K)):
            c = np.linalg.cond(K[f])
            assert np.abs(B[f] @ K[f] - np.eye(ncf)).max() < 10 * ncf * c * eps


def test_no_workspace(tmp_path):
    """Matrices below 64 FP64 rows take no workspace: a handle of many small elements holds its fields, geometry,
    element blocks and Krylov basis (13.7 KB per element here), and the inversion of the face blocks allocates
    nothing.  (A pivot workspace per matrix was 1 KB, one for triangle inverses 32 KB.)"""
    from exasim_amd import cases
    from exasim_amd.hdg import HDGSolver
    info = cases.poisson2d(str(tmp_path), n=200, porder=1, pgauss=2, precond="bjacobi")
    torch.cuda.synchronize()
    free = [torch.cuda.mem_get_info()[0]]
    with HDGSolver(str(tmp_path), info["model"]) as S:
        S.sync()
        free.append(torch.cuda.mem_get_info()[0])
        S.get_q()
        S.assemble()
        S.sync()
        free.append(torch.cuda.mem_get_info()[0])
        z = S.sizes
    print("created", free[0] - free[1], "assembled", free[1] - free[2], z, flush=True)
    assert free[0] - free[1] < 18e3 * z["ne"]
    assert free[1] - free[2] < 128 * z["nf"]
