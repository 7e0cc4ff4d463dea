"""The batched LU's one-wave panels (lu.hip) over the matrix sizes where they change: one to four rows per
lane (n up to 64, 128, 192, 256), a last panel of one column and of all, 64-, 32- and 16-column panels, and
more rows than the wave holds (the LDS panel).  The element matrices are assembled ones; their solves are
checked through D^{-1} F against the oracle, and in the mixed form the refinement's replay of the pivots
through the solution."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [  # builder, arguments, n
    ("convdiff3d", dict(n=2, porder=1, ncu=2), 16),
    ("navierstokes2d", dict(nx=2, ny=2, porder=3, nsteps=1, cartgridpart=False), 64),
    ("poisson2d", dict(n=2, porder=3, pgauss=6, nd=3), 64),
    ("navierstokes2d", dict(nx=2, ny=2, porder=4, nsteps=1, cartgridpart=False), 100),
    ("convdiff3d", dict(n=2, porder=3), 128),
    ("navierstokes2d", dict(nx=2, ny=2, porder=5, nsteps=1, cartgridpart=False), 144),
    ("navierstokes2d", dict(nx=2, ny=2, porder=6, nsteps=1, cartgridpart=False), 196),
    ("convdiff3d", dict(n=2, porder=4), 250),
    ("navierstokes2d", dict(nx=2, ny=2, porder=7, pgauss=14, nsteps=1, cartgridpart=False), 256),
    ("poisson2d", dict(n=1, porder=6, pgauss=12, nd=3), 343),
]


@pytest.mark.parametrize("builder,kw,n", CASES)
def test_condensation(tmp_path, builder, kw, n):
    from exasim_amd import cases
    from exasim_amd.hdg import HDGSolver
    from oracle import hdg as ora
    info = getattr(cases, builder)(str(tmp_path), precond="bjacobi", **kw)
    P = ora.HDGProblem(str(tmp_path), info["model"])
    P.get_q(P.udg, P.uh)
    _, S, _ = P.assemble()
    F = S["DinvF"].transpose(0, 2, 1).reshape(-1)
    cond = max(np.linalg.cond(d) for d in S["D"])
    for precision, eps in ((0, 2.0 ** -53), (1, 2.0 ** -24)):
        print(builder, kw, "n", n, "precision", precision, "cond", cond, flush=True)
        with HDGSolver(str(tmp_path), info["model"]) as G:
            G.set_option("precision", precision)
            assert G.sizes["n"] == n
            G.get_q()
            G.assemble()
            # backward stability with partial pivoting (growth n at worst here) and the assembly's own rounding
            assert np.abs(G.get("DinvF") - F).max() < n * cond * eps * np.abs(F).max()


@pytest.mark.parametrize("porder", [2, 3, 4, 5])
def test_refinement(tmp_path, porder):
    from exasim_amd import cases
    from exasim_amd.hdg import HDGSolver
    info = cases.navierstokes2d(str(tmp_path), nx=6, ny=4, porder=porder, nsteps=1, cartgridpart=False, precond="eas",
                                gmres_tol=1e-10, newton_tol=1e-10)
    out = []
    for precision in (0, 1):
        print("navierstokes2d 6x4 p", porder, "precision", precision, flush=True)
        with HDGSolver(str(tmp_path), info["model"]) as G:
            G.set_option("precision", precision)
            G.set_option("refine_first_tol", 1e-5)
            G.set_option("refine_tol", 1e-5)
            G.solve()
            out.append((G.get("udg"), G.state()["refinements"]))
    assert out[1][1] > 0
    # both forms stop at a Newton residual of 1e-10 (the mixed form's bound against FP64 elsewhere: 1e-8)
    assert np.abs(out[0][0] - out[1][0]).max() < 1e-8 * np.abs(out[0][0]).max()
