"""The Arnoldi step's kernels (krylov.hip) over the vector lengths where their forms change: a vector in
one workgroup (MGS up to 8192 entries, one problem), one chunk, the last chunk and piece partly filled,
sums repeated by every block and sums with a launch of their own (MGS beyond 1024 chunks of 512, CGS
beyond 256); Hessenberg columns staged in LDS and not (restart above 127); and restarts.  Every form runs the
same algorithm: the counts of equal restarts agree, and the solutions to the solve's tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    dict(n=2, porder=1, pgauss=2),                 # 24 entries
    dict(n=16, porder=3, pgauss=6),                # 2,176
    dict(n=31, porder=3, pgauss=6),                # 7,936: the longest of these in one workgroup
    dict(n=32, porder=3, pgauss=6),                # 8,448
    dict(n=60, porder=4, pgauss=8),                # 36,600
    dict(n=17, porder=3, pgauss=6, nd=3),          # 249,696
    dict(n=20, porder=4, pgauss=8, nd=3),          # 630,000
]


@pytest.mark.parametrize("kw", CASES)
@pytest.mark.parametrize("ortho", [0, 1])
def test_forms_agree(tmp_path, kw, ortho):
    from exasim_amd import cases
    from exasim_amd.hdg import HDGSolver
    # a constant-diffusion problem whose source is no eigenfunction of the preconditioned operator
    cases.poisson2d(str(tmp_path), model="poisson_poly", precond="eas", gmres_tol=1e-11, gmres_maxit=5000, restart=100,
                    ortho=ortho, **kw)
    out = []
    for batch in (False, True):
        for restart in (100, 130, 12):
            print(kw, "ortho", ortho, "batch handle", batch, "restart", restart, flush=True)
            S = HDGSolver.batch([str(tmp_path)], "poisson_poly") if batch else HDGSolver(str(tmp_path), "poisson_poly")
            with S:
                S.set_option("gmres_restart", restart)
                _, it, norm = S.solve()
                out.append((restart, it, norm, S.get("uh")))
                S.reset()
                _, again, _ = S.solve()
                assert again == it and np.array_equal(S.get("uh"), out[-1][3])
    ref = out[0]
    first = {}
    for restart, it, norm, uh in out:
        # one problem and a batch of one restart at the same steps: rounding moves the residual estimate at
        # the tolerance by far less than one step does; restarted after 12 the solves crawl (a step gains a few
        # per cent) and rounding may move the end by some of them
        assert abs(it - first.setdefault(restart, it)) <= (1 if restart != 12 else max(12, it // 20))
        # two solutions with residuals of 1e-11 differ by at most the condition number times that, which
        # grows as (p^2 / h)^2 ~ 1e5 at most over these meshes
        assert norm < 1e-8
        assert np.abs(uh - ref[3]).max() < 1e-6 * np.abs(ref[3]).max()
