"""The Arnoldi step's kernels (krylov.hip) over the vector lengths where their forms change: a vector in
one workgroup (MGS up to 8192 entries, one problem), one chunk, the last chunk and piece partly filled,
sums repeated by every block and sums with a launch of their own (MGS beyond 1024 chunks of 512, CGS
beyond 256); Hessenberg columns staged in LDS and not (restart above 127); and restarts.  Every form runs the
same algorithm: the counts of equal restarts agree, and the solutions to the solve's tolerance."""
import numpy as np
import pytest
import torch

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


@pytest.mark.parametrize("kw", [dict(n=2, porder=1, pgauss=2), dict(n=32, porder=3, pgauss=6),
                                dict(n=17, porder=3, pgauss=6, nd=3), dict(n=20, porder=4, pgauss=8, nd=3),
                                dict(n=24, porder=4, pgauss=8, nd=3)])
@pytest.mark.parametrize("ortho", [0, 1])
def test_steps(tmp_path, kw, ortho):
    """The solution after k steps against the minimiser over the same Krylov space, formed with torch and
    orthogonalised twice: k where the dots' and the update's waves take other shares of the vectors, on one
    chunk, many, and enough for the norm's partials to be summed in groups (MGS beyond 1,048,576 entries, CGS
    beyond 131,072)."""
    from exasim_amd import cases
    from exasim_amd.hdg import HDGSolver
    cases.poisson2d(str(tmp_path), model="poisson_poly", precond="eas", gmres_tol=1e-14, ortho=ortho, **kw)
    eps = np.finfo(float).eps
    with HDGSolver(str(tmp_path), "poisson_poly") as S:
        S.get_q()
        S.assemble()
        N = S.sizes["N"]
        b = torch.from_numpy(np.random.default_rng(N).standard_normal(N)).cuda()

        def product(v):
            w = torch.empty_like(v)
            torch.cuda.synchronize()
            S.matvec(v.data_ptr(), w.data_ptr())
            S.precond(w.data_ptr())
            S.sync()
            return w
        steps = [k for k in (1, 3, 4, 5, 8, 9, 12, 13, 16, 17, 33) if k <= N // 2]
        z = b.clone()
        torch.cuda.synchronize()
        S.precond(z.data_ptr())
        S.sync()
        V, H, beta = [z / z.norm()], np.zeros((steps[-1] + 1, steps[-1])), float(z.norm())
        for k in range(steps[-1]):
            w = product(V[k])
            for _ in range(2):
                for i, v in enumerate(V):
                    h = torch.dot(v, w)
                    H[i, k] += float(h)
                    w = w - h * v
            H[k + 1, k] = float(w.norm())
            V.append(w / w.norm())
        for k in steps:
            h = H[:k + 1, :k]
            y = np.linalg.lstsq(h, beta * np.eye(k + 1)[0], rcond=None)[0]
            ref = sum(float(c) * v for c, v in zip(y, V))
            S.set_option("gmres_maxit", k)
            x = torch.zeros_like(b)
            torch.cuda.synchronize()
            S.gmres(b.data_ptr(), x.data_ptr())
            S.sync()
            # orthogonalised once, the basis is orthogonal to about eps cond^2 (CGS) or eps cond (MGS), cond the
            # projected operator's, and the solution over it moves by as much; N-term sums keep well below N eps
            c = np.linalg.cond(h)
            print(kw, "ortho", ortho, "k", k, "cond", c, "err", float((x - ref).norm() / ref.norm()), flush=True)
            assert float((x - ref).norm()) <= 10 * k * eps * c ** 2 * float(ref.norm())


@pytest.mark.parametrize("ortho", [0, 1])
def test_batch_with_a_long_instance(tmp_path, ortho):
    """An instance's sums do not depend on the batch it is in: a short one beside others whose norm is long enough
    to be summed in groups (157,920 entries and more), and all of them where the batch's chunks (1,070) give one
    wave a piece of the update and the instances' own (404 at most) four."""
    from exasim_amd import cases
    from exasim_amd.hdg import HDGSolver
    paths = []
    for n in (16, 140, 150, 160):
        paths.append(str(tmp_path / str(n)))
        cases.poisson2d(paths[-1], n=n, porder=3, pgauss=6, model="poisson_poly", precond="eas", gmres_tol=1e-10,
                        restart=60, gmres_maxit=300, ortho=ortho)
    alone = []
    for p in paths:
        with HDGSolver.batch([p], "poisson_poly") as S:
            S.solve()
            alone.append(S.get("uh"))
    with HDGSolver.batch(paths, "poisson_poly") as S:
        S.solve()
        assert np.array_equal(S.get("uh"), np.concatenate(alone))
