"""GMRES steps replayed from HIP graphs (option gmres_graph) against the same steps queued one by one: the same
kernels on the same buffers, so counts and solutions are equal bit for bit.  Orthogonalisation in one workgroup,
by segments and of a batch, every preconditioner, the mixed form, cycles that end within the captured columns,
and several solves with other work between the replays."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # builder, arguments, options
    ("poisson2d", dict(n=16, porder=3, pgauss=6, precond="bjacobi"), {}),
    ("poisson2d", dict(n=33, porder=3, pgauss=6, precond="eas"), {}),
    ("poisson2d", dict(n=33, porder=3, pgauss=6, precond="eas", ortho=1), dict(gmres_restart=11)),
    ("poisson2d", dict(n=11, porder=3, pgauss=6, nd=3, precond="bjacobi", ortho=1), dict(gmres_restart=9)),
    ("convdiff3d", dict(n=4, porder=3, precond="bilu0", cartgridpart=[3, 4, 4, 4, 2, 2, 2, 0]), {}),
    ("convdiff3d", dict(n=4, porder=3, precond="eas", ortho=1), dict(precision=1, precond_bf16=1, gmres_restart=8)),
    ("convdiff3d", dict(n=4, porder=2, precond="bilu0", cartgridpart=[3, 4, 4, 4, 2, 2, 2, 0]),
     dict(precision=1, precond_bf16=1)),
]


def run(S, graph, options):
    for k, v in options.items():
        S.set_option(k, v)
    S.set_option("gmres_graph", graph)
    out = []
    for _ in range(3):
        S.reset()
        stats = S.solve()
        out.append((stats, S.get("uh"), S.get("udg")))
        S.residual()  # other work on the handle's buffers between the replays
        v = torch.randn(S.sizes["N"], dtype=torch.float64, device="cuda")
        w = torch.empty_like(v)
        torch.cuda.synchronize()
        S.matvec(v.data_ptr(), w.data_ptr())
        S.sync()
    return out


def same(a, b):
    for (sa, ua, qa), (sb, ub, qb) in zip(a, b):
        assert sa == sb and np.array_equal(ua, ub) and np.array_equal(qa, qb)
    assert np.isfinite(a[0][1]).all()


@pytest.mark.parametrize("builder,kw,options", CASES)
def test_replay(tmp_path, builder, kw, options):
    from exasim_amd import cases
    from exasim_amd.hdg import HDGSolver
    info = getattr(cases, builder)(str(tmp_path), **kw)
    print(builder, kw, options, flush=True)
    with HDGSolver(str(tmp_path), info["model"]) as S:
        eager = run(S, 0, options)
        replayed = run(S, 1, options)
        same(eager, replayed)
        same(eager[:1] * 3, eager)
        # another option drops the captured steps
        S.set_option("ortho", 1 - kw.get("ortho", 0))
        again = run(S, 1, {})
        same(run(S, 0, {}), again)


def test_replay_of_a_batch(tmp_path):
    from exasim_amd import cases
    from exasim_amd.hdg import HDGSolver
    paths = []
    for i, n in enumerate((8, 16, 24)):
        paths.append(str(tmp_path / str(i)))
        cases.convdiff2d_param(paths[-1], n=n, porder=3, kappa=10.0 ** -i, angle=0.3 + i, k=1 + i, precond="eas",
                               restart=20, ortho=1)
    with HDGSolver.batch(paths, "cd2d") as S:
        same(run(S, 0, {}), run(S, 1, {}))
