"""The face terms of the residual against the oracle where the kernel's shapes change: several elements per
workgroup with the last one partly filled, one element per workgroup, more entries than threads (m > 256),
and element blocks that end within a workgroup."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    ("poisson2d", dict(n=3, porder=1, pgauss=2), {}, 8),
    ("poisson2d", dict(n=5, porder=3, pgauss=6, elemtype=0), {}, 12),
    ("poisson2d", dict(n=3, porder=2, pgauss=4, nd=3), {}, 54),
    ("convdiff3d", dict(n=2, porder=3), {}, 192),
    ("convdiff3d", dict(n=2, porder=4), {}, 300),
    ("convdiff3d", dict(n=3, porder=1), dict(workspace_bytes=1e5), 48),
    ("navierstokes2d", dict(nx=5, ny=3, porder=3, nsteps=1, cartgridpart=False), {}, 64),
]


@pytest.mark.parametrize("builder,kw,options,m", CASES)
def test_residual(tmp_path, builder, kw, options, m):
    from exasim_amd import cases
    from exasim_amd.hdg import HDGSolver
    from oracle import hdg as ora
    info = getattr(cases, builder)(str(tmp_path), precond="bjacobi", **kw)
    P = ora.HDGProblem(str(tmp_path), info["model"])
    P.get_q(P.udg, P.uh)
    b, Ru = P.residual()[:2]
    print(builder, kw, flush=True)
    with HDGSolver(str(tmp_path), info["model"]) as S:
        for k, v in options.items():
            S.set_option(k, v)
        assert S.sizes["m"] == m
        S.get_q()
        S.residual()
        # sums of at most a few hundred products of values of the largest entries' size or less, which the
        # volume and face parts cancel: the bound of the other assembly tests
        for got, ref in ((S.get("res_b"), b), (S.get("res_Ru"), Ru)):
            assert np.abs(got.reshape(-1) - ref.reshape(-1)).max() < 1e-11 * max(1.0, np.abs(ref).max())
