"""The elimination of q from the trace rows over the face nodes alone (gemm.hip, k_face_elim) against
the oracle's dense elimination: faces of less than one 16-row tile up to more than one 64-row tile, K
loops shorter than a block and with remainders, tensor and simplex elements, one and several components,
element blocks of one and of several elements."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    ("poisson2d", dict(n=3, porder=1, pgauss=2), {}),
    ("poisson2d", dict(n=3, porder=3, pgauss=6, elemtype=0), {}),
    ("poisson2d", dict(n=2, porder=7, pgauss=14), {}),
    ("poisson2d", dict(n=2, porder=2, pgauss=4, nd=3, elemtype=0), {}),
    ("poisson2d", dict(n=2, porder=3, pgauss=6, nd=3), {}),
    ("convdiff3d", dict(n=2, porder=2), {}),
    ("convdiff3d", dict(n=2, porder=4), {}),
    ("convdiff3d", dict(n=2, porder=5), {}),
    ("convdiff3d", dict(n=3, porder=1), dict(workspace_bytes=1e5)),
    ("navierstokes2d", dict(nx=3, ny=2, porder=3, nsteps=1, cartgridpart=False), {}),
]


@pytest.mark.parametrize("builder,kw,options", CASES)
def test_trace_rows(tmp_path, builder, kw, options):
    from exasim_amd import cases
    from exasim_amd.hdg import HDGSolver
    from oracle import hdg as ora
    info = getattr(cases, builder)(str(tmp_path), precond="bjacobi", **kw)
    P = ora.HDGProblem(str(tmp_path), info["model"])
    P.get_q(P.udg, P.uh)
    _, S, _ = P.assemble()
    H = S["H"].transpose(0, 2, 1).reshape(-1)
    # FP64: rounding through the condensation (as the other assembly tests); FP32: its eps, amplified by
    # the element matrix D, which is scaled the same in every case
    for precision, tol in ((0, 1e-11), (1, 2e-4)):
        print(builder, kw, "precision", precision, flush=True)
        with HDGSolver(str(tmp_path), info["model"]) as G:
            for k, v in options.items():
                G.set_option(k, v)
            G.set_option("precision", precision)
            G.get_q()
            G.assemble()
            if options:
                assert G.sizes["ne"] > G.state()["neb"]
            assert np.abs(G.get("H") - H).max() < tol * np.abs(H).max()
