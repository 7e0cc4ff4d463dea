"""The block-ILU(0) apply with one wave per superelement for small face blocks (bilu.hip) against the
256-thread kernel on the same factors: block rows of 2 to 32 (one to eight columns per lane, idle lanes,
blocks of fewer columns than the lanes cover), odd sizes (one row per lane), programs shorter than the
blocks loaded ahead and longer than 64 entries, FP64, FP32 and BF16 factors."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # builder, arguments, ncf
    ("poisson2d", dict(n=2, porder=1, pgauss=2, cartgridpart=[2, 2, 2, 1, 1, 0]), 2),
    ("poisson2d", dict(n=4, porder=2, pgauss=4, cartgridpart=[2, 4, 4, 2, 2, 0]), 3),
    ("poisson2d", dict(n=4, porder=4, pgauss=8, cartgridpart=[2, 4, 4, 4, 4, 0]), 5),
    ("navierstokes2d", dict(nx=4, ny=4, porder=4, nsteps=1), 20),
    ("navierstokes2d", dict(nx=4, ny=4, porder=5, nsteps=1), 24),
    ("navierstokes2d", dict(nx=8, ny=8, porder=2, nsteps=1, se=4), 12),
    ("poisson2d", dict(n=2, porder=2, pgauss=4, nd=3, cartgridpart=[3, 2, 2, 2, 2, 2, 2, 0]), 9),
    ("convdiff3d", dict(n=2, porder=2, cartgridpart=[3, 2, 2, 2, 2, 2, 2, 0]), 18),
    ("convdiff3d", dict(n=4, porder=3, cartgridpart=[3, 4, 4, 4, 2, 2, 2, 0]), 32),
]


@pytest.mark.parametrize("builder,kw,ncf", CASES)
def test_apply(tmp_path, builder, kw, ncf):
    from exasim_amd import cases
    from exasim_amd.hdg import HDGSolver
    info = getattr(cases, builder)(str(tmp_path), precond="bilu0", **kw)
    # sums of at most a row of blocks in FP64; with FP32 and BF16 factors the row results are kept in FP32 and
    # a difference in their last bit passes through the later rows' sums
    for precision, bf16, tol in ((0, 0, 1e-12), (1, 0, 1e-5), (1, 1, 1e-5)):
        print(builder, kw, "precision", precision, "bf16", bf16, flush=True)
        with HDGSolver(str(tmp_path), info["model"]) as S:
            S.set_option("precision", precision)
            S.set_option("precond_bf16", bf16)
            z = S.sizes
            assert z["npf"] * z["ncu"] == ncf
            S.get_q()
            S.assemble()
            x = np.random.default_rng(ncf).standard_normal(z["N"])
            out = []
            try:
                for wave in (0, 1):
                    S.set_option("ilu_wave", wave)
                    xd = torch.from_numpy(x).cuda()
                    torch.cuda.synchronize()
                    S.precond(xd.data_ptr())
                    S.sync()
                    out.append(xd.cpu().numpy())
            finally:
                S.set_option("ilu_wave", -1)
            assert np.isfinite(out[0]).all()
            assert np.abs(out[1] - out[0]).max() < tol * np.abs(out[0]).max()
