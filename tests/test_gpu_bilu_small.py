"""The block-ILU(0) apply with one wave per superelement for small face blocks (bilu.hip) against the
256-thread kernel on the same factors: block rows of 2 to 32 (one to eight columns per lane, idle lanes,
blocks of fewer columns than the lanes cover), odd sizes (one row per lane), programs shorter than the
blocks loaded ahead and longer than 64 entries, FP64, FP32 and BF16 factors.  The shape rule's answer is checked
with each: a shape it left to the 256-thread kernel would compare that with itself."""
import ctypes

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
    ("navierstokes2d", dict(nx=8, ny=8, porder=6, nsteps=1), 28),
    ("navierstokes2d", dict(nx=64, ny=32, porder=7, nsteps=1), 32),
    ("poisson2d", dict(n=4, porder=4, pgauss=8, nd=3, cartgridpart=[3, 4, 4, 4, 2, 2, 2, 0]), 25),
]


def columns_per_lane(z, ncf, size):
    from exasim_amd import hdg
    f = hdg.load()._ZN3exa18bilu_small_columnsEiiiii
    f.restype = ctypes.c_int
    # a block of the factors occurs once in the sweeps' program
    return f(ncf, size, z["ilu_nse"], z["ilu_nfse"], z["ilu_nnz"])


def expected(ncf, size, nse):
    """Two rows per lane in even sizes, one in odd ones; at most 7 columns per lane, and 8 in the smaller types on
    512 superelements or more."""
    parts = 64 // (ncf // 2 if ncf % 2 == 0 else ncf)
    c = -(-ncf // parts)
    return c if c < 8 or (c == 8 and size < 8 and nse >= 512) else 0


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
            z, size = S.state(), (2 if bf16 else 4) if precision else 8
            assert columns_per_lane(z, ncf, size) == expected(ncf, size, z["ilu_nse"])
            z["N"] = S.sizes["N"]
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
