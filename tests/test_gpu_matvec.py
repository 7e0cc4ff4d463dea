"""The element products (matvec.hip) against numpy over the trace block sizes m where the kernels
differ: loads of 1, 2 and 4 rows per lane (odd m, m = 2 mod 4, multiples of 4), one and four waves per
element, several columns per load (m < 64) and one, the last lanes idle, and the row-block kernel
above (m = 2 mod 4: its form of two rows per lane, in FP32 and BF16).  FP64 and FP32 operators, and the Schwarz blocks in FP64, FP32 and BF16 (8 rows per load)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # builder arguments, m
    ("poisson2d", dict(n=3, porder=2, pgauss=4, elemtype=0), 9),
    ("poisson2d", dict(n=5, porder=1, pgauss=2), 8),
    ("poisson2d", dict(n=3, porder=4, pgauss=8, elemtype=0), 15),
    ("poisson2d", dict(n=5, porder=5, pgauss=10), 24),
    ("poisson2d", dict(n=3, porder=7, pgauss=14), 32),
    ("poisson2d", dict(n=2, porder=2, pgauss=4, nd=3), 54),
    ("poisson2d", dict(n=2, porder=3, pgauss=6, nd=3), 96),
    ("convdiff3d", dict(n=2, porder=2), 108),
    ("poisson2d", dict(n=2, porder=4, pgauss=8, nd=3), 150),
    ("convdiff3d", dict(n=2, porder=3), 192),
    ("convdiff3d", dict(n=2, porder=4), 300),
]


def products(blocks, con, ncu, N, v):
    """sum_e scatter(blocks_e gather_e(v)), and the same with absolute values (for the bound)."""
    ne, m = blocks.shape[0], blocks.shape[1]
    idx = (con.reshape(ne, -1)[:, :, None] * ncu + np.arange(ncu)).reshape(ne, m)
    w, a = np.zeros(N), np.zeros(N)
    np.add.at(w, idx, np.einsum("eij,ej->ei", blocks, v[idx]))
    np.add.at(a, idx, np.einsum("eij,ej->ei", np.abs(blocks), np.abs(v[idx])))
    return w, a


@pytest.mark.parametrize("builder,kw,m", CASES)
def test_element_products(tmp_path, builder, kw, m):
    from exasim_amd import cases
    from exasim_amd.hdg import HDGSolver
    info = getattr(cases, builder)(str(tmp_path), precond="eas", **kw)
    eps = np.finfo(float).eps
    for mixed, bf16 in ((0, 0), (1, 0), (1, 1)):
        print(builder, kw, "precision", mixed, "bf16 blocks", bf16, flush=True)
        with HDGSolver(str(tmp_path), info["model"]) as S:
            S.set_option("precision", mixed)
            S.set_option("precond_bf16", bf16)
            S.get_q()
            S.assemble()
            z = S.sizes
            assert z["m"] == m
            con = S.get("elemcon").astype(np.int64)
            v = np.random.default_rng(m).standard_normal(z["N"])
            vd = torch.from_numpy(v).cuda()
            wd, pd = torch.empty_like(vd), vd.clone()
            torch.cuda.synchronize()
            S.matvec(vd.data_ptr(), wd.data_ptr())
            S.precond(pd.data_ptr())
            S.sync()
            H = S.get("H").reshape(z["ne"], m, m).transpose(0, 2, 1)
            B = S.get("BEeas").reshape(z["ne"], m, m).transpose(0, 2, 1)
            if bf16:  # round to nearest even on the upper 16 bits
                u = B.astype(np.float32).view(np.uint32)
                u = (u + 0x7FFF + ((u >> 16) & 1)) & np.uint32(0xFFFF0000)
                B = u.view(np.float32).astype(np.float64)
            for blocks, out in ((H, wd), (B, pd)):
                w, a = products(blocks, con, z["ncu"], z["N"], v)
                # m products and sums of one element and the two sides' sum, each within eps/2
                assert np.all(np.abs(out.cpu().numpy() - w) <= (m + 2) * eps * a + 1e-300)


@pytest.mark.parametrize("mixed", [0, 1])
def test_operator_of_large_blocks(tmp_path, mixed):
    """m = 432: four row blocks in FP64, two in FP32 (Schwarz blocks have at most 400 rows)."""
    from exasim_amd import cases
    from exasim_amd.hdg import HDGSolver
    info = cases.convdiff3d(str(tmp_path), n=2, porder=5, precond="bjacobi")
    m = 432
    with HDGSolver(str(tmp_path), info["model"]) as S:
        S.set_option("precision", mixed)
        S.get_q()
        S.assemble()
        z = S.sizes
        assert z["m"] == m
        v = np.random.default_rng(m).standard_normal(z["N"])
        vd = torch.from_numpy(v).cuda()
        wd = torch.empty_like(vd)
        torch.cuda.synchronize()
        S.matvec(vd.data_ptr(), wd.data_ptr())
        S.sync()
        H = S.get("H").reshape(z["ne"], m, m).transpose(0, 2, 1)
        w, a = products(H, S.get("elemcon").astype(np.int64), z["ncu"], z["N"], v)
        assert np.all(np.abs(wd.cpu().numpy() - w) <= (m + 2) * np.finfo(float).eps * a + 1e-300)
