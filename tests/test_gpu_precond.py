"""The block-Jacobi apply over the face block sizes ncf where its loads and lanes change (1, 2 and 4 rows per
load; one and four waves per block), FP64 and FP32, against numpy; and the Krylov step's P A v, which sums the
element products as the preconditioner reads them, against the operator and the preconditioner applied one
after the other."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # builder arguments, ncf
    ("poisson2d", dict(n=5, porder=1, pgauss=2), 2),
    ("poisson2d", dict(n=3, porder=2, pgauss=4, elemtype=0), 3),
    ("poisson2d", dict(n=2, porder=3, pgauss=6, nd=3), 16),
    ("convdiff3d", dict(n=2, porder=2), 18),
    ("convdiff3d", dict(n=2, porder=5, pgauss=10), 72),
]


@pytest.mark.parametrize("builder,kw,ncf", CASES)
@pytest.mark.parametrize("mixed", [0, 1])
def test_preconditioned_product(tmp_path, builder, kw, ncf, mixed):
    from exasim_amd import cases
    from exasim_amd.hdg import HDGSolver
    info = getattr(cases, builder)(str(tmp_path), **kw)
    eps = np.finfo(float).eps
    for precond in (0, 1) if ncf < 72 else (0,):  # Schwarz blocks have at most 400 rows
        print(builder, kw, "precision", mixed, "preconditioner", precond, flush=True)
        with HDGSolver(str(tmp_path), info["model"]) as S:
            S.set_option("preconditioner", precond)
            S.set_option("precision", mixed)
            S.set_option("gmres_maxit", 1)
            S.set_option("gmres_tol", 1e-14)
            S.get_q()
            S.assemble()
            N = S.sizes["N"]
            assert info["npf"] * info["ncu"] == ncf
            b = torch.from_numpy(np.random.default_rng(ncf).standard_normal(N)).cuda()
            z, w, x = b.clone(), torch.empty_like(b), torch.zeros_like(b)
            torch.cuda.synchronize()
            S.precond(z.data_ptr())
            S.sync()
            if precond == 0:
                B = S.get("BE").reshape(-1, ncf, ncf).transpose(0, 2, 1)
                B = B.astype(np.float32).astype(float) if mixed else B
                v = b.cpu().numpy().reshape(-1, ncf)
                ref, a = np.einsum("fij,fj->fi", B, v), np.einsum("fij,fj->fi", np.abs(B), np.abs(v))
                # ncf products and their sums, on both sides
                assert np.all(np.abs(z.cpu().numpy().reshape(-1, ncf) - ref) <= (ncf + 2) * eps * a + 1e-300)
            beta = z.norm()
            v0 = z / beta
            torch.cuda.synchronize()
            S.matvec(v0.data_ptr(), w.data_ptr())
            S.sync()
            S.precond(w.data_ptr())
            S.gmres(b.data_ptr(), x.data_ptr())
            S.sync()
            # one step from zero: x = v0 beta <w, v0> / <w, w> with w = P A v0.  The gather adds the same two
            # values in the same order, so w differs by the rounding of v0 alone (it is scaled by 1 / beta there:
            # eps per entry, times at most the condition below); the two sums are within N eps of |w| and |w|^2
            xr = v0 * (beta * torch.dot(w, v0) / torch.dot(w, w))
            tol = 4 * (N + S.sizes["m"]) * eps * beta / w.norm() * cond(S, w, v0)
            assert float((x - xr).norm()) <= float(tol)


def cond(S, w, v0):
    """max over random directions of |P A u| / |P A v0|: what a rounding of v0 is multiplied by."""
    g = torch.Generator(device="cpu").manual_seed(1)
    c = 1.0
    for _ in range(4):
        u = torch.randn(len(v0), dtype=torch.float64, generator=g).cuda()
        u /= u.norm()
        t = torch.empty_like(u)
        torch.cuda.synchronize()
        S.matvec(u.data_ptr(), t.data_ptr())
        S.sync()
        S.precond(t.data_ptr())
        S.sync()
        c = max(c, float(t.norm() / w.norm()))
    return c
