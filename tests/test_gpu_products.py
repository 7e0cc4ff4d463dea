"""The dense kernels called by themselves on matrices of their own, against numpy in 64 bits: the batched
products (gemm.hip, k_gemm) over every tile, remainders of M, N and K, gathered and in-place operands and
padded leading dimensions; the one-column trace product (matvec.hip, k_trace_rhs); the batched LU with its
solves (lu.hip) by their backward error; and the refinement's solve with the FP32 factors, which replays their
row exchanges.  The entries are C++ functions of the library, called through their symbols."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

_P, _I, _L, _F = ctypes.c_void_p, ctypes.c_int, ctypes.c_long, ctypes.c_double


class Gemm(ctypes.Structure):
    _fields_ = ([(k, _I) for k in ("M", "N", "K")] + [("alpha", _F), ("beta", _F)]
                + [(k, t) for o in "ABC" for k, t in ((o, _P), ("ld" + o.lower(), _L), ("s%s0" % o, _L),
                                                      ("s%s1" % o, _L), ("s%s2" % o, _L))]
                + [(k, _I) for k in ("nb0", "nb1", "nb2")] + [(k, _P) for k in ("iA", "iB", "iC")]
                + [("fp32", _I)] + [(k, _P) for k in ("Af", "Bf", "Cf")])


class Dims(ctypes.Structure):
    _fields_ = [(k, _I) for k in ("nd", "ncu", "nc", "nco", "npe", "npf", "nfe", "nge", "ngf", "ne", "nf", "n", "m",
                                  "ncf", "ndf")] + [("N", _L)]


def call(symbol, *args):
    from exasim_amd import hdg
    lib = hdg.load()
    torch.cuda.synchronize()
    f = getattr(lib, symbol)
    f.restype = None
    f(*args)
    lib.hipDeviceSynchronize()


def ptr(t):
    return _P(t.data_ptr())


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def gemm(g, fp32, a, b, c):
    for o, t in zip("ABC", (a, b, c)):
        setattr(g, o + "f" if fp32 else o, t.data_ptr())
    g.fp32 = fp32
    call("_ZN3exa4gemmERKNS_4GemmEP12ihipStream_t", ctypes.byref(g), None)


@pytest.fixture(params=range(-1, 5))
def tile(request):
    call("_ZN3exa13set_gemm_tileEi", request.param)
    yield request.param
    call("_ZN3exa13set_gemm_tileEi", -1)


SHAPES = [(1, 1, 1), (3, 2, 5), (16, 16, 16), (15, 17, 15), (17, 15, 17), (33, 31, 3), (31, 65, 33), (64, 64, 64),
          (63, 1, 65), (65, 63, 4), (66, 40, 16), (129, 130, 31), (130, 66, 48), (5, 200, 100)]


def bound(K, eps, a, b, beta, c):
    """K products and sums, the scaling and the sum with C, each within eps / 2 of the terms' sizes."""
    return (K + 3) * eps * (np.abs(a) @ np.abs(b) + abs(beta) * np.abs(c))


@pytest.mark.parametrize("fp32", [0, 1])
def test_products(tile, fp32):
    dt = np.float32 if fp32 else np.float64
    eps = float(np.finfo(dt).eps)
    rng = np.random.default_rng(7)
    for M, N, K in SHAPES:
        for beta in (0.0, 1.0):
            # 3 x 2 products; A and C gathered through lists, B shared by the second batch index
            nb0, nb1, pa, pc = 3, 2, M + 3, M + 1
            A, B = rng.standard_normal((nb1, 5, K, pa)).astype(dt), rng.standard_normal((nb0, N, K + 2)).astype(dt)
            C = rng.standard_normal((nb1, 4, N, pc)).astype(dt)
            iA, iC = np.array([4, 0, 2], dtype=np.int32), np.array([1, 3, 0], dtype=np.int32)
            a, b, c, ia, ic = dev(A), dev(B), dev(C), dev(iA), dev(iC)
            print("tile", tile, "fp32", fp32, M, N, K, "beta", beta, flush=True)
            g = Gemm(M=M, N=N, K=K, alpha=-1.0, beta=beta, lda=pa, sA0=K * pa, sA1=5 * K * pa, ldb=K + 2,
                     sB0=N * (K + 2), sB1=0, ldc=pc, sC0=N * pc, sC1=4 * N * pc, nb0=nb0, nb1=nb1, nb2=1,
                     iA=ia.data_ptr(), iC=ic.data_ptr())
            gemm(g, fp32, a, b, c)
            got = c.cpu().numpy()
            want = C.copy()
            for b1 in range(nb1):
                for b0 in range(nb0):
                    Ab = A[b1, iA[b0], :, :M].T.astype(float)
                    Bb = B[b0, :, :K].T.astype(float)
                    Cb = C[b1, iC[b0], :, :M].T.astype(float)
                    r = -(Ab @ Bb) + (beta * Cb if beta else 0.0)
                    err = np.abs(got[b1, iC[b0], :, :M].T.astype(float) - r)
                    assert np.all(err <= bound(K, eps, Ab, Bb, beta, Cb)), (M, N, K, err.max())
                    want[b1, iC[b0], :, :M] = got[b1, iC[b0], :, :M]
            assert np.array_equal(got, want)  # rows of the padding and blocks that no list names


@pytest.mark.parametrize("fp32", [0, 1])
def test_products_in_place(tile, fp32):
    dt = np.float32 if fp32 else np.float64
    eps = float(np.finfo(dt).eps)
    rng = np.random.default_rng(8)
    for M, N in ((1, 3), (16, 40), (31, 65), (33, 100), (64, 130), (58, 301)):
        nb = 70
        A, X = rng.standard_normal((nb, M, M)).astype(dt), rng.standard_normal((nb, N, M + 5)).astype(dt)
        a, x = dev(A), dev(X)
        print("in place, tile", tile, "fp32", fp32, M, N, flush=True)
        g = Gemm(M=M, N=N, K=M, alpha=1.0, beta=0.0, lda=M, sA0=M * M, ldb=M + 5, sB0=N * (M + 5), ldc=M + 5,
                 sC0=N * (M + 5), nb0=nb, nb1=1, nb2=1)
        gemm(g, fp32, a, x, x)
        got = x.cpu().numpy()
        Ab, Xb = A.transpose(0, 2, 1).astype(float), X[:, :, :M].transpose(0, 2, 1).astype(float)
        assert np.all(np.abs(got[:, :, :M].transpose(0, 2, 1) - Ab @ Xb) <= bound(M, eps, Ab, Xb, 0.0, Xb))
        assert np.array_equal(got[:, :, M:], X[:, :, M:])


@pytest.mark.parametrize("kinds", ["dd", "ff", "fd"])
def test_trace_products(kinds):
    tk, tu = (np.float64 if k == "d" else np.float32 for k in kinds)
    rng = np.random.default_rng(9)
    # loads of 1, 2 and 4 rows; a column in part of a wave's loads, in one, in several; fewer columns than waves
    for m, n, ne in ((1, 1, 1), (3, 2, 5), (6, 3, 3), (8, 4, 9), (15, 25, 4), (54, 27, 3), (96, 64, 5), (150, 125, 3),
                     (192, 128, 2), (257, 33, 2), (300, 250, 3), (514, 7, 2)):
        K, U = rng.standard_normal((ne, n, m)).astype(tk), rng.standard_normal((ne, n + 3)).astype(tu)
        R = rng.standard_normal((ne, m))
        k, u, r = dev(K), dev(U), dev(R)
        print("trace product", kinds, m, n, ne, flush=True)
        d = Dims(m=m, n=n)
        call("_ZN3exa9trace_rhsI%sEEvRKNS_4DimsEiPKT_PKT0_lPdP12ihipStream_t" % kinds, ctypes.byref(d), _I(ne), ptr(k),
             ptr(u), _L(n + 3), ptr(r), None)
        Kb, ub = K.transpose(0, 2, 1).astype(float), U[:, :n, None].astype(float)
        ref, a = R - (Kb @ ub)[..., 0], np.abs(R) + (np.abs(Kb) @ np.abs(ub))[..., 0]
        assert np.all(np.abs(r.cpu().numpy() - ref) <= (n + 2) * np.finfo(float).eps * a), (m, n)


# one to four rows per lane (up to 64, 128, 192, 256), the LDS panel above; last panels of one column and of all;
# 64-, 32- and 16-column panels; below 64 FP64 rows the register widths of k_lu_small and their splits
LU_SIZES = [(1, 1), (2, 40), (3, 7), (9, 8), (16, 16), (25, 21), (25, 120), (36, 25), (63, 1), (63, 200), (64, 65),
            (65, 97), (100, 81), (128, 193), (129, 30), (144, 97), (192, 17), (193, 16), (196, 113), (250, 301),
            (256, 129), (257, 40), (343, 50)]


def factor(A, R, f32, pivots=False, inverses=False):
    """lu_solve on [A | R]: the factored matrix, the solutions, info and the panels' pivots."""
    nb, n, nr = A.shape[0], A.shape[1], R.shape[2]
    dt = np.float32 if f32 else np.float64
    aug = dev(np.concatenate([A, R], axis=2).transpose(0, 2, 1).astype(dt))
    info = torch.full((nb,), -1, dtype=torch.int32).cuda()
    piv = torch.full((nb, n), -1, dtype=torch.int32).cuda()
    ws = torch.zeros(nb * 260, dtype=torch.int32).cuda()
    tri = torch.zeros(nb * 64 * 64, dtype=torch.float64).cuda()
    call("_ZN3exa8lu_solveEP%siiliPiP12ihipStream_tS1_S1_Pv" % ("f" if f32 else "d"), ptr(aug), _I(n), _I(n + nr),
         _L(n * (n + nr)), _I(nb), ptr(info), None, ptr(piv) if pivots else None, ptr(ws), ptr(tri) if inverses else None)
    out = aug.cpu().numpy().transpose(0, 2, 1)
    return out[:, :, :n], out[:, :, n:].astype(float), info.cpu().numpy(), piv.cpu().numpy()


@pytest.mark.parametrize("f32,inverses", [(0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("n,nr", LU_SIZES)
def test_lu_backward_error(n, nr, f32, inverses):
    dt = np.float32 if f32 else np.float64
    eps = float(np.finfo(dt).eps)
    rng = np.random.default_rng(n + 1000 * nr)
    nb = 5
    A, R = (rng.standard_normal((nb, n, k)).astype(dt).astype(float) for k in (n, nr))
    A[0] = A[0][rng.permutation(n)] + 0.0
    A[1] *= 10.0 ** rng.uniform(-3, 3, (n, 1)).astype(float)  # rows of very different sizes
    A[1] = A[1].astype(dt).astype(float)
    print("lu", n, nr, "fp32" if f32 else "fp64", "inverses" if inverses else "", flush=True)
    LU, X, info, piv = factor(A, R, f32, inverses=inverses)
    assert np.all(info == 0)
    # the solutions solve a system within c n eps of the given one, whatever its condition: growth stays below 10
    # on these matrices with partial pivoting (inverted triangles: times a diagonal block's condition, some tens
    # where pivots are the columns' largest)
    c = 100.0 if inverses else 10.0
    big = np.abs(A).max(axis=(1, 2))[:, None, None]
    res = np.abs(A @ X - R).max(axis=1, keepdims=True)
    scale = n * big * np.abs(X).max(axis=1, keepdims=True) + np.abs(R).max(axis=1, keepdims=True)
    print("  backward error / eps", (res / scale).max() / eps, flush=True)
    assert np.all(res <= c * eps * scale)


def test_lu_tiny_pivots():
    """Pivots that have no finite reciprocal: the quotients are what the division gives."""
    n, nr = 5, 4
    rng = np.random.default_rng(3)
    T = np.triu(rng.uniform(1.0, 2.0, (n, n)), 0) * 2.0 ** -1030
    X0 = rng.integers(1, 9, (n, nr)).astype(float)
    T, R = np.diag(np.diag(T))[None], (np.diag(np.diag(T)) @ X0)[None]
    _, X, info, _ = factor(T, R, 0)
    assert info[0] == 0
    # the products carry the denormals' spacing 2^-1074 relative to 2^-1030
    assert np.all(np.abs(X[0] - X0) <= 2.0 ** -43 * X0 * 2)


@pytest.mark.parametrize("n", [1, 16, 63, 64, 65, 100, 128, 144, 192, 193, 250, 256, 257, 343])
def test_refinement_solve(n):
    """RuS = U^-1 L^-1 P Ru with the FP32 factors and the panels' pivots, in 64 bits; Rh -= K RuS."""
    m, ne = 33, 4
    rng = np.random.default_rng(n)
    A = rng.standard_normal((ne, n, n)).astype(np.float32).astype(float)
    LU, _, info, piv = factor(A, np.ones((ne, n, 1)), 1, pivots=True)
    assert np.all(info == 0) and np.all(piv >= 0)
    K, Ru, Rh = rng.standard_normal((ne, m, n)).astype(np.float32), rng.standard_normal((ne, n)), rng.standard_normal((ne, m))
    lu, pv, k, ru, rh = dev(LU.transpose(0, 2, 1)), dev(piv), dev(K.transpose(0, 2, 1)), dev(Ru), dev(Rh)
    rus = torch.full((ne, n), float("nan"), dtype=torch.float64).cuda()
    print("refinement solve n", n, flush=True)
    d = Dims(m=m, n=n, ne=ne)
    call("_ZN3exa10refine_rhsERKNS_4DimsEPKfPKiS4_PKdPdS9_P12ihipStream_t", ctypes.byref(d), ptr(lu), ptr(pv), ptr(k),
         ptr(ru), ptr(rus), ptr(rh), None)
    x = rus.cpu().numpy()
    # the panel width that the FP32 factorisation takes for n rows
    w = 64 if n <= 250 else 32 if n * 32 * 4 <= 64000 else 16
    eps = np.finfo(float).eps
    for e in range(ne):
        p, F = np.arange(n), LU[e].astype(float)
        for j in range(n):  # a panel's exchanges reach the columns of the panels before it only here
            k0 = j // w * w
            r = k0 + piv[e, j]
            p[[j, r]] = p[[r, j]]
            F[[j, r], :k0] = F[[r, j], :k0]
        L, U = np.tril(F, -1) + np.eye(n), np.triu(F)
        # substitution is componentwise backward stable: n products and sums for each triangle
        assert np.all(np.abs(L @ (U @ x[e]) - Ru[e][p]) <= 2 * (n + 2) * eps * (np.abs(L) @ (np.abs(U) @ np.abs(x[e]))))
    Kd = K.astype(float)
    ref, a = Rh - (Kd @ x[..., None])[..., 0], np.abs(Rh) + (np.abs(Kd) @ np.abs(x)[..., None])[..., 0]
    assert np.all(np.abs(rh.cpu().numpy() - ref) <= (n + 2) * eps * a)


def test_refinement_quotients():
    """The rows of a diagonal matrix are divided, not multiplied by a rounded reciprocal."""
    n, ne = 100, 3
    rng = np.random.default_rng(5)
    D = rng.uniform(0.5, 2.0, (ne, n)).astype(np.float32)
    LU, Ru = np.zeros((ne, n, n), dtype=np.float32), rng.standard_normal((ne, n))
    LU[:, np.arange(n), np.arange(n)] = D
    pv = np.tile((np.arange(n) % 64).astype(np.int32), (ne, 1))
    lu, piv, k, ru, rh = dev(LU), dev(pv), dev(np.zeros((ne, n, 4), dtype=np.float32)), dev(Ru), dev(np.zeros((ne, 4)))
    rus = torch.zeros((ne, n), dtype=torch.float64).cuda()
    d = Dims(m=4, n=n, ne=ne)
    call("_ZN3exa10refine_rhsERKNS_4DimsEPKfPKiS4_PKdPdS9_P12ihipStream_t", ctypes.byref(d), ptr(lu), ptr(piv), ptr(k),
         ptr(ru), ptr(rus), ptr(rh), None)
    assert np.array_equal(rus.cpu().numpy(), Ru / D.astype(float))
