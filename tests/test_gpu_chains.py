"""Serial-chain kernels whose products are formed by other waves (gemv!, symv!,
the exact backward substitution) at the edges of their chunks, against the
oracle, bit for bit."""
import numpy as np
import pytest
import torch

from mfutil import assert_bitwise, case_seed, rand_mf

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


# 16 outputs take chunks of 48 columns, 64 outputs (over 8192 in all) chunks of 12
@pytest.mark.parametrize("N", [2, 3, 4])
@pytest.mark.parametrize("m,n", [(1, 1), (15, 47), (16, 48), (17, 49), (64, 97), (8193, 11), (8200, 13), (12, 8250), (5, 0)])
def test_gemv_chunk_edges(oracle, N, m, n):
    import mfla

    rng = np.random.default_rng(case_seed(N, m, n))
    A = rand_mf(rng, N, m, n) if m * n else np.zeros((N, n, m))
    # a view with a leading dimension and an offset of its own
    big = torch.full((N, n + 1, m + 3), float("nan"), dtype=torch.float64, device="cuda")
    big[:, 1:, 2:m + 2] = dev(A)
    for trans in "NT":
        x = rand_mf(rng, N, n if trans == "N" else m) if m * n else np.zeros((N, n if trans == "N" else m))
        y = rand_mf(rng, N, m if trans == "N" else n) if m * n else np.zeros((N, m if trans == "N" else n))
        for a, b in ((1.0, 0.0), (-1.0, 1.0)):
            yd = dev(y)
            mfla.gemv_(yd, big[:, 1:, 2:m + 2], dev(x), a, b, trans=trans)
            assert_bitwise(host(yd), oracle.gemv(y.copy(), A, x, a, b, trans), f"gemv x{N} {m}x{n} {trans}")


@pytest.mark.parametrize("N", [2, 3, 4])
@pytest.mark.parametrize("n", [1, 16, 49, 130])
def test_symv_chunk_edges(oracle, N, n):
    import mfla

    rng = np.random.default_rng(case_seed(N, n))
    A, x, y = rand_mf(rng, N, n, n), rand_mf(rng, N, n), rand_mf(rng, N, n)
    for uplo in ("lower", "upper"):
        B = A.copy()
        i = np.arange(n)                       # the other triangle is never read
        B[:, (i[:, None] > i[None, :]) if uplo == "lower" else (i[:, None] < i[None, :])] = np.nan
        yd = dev(y)
        mfla.symv_(yd, dev(B), dev(x), -1.0, 1.0, uplo=uplo)
        assert_bitwise(host(yd), oracle.symv(y.copy(), A, x, -1.0, 1.0, uplo), f"symv x{N} {n} {uplo}")


# one right-hand side takes chunks of 192 terms, 16 (over 256 right-hand
# sides) of 24, 64 (over 4096) of 9
@pytest.mark.parametrize("N,n,nrhs", [(4, 1, 1), (4, 2, 3), (4, 3, 1), (2, 194, 2), (3, 195, 1), (4, 196, 1), (4, 256, 2), (2, 25, 257), (4, 26, 259),
                                      (2, 27, 300), (4, 11, 4097), (2, 21, 4100)])
@pytest.mark.parametrize("side,uplo,trans", [("left", "lower", "T"), ("left", "upper", "N"), ("right", "lower", "N")])
def test_exact_backward_chunk_edges(oracle, N, n, nrhs, side, uplo, trans):
    import mfla

    rng = np.random.default_rng(case_seed(N, n, nrhs, side, uplo, trans))
    A = rand_mf(rng, N, n, n, scale=1.0 / n)
    A[0, np.arange(n), np.arange(n)] = 1.0 + np.arange(n) % 3
    A[1:, np.arange(n), np.arange(n)] = 0.0
    for diag in ("nonunit", "unit"):
        B = rand_mf(rng, N, n, nrhs) if side == "left" else rand_mf(rng, N, nrhs, n)
        Bd = dev(B)
        mfla.trsm_(Bd, dev(A), side=side, uplo=uplo, trans=trans, diag=diag, config=mfla.KernelConfig(trsm_order="exact"))
        assert_bitwise(host(Bd), oracle.trsm(B.copy(), A, 1.0, side, uplo, trans, diag), f"trsm x{N} n={n} nrhs={nrhs}")
