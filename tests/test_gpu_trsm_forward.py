"""Forward triangular solves where their diagonal kernels change, bit for bit
against the oracle: four limbs (coefficients read from memory) at the edges of
a block of 64 and with few and many right-hand sides, two limbs on both sides
of the size from which the streamed steps branch (n times right-hand sides =
96 * 1024)."""
import numpy as np
import pytest
import torch

from mfutil import assert_bitwise, case_seed, rand_mf

pytestmark = pytest.mark.gpu


FORMS = [("left", "lower", "N", "nonunit"), ("left", "upper", "T", "unit"), ("right", "upper", "N", "nonunit")]
SIZES = [(4, 33, 1), (4, 63, 5), (4, 64, 4), (4, 65, 3), (4, 128, 70), (4, 192, 6), (4, 200, 66), (4, 257, 130), (4, 260, 270)]
CASES = [s + f for s in SIZES for f in FORMS] + [s + f for s in [(2, 1535, 64), (2, 1536, 64), (2, 1600, 63)] for f in FORMS[:2]]


@pytest.mark.parametrize("N,n,nrhs,side,uplo,trans,diag", CASES)
def test_forward(oracle, N, n, nrhs, side, uplo, trans, diag):
    import mfla

    rng = np.random.default_rng(case_seed("forward", N, n, nrhs))
    A = rand_mf(rng, N, n, n, scale=1.0 / n)
    A[0, np.arange(n), np.arange(n)] = 1.0 + np.arange(n) % 3
    A[1:, np.arange(n), np.arange(n)] = 0.0
    B = rand_mf(rng, N, n, nrhs) if side == "left" else rand_mf(rng, N, nrhs, n)
    Bd = torch.from_numpy(B.copy()).cuda()
    mfla.trsm_(Bd, torch.from_numpy(A).cuda(), side=side, uplo=uplo, trans=trans, diag=diag)
    torch.cuda.synchronize()
    assert_bitwise(Bd.cpu().numpy(), oracle.trsm(B.copy(), A, 1.0, side, uplo, trans, diag, threads=8), f"trsm x{N} {n}x{nrhs} {side} {uplo} {trans}")
