"""gemm!'s 16x16 tile with and without operands read ahead: at the number of
workgroups that decides for four limbs (4096), at odd and single-term
reductions, against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

from mfutil import assert_bitwise, case_seed, rand_mf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,m,n,k", [(4, 1008, 1040, 1), (4, 1008, 1040, 15), (4, 1024, 1024, 1), (4, 1024, 1024, 15), (4, 1010, 1030, 16),
                                     (1, 130, 70, 17), (2, 130, 70, 33), (3, 131, 70, 15), (4, 130, 70, 31)])
def test_reads_ahead(oracle, N, m, n, k):
    import mfla

    rng = np.random.default_rng(case_seed("ahead", N, m, n, k))
    A, B, C = rand_mf(rng, N, m, k), rand_mf(rng, N, k, n), rand_mf(rng, N, m, n)
    Cd = torch.from_numpy(C.copy()).cuda()
    mfla.gemm_(Cd, torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda(), -1.0, 1.0, config=mfla.KernelConfig(gemm_tile=0))
    assert_bitwise(Cd.cpu().numpy(), oracle.gemm(C.copy(), A, B, -1.0, 1.0), f"x{N} {m}x{k}x{n}")
