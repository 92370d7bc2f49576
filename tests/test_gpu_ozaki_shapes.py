"""The digit products' workgroup shapes and digit widths at their edges, against
the exact accumulator within test_gpu_ozaki's bound: outputs just below and at
the 1024 and 4096 blocks of 16 x 16 where four limbs change shape, odd numbers
of block columns, reductions shorter than a workgroup's four k steps, and both
sides of the 8-bit digits' last reduction length."""
import numpy as np
import pytest
import torch

from mfutil import case_seed, rand_mf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,m,k,n", [(4, 500, 70, 530), (4, 512, 70, 512), (4, 1023, 130, 1009), (4, 1025, 65, 1015), (4, 1030, 70, 1100), (4, 17, 1, 16),
                                     (4, 16, 4096, 33), (4, 33, 4097, 16), (3, 40, 64, 17), (3, 30, 4096, 20), (3, 20, 4100, 33), (2, 33, 193, 40),
                                     (2, 16, 4096, 17), (2, 17, 8192, 16), (1, 40, 300, 33), (1, 20, 5000, 17)])
def test_digit_product_edges(oracle, N, m, k, n):
    import mfla as M

    rng = np.random.default_rng(case_seed(N, m, k, n))
    A, B, C0 = rand_mf(rng, N, m, k, spread=6), rand_mf(rng, N, k, n, spread=6), rand_mf(rng, N, m, n)
    if k == 4096:
        A[0] = np.where(A[0] < 0, -1.0, 1.0) * (2.0 - 2.0**-40)      # the largest digit sums
        A[1:] = 0.0
        B[0] = A[0, 0, 0] * np.where(B[0] < 0, 1.0, -1.0)
        B[1:] = 0.0
    C = torch.from_numpy(C0).cuda()
    M.gemm_(C, torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda(), -1.0, 1.0, config=M.KernelConfig(gemm_strategy="ozaki"))
    rows = np.concatenate([rng.integers(0, m, 200), [0, m - 1, 0, m - 1]])
    cols = np.concatenate([rng.integers(0, n, 200), [0, 0, n - 1, n - 1]])
    pad = lambda X: np.concatenate([X, np.zeros_like(X)], axis=0)          # noqa: E731
    err, _ = oracle.exact_axpb(pad(A), pad(B), np.concatenate([C.cpu().numpy(), -C0], axis=0), sab=-1, sc=-1, rows=rows, cols=cols)
    tol = 2.0 ** (-52 * N + 7) * (k * np.abs(A[0]).max(axis=0)[rows] * np.abs(B[0]).max(axis=1)[cols] + np.abs(C0[0][cols, rows]))
    assert np.all(np.abs(err) <= tol), np.max(np.abs(err) / tol)
