"""cholesky! in one kernel per panel, at the edges of its panels and of its
workgroups' rows, factors and failure states against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

from mfutil import assert_bitwise, case_seed, rand_mf

pytestmark = pytest.mark.gpu


def spd(oracle, rng, N, n):
    R = rand_mf(rng, N, n, n)
    S = np.zeros((N, n, n))
    oracle.gemm(S, R, np.ascontiguousarray(np.transpose(R, (0, 2, 1))), fused=False)
    S[0, np.arange(n), np.arange(n)] += n
    return S


# 12 rows a workgroup; panels of 16 with a last one of 1..16
@pytest.mark.parametrize("N,n", [(N, n) for N in (1, 2, 3, 4) for n in (1, 15, 16, 17, 28, 29, 64, 65, 81, 130)])
def test_panel_edges(oracle, N, n):
    import mfla as M

    rng = np.random.default_rng(case_seed(N, n))
    S = spd(oracle, rng, N, n)
    for block in (16, 5) if n in (17, 65) else (16,):
        ref = S.copy()
        assert oracle.potrf(ref, block) == 0
        big = torch.full((N, n, n + 2), float("nan"), dtype=torch.float64, device="cuda")
        A = big[:, :, 1:n + 1]
        A.copy_(torch.from_numpy(S))
        assert M.cholesky_(A, config=M.KernelConfig(cholesky_block=block)).info == 0
        assert_bitwise(A.cpu().numpy(), ref, f"cholesky x{N} n={n} block {block}")


@pytest.mark.parametrize("N", [2, 4])
@pytest.mark.parametrize("n,bad", [(20, 0), (20, 15), (20, 16), (20, 19), (100, 40), (100, 63), (100, 99)])
def test_failure_states(oracle, N, n, bad):
    import mfla as M

    rng = np.random.default_rng(case_seed(N, n, bad))
    S = spd(oracle, rng, N, n)
    S[0, bad, bad] = -1.0
    ref = S.copy()
    info = oracle.potrf(ref, 16)
    A = torch.from_numpy(S).cuda()
    F = M.cholesky_(A, check=False)
    assert F.info == info == bad + 1
    assert_bitwise(A.cpu().numpy(), ref, f"failed cholesky x{N} n={n} at {bad}")


def test_wide_rows(oracle):
    """8 rows a wave (over 3072 rows below the first panels)"""
    import mfla as M

    n, N = 3120, 2
    g = torch.Generator(device="cuda").manual_seed(5)
    S = torch.zeros((N, n, n), dtype=torch.float64, device="cuda")
    S[0] = torch.rand((n, n), generator=g, dtype=torch.float64, device="cuda") * 0.1
    S[1] = S[0] * 2.0**-54
    S[0].diagonal().add_(float(n))
    A, ref = S.clone(), S.cpu().numpy()
    assert M.cholesky_(A).info == 0 and oracle.potrf(ref, 16, threads=16) == 0
    assert_bitwise(A.cpu().numpy(), ref, "cholesky x2 n=3120")
