"""ybar S^-1, whose forward solve ends each block of rows at its last column:
the blocks' edges (64 rows; look-ahead from 193, device counters up to 256
right-hand sides) against the solve with the full identity, bit for bit, and
the exact residual."""
import numpy as np
import pytest
import torch

from mfutil import case_seed, eps, rand_mf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,n", [(4, 1), (2, 63), (3, 64), (4, 65), (2, 129), (4, 192), (4, 193), (2, 257), (4, 256), (3, 330), (2, 520)])
def test_inverse_at_block_edges(oracle, N, n):
    import mfla as M
    from mfla import autodiff as AD

    rng = np.random.default_rng(case_seed(N, n))
    R = rand_mf(rng, N, n, n)
    S = np.zeros((N, n, n))
    oracle.gemm(S, R, np.ascontiguousarray(np.transpose(R, (0, 2, 1))), fused=False)
    S[0, np.arange(n), np.arange(n)] += n
    F = M.cholesky_(torch.from_numpy(S).cuda())
    one = np.zeros(N)
    one[0] = 1.0
    G = AD.logdet_adjoint(F, one).cpu().numpy()
    assert np.array_equal(G, np.transpose(G, (0, 2, 1)))
    full = M.solve(F, torch.from_numpy(np.where(np.eye(n) == 1, one[:, None, None], 0.0)).cuda(), config=M.KernelConfig(trsm_order="blocked"))
    sym = M.arith("add", full.reshape(N, -1), full.transpose(1, 2).reshape(N, -1)).cpu().numpy().reshape(N, n, n) * 0.5
    assert np.array_equal(G, sym)
    # S holds S below the diagonal's mirror too (symmetric input); I - S G, exactly
    low = np.tril_indices(n, -1)
    S[:, low[0], low[1]] = S[:, low[1], low[0]]
    I = np.zeros((N, n, n))
    I[0, np.arange(n), np.arange(n)] = 1.0
    rows, cols = rng.integers(0, n, 400), rng.integers(0, n, 400)
    err, scale = oracle.exact_axpb(S, G, I, sab=-1, sc=1, rows=rows, cols=cols)
    assert np.max(np.abs(err) / scale) <= 64 * n * eps(N)
    half = AD.logdet_adjoint(F, one * 0.5).cpu().numpy()
    assert np.array_equal(half, G * 0.5)


@pytest.mark.parametrize("N,n", [(2, 70), (4, 130), (3, 256)])
def test_solve_adjoint_keeps_a_stated_order(oracle, N, n):
    """"exact" and "blocked" give the bits of a solve in that order; the order
    left open is the blocked one, also at n <= 256."""
    import mfla as M
    from mfla import autodiff as AD

    rng = np.random.default_rng(case_seed("order", N, n))
    R = rand_mf(rng, N, n, n)
    S = np.zeros((N, n, n))
    oracle.gemm(S, R, np.ascontiguousarray(np.transpose(R, (0, 2, 1))), fused=False)
    S[0, np.arange(n), np.arange(n)] += n
    F = M.cholesky_(torch.from_numpy(S).cuda())
    X, Xbar = torch.from_numpy(rand_mf(rng, N, n, 3)).cuda(), torch.from_numpy(rand_mf(rng, N, n, 3)).cuda()
    solved = {o: M.solve(F, Xbar, config=M.KernelConfig(trsm_order=o)).cpu().numpy() for o in ("exact", "blocked")}
    assert not np.array_equal(solved["exact"], solved["blocked"])
    for order, want in (("exact", "exact"), ("blocked", "blocked"), ("auto", "blocked")):
        Bbar, _ = AD.solve_adjoint(F, X, Xbar, config=M.KernelConfig(trsm_order=order))
        assert np.array_equal(Bbar.cpu().numpy(), solved[want]), order
