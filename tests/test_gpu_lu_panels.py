"""lu! with a whole panel in one kernel, at the edges of its panels and of its
workgroups' rows, against the oracle, bit for bit: factors, pivots and failure
states, ties and rows that repeat."""
import numpy as np
import pytest
import torch

from mfutil import assert_bitwise, case_seed, rand_mf

pytestmark = pytest.mark.gpu


def check(oracle, A, block=16, threads=0):
    import mfla as M

    N, n, m = A.shape
    ref = A.copy()
    out = oracle.getrf(ref, block, threads=threads)
    big = torch.full((N, n, m + 3), float("nan"), dtype=torch.float64, device="cuda")
    V = big[:, :, 2:m + 2]
    V.copy_(torch.from_numpy(A))
    F = M.lu_(V, check=False, config=M.KernelConfig(lu_block=block))
    info, ipiv = out[0], out[1]
    assert F.info == info
    assert np.array_equal(F.ipiv.cpu().numpy(), ipiv)
    assert_bitwise(V.cpu().numpy(), ref, f"lu x{N} {m}x{n}")
    return info


@pytest.mark.parametrize("N,m,n", [(N, m, n) for N in (1, 2, 3, 4) for m, n in
                                   ((1, 1), (15, 15), (16, 16), (17, 17), (33, 20), (20, 33), (130, 130), (200, 7), (7, 200))])
def test_panel_edges(oracle, N, m, n):
    rng = np.random.default_rng(case_seed(N, m, n))
    assert check(oracle, rand_mf(rng, N, m, n)) == 0
    if m == 130:
        assert check(oracle, rand_mf(rng, N, m, n), block=5) == 0


# one row a thread up to 1024 rows (64 workgroups), two up to 2048, four up to
# 8192, then column kernels; 1040 and 2060 cross an edge between panels
@pytest.mark.parametrize("N,m", [(2, 2048), (2, 2049), (4, 2060), (3, 4096), (2, 4097), (4, 4110), (2, 8192), (2, 8193),
                                 (2, 1024), (3, 1024), (4, 1024), (2, 1025), (3, 1025), (4, 1025), (2, 1040), (3, 1040), (4, 1040), (3, 1700),
                                 (3, 2049), (4, 8192)])
def test_tall_panels(oracle, N, m):
    rng = np.random.default_rng(case_seed(N, m))
    assert check(oracle, rand_mf(rng, N, m, 37), threads=8) == 0


@pytest.mark.parametrize("N", [2, 4])
def test_ties_zero_pivots_and_lower_limbs(oracle, N):
    rng = np.random.default_rng(case_seed("ties", N))
    A = rand_mf(rng, N, 300, 40)
    A[0] = np.sign(A[0])                       # every leading limb +-1: lower limbs and rows decide
    check(oracle, A)
    A[1:] = 0.0                                # exact ties everywhere
    check(oracle, A)
    B = rand_mf(rng, N, 90, 90)
    B[:, 40, :] = 0.0                          # a zero column: the pivot of column 41 vanishes
    assert check(oracle, B) == 41
    B = rand_mf(rng, N, 64, 64)
    B[:, 0, :] = 0.0
    assert check(oracle, B) == 1
