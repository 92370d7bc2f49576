"""The waves of ldlt!'s unblocked body, on the host: whatever order they run
in between barriers, they take the same branches (or their barriers pair up
wrongly, and an index comes from another reduction's buffer) and give the
oracle's bits. Cases: an indefinite matrix with many 2x2 pivots, a singular
one, a KKT matrix of the batched kernel's workgroup."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from mfutil import assert_bitwise, case_seed, rand_mf

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "multifloatlinearalgebra.jl_amd", "csrc")


@pytest.fixture(scope="module")
def waves(tmp_path_factory):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no host compiler")
    so = str(tmp_path_factory.mktemp("waves") / "ldlt_waves.so")
    here = os.path.join(HERE, "host_waves")
    subprocess.run([cxx, "-std=c++17", "-O1", "-mfma", "-ffp-contract=off", "-w", "-shared", "-fPIC", "-I", here, "-I", CSRC,
                    os.path.join(here, "ldlt_waves.cpp"), "-o", so], check=True)
    return ctypes.CDLL(so).ldlt_waves


def matrix(kind, N, n):
    rng = np.random.default_rng(case_seed("waves", kind, N, n))
    G = rand_mf(rng, N, n, n)
    A = G + np.transpose(G, (0, 2, 1))
    if kind == "singular":
        A[:, n // 4, :] = 0.0
        A[:, :, n // 4] = 0.0
    if kind == "kkt":
        m = 2 * n // 3
        A[:, :m, :m] *= 1e-3
        A[:, m:, m:] = 0.0
        A[0, np.arange(m, n), np.arange(m, n)] = -1e-8
    return A


@pytest.mark.parametrize("kind,N,n,threads,coefs", [("indefinite", 4, 64, 512, 0), ("singular", 4, 70, 512, 0), ("kkt", 3, 100, 256, 1),
                                                    ("kkt", 2, 90, 128, 1), ("indefinite", 1, 64, 64, 1)])
def test_any_order_of_the_waves(oracle, waves, kind, N, n, threads, coefs):
    A = matrix(kind, N, n)
    F = A.copy()
    info, dsub, piv, blk, _ = oracle.sytrf(F, "unblocked")
    assert (info > 0) == (kind == "singular") and (blk == 2).any()
    p = lambda a, t: a.ctypes.data_as(ctypes.POINTER(t))  # noqa: E731
    for seed in range(1, 4):
        B, d = A.copy(), np.zeros((N, n))
        pv, bk, got = np.arange(1, n + 1), np.zeros(n, dtype=np.uint8), ctypes.c_int64(0)
        barriers = waves(ctypes.c_int(N), ctypes.c_int64(n), p(B, ctypes.c_double), p(d, ctypes.c_double), p(pv, ctypes.c_int64),
                         p(bk, ctypes.c_uint8), ctypes.byref(got), ctypes.c_int(threads), ctypes.c_int(coefs), ctypes.c_uint64(seed))
        assert barriers > n, f"seed {seed}: waves at different barriers"
        assert got.value == info and np.array_equal(pv, piv) and np.array_equal(bk, blk), seed
        assert_bitwise(B, F, f"{kind} x{N} n={n} seed {seed}")
        assert_bitwise(d, dsub, f"{kind} x{N} n={n} dsub seed {seed}")
