"""lu! and ldlt! on several handles at once, on one stream mask and on the
device's CUs: the panels' workgroups wait for each other, so only as many
calls as their CUs hold run them, the others panels that do not wait. Every
call's results are those of a call alone, bit for bit."""
import ctypes
import threading

import numpy as np
import pytest
import torch

from mfutil import assert_bitwise, case_seed, rand_mf

pytestmark = pytest.mark.gpu


def masked_stream(cus):
    """A stream on the mask's first `cus` CUs, from the runtime torch loaded."""
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    words = (cus + 31) // 32
    mask = (ctypes.c_uint32 * words)(*[0xFFFFFFFF if 32 * (w + 1) <= cus else (1 << (cus % 32)) - 1 for w in range(words)])
    s = ctypes.c_void_p()
    assert ctypes.CDLL(path).hipExtStreamCreateWithCUMask(ctypes.byref(s), words, mask) == 0
    return s


class Caller:
    """A handle of its own on a stream of its own, through the C ABI."""

    def __init__(self, stream):
        from mfla import _lib

        self.lib, self.h, self.stream = _lib.load(), ctypes.c_void_p(), stream
        assert self.lib.mfla_handle_create(ctypes.byref(self.h)) == 0
        assert self.lib.mfla_handle_set_stream(self.h, stream) == 0

    def close(self):
        assert self.lib.mfla_handle_destroy(self.h) == 0

    def matrix(self, t):
        from mfla import _lib

        N, cols, rows = t.shape
        return _lib.MFMatrix(t.data_ptr(), rows, cols, rows, rows * cols)

    def error(self, rc):
        return self.lib.mfla_last_error().decode() if rc else ""

    def lu(self, A):
        N, n, m = A.shape
        ipiv = torch.empty(min(m, n), dtype=torch.int64, device="cuda")
        om, info = (ctypes.c_double * 4)(), ctypes.c_int64(-9)
        torch.cuda.synchronize()
        rc = self.lib.mfla_getrf(self.h, N, self.matrix(A), ipiv.data_ptr(), om, ctypes.byref(info), None, None)
        return self.error(rc), info.value, [A.cpu().numpy(), ipiv.cpu().numpy()]

    def ldlt(self, A):
        N, n, _ = A.shape
        dsub = torch.zeros((N, 1, n), dtype=torch.float64, device="cuda")
        piv, blk = torch.empty(n, dtype=torch.int64, device="cuda"), torch.empty(n, dtype=torch.uint8, device="cuda")
        om, info = (ctypes.c_double * 4)(), ctypes.c_int64(-9)
        torch.cuda.synchronize()
        rc = self.lib.mfla_sytrf(self.h, N, self.matrix(A), self.matrix(dsub), piv.data_ptr(), blk.data_ptr(), om, ctypes.byref(info), None, None)
        return self.error(rc), info.value, [A.cpu().numpy(), dsub.cpu().numpy(), piv.cpu().numpy(), blk.cpu().numpy()]


def at_once(callers, jobs):
    """jobs[i] on callers[i], all started together."""
    start, out = threading.Barrier(len(jobs)), [None] * len(jobs)

    def go(i):
        start.wait(30)
        out[i] = jobs[i](callers[i])

    threads = [threading.Thread(target=go, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert all(o is not None for o in out)
    return out


def same(got, want, what):
    assert got[0] == want[0] == "" and got[1] == want[1] == 0, (what, got[:2], want[:2])
    for g, w in zip(got[2], want[2]):
        if g.dtype == np.float64:
            assert_bitwise(g, w, what)
        else:
            assert np.array_equal(g, w), what


# 64 waiting workgroups each: a 32-CU mask takes one such call, an 8-CU mask none
@pytest.mark.parametrize("N", [2, 4])
@pytest.mark.parametrize("cus", [(None,) * 3, (32,) * 3, (8, 32, None)])
def test_lu_calls_at_once(oracle, N, cus):
    rng = np.random.default_rng(case_seed("lu at once", N))
    A = rand_mf(rng, N, 1024, 40)
    ref = A.copy()
    info, ipiv = oracle.getrf(ref, 16, threads=8)[:2]
    callers = [Caller(ctypes.c_void_p(torch.cuda.Stream().cuda_stream) if c is None else masked_stream(c)) for c in cus]
    try:
        for rep in range(3):
            out = at_once(callers, [lambda c, a=torch.from_numpy(A).cuda(): c.lu(a) for _ in callers])
            for o in out:
                same(o, ("", info, [ref, ipiv]), f"lu x{N} on {cus}")
    finally:
        for c in callers:
            c.close()


# look-ahead: 9 waiting workgroups a call on the handles' panel streams, whose
# 32 CUs are the same for every handle: two calls have places there
@pytest.mark.parametrize("N,calls", [(2, 2), (2, 4)])
def test_ldlt_calls_at_once(N, calls):
    rng = np.random.default_rng(case_seed("ldlt at once", N))
    n = 1600
    G = rand_mf(rng, N, n, n)
    A = G + np.transpose(G, (0, 2, 1))
    A[0, np.arange(n), np.arange(n)] += 4.0 * np.sqrt(n)
    callers = [Caller(ctypes.c_void_p(torch.cuda.Stream().cuda_stream)) for _ in range(calls)]
    try:
        want = callers[0].ldlt(torch.from_numpy(A).cuda())
        out = at_once(callers, [lambda c, a=torch.from_numpy(A).cuda(): c.ldlt(a) for _ in callers])
        for o in out:
            same(o, want, f"ldlt x{N}, {calls} at once")
    finally:
        for c in callers:
            c.close()


def test_lu_beside_a_batch(oracle):
    """lu!'s waiting panels beside a batch whose workgroups fill the device
    and end by themselves."""
    from mfla.batched import Batch

    rng = np.random.default_rng(case_seed("lu beside a batch"))
    N = 2
    systems = []
    for i in range(600):
        n = 100 + i % 100
        S = np.zeros((N, n, n))
        G = rng.standard_normal((n, n))
        S[0] = G @ G.T + n * np.eye(n)
        systems.append((0, S, rng.standard_normal((N, 2, n)) * np.array([1.0, 2.0**-53])[:, None, None]))
    A = rand_mf(rng, N, 1024, 40)
    ref = A.copy()
    info, ipiv = oracle.getrf(ref, 16, threads=8)[:2]
    b = Batch(systems, N)
    b.solve()
    want = [r["A"].copy() for r in b.results()[:20]]
    caller, q = Caller(ctypes.c_void_p(torch.cuda.Stream().cuda_stream)), torch.cuda.Stream()
    try:
        for rep in range(3):
            Ad = torch.from_numpy(A).cuda()
            b.restore()
            torch.cuda.synchronize()
            with torch.cuda.stream(q):
                b.solve()
            ipd = torch.empty(40, dtype=torch.int64, device="cuda")
            om, inf = (ctypes.c_double * 4)(), ctypes.c_int64(-9)
            rc = caller.lib.mfla_getrf(caller.h, N, caller.matrix(Ad), ipd.data_ptr(), om, ctypes.byref(inf), None, None)   # no wait for the batch
            torch.cuda.synchronize()
            same((caller.error(rc), inf.value, [Ad.cpu().numpy(), ipd.cpu().numpy()]), ("", info, [ref, ipiv]), "lu beside a batch")
            for r, w in zip(b.results()[:20], want):
                assert r["info"] == 0
                assert_bitwise(r["A"], w, "batch beside lu")
    finally:
        caller.close()
