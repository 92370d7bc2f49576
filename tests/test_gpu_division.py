"""Division and square root on the GPU against the oracle, bit for bit, where
their shortened operations could differ: vanishing remainders, zero limbs of
either sign, extreme exponents and non-finite operands."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def limbs(rng, hi, N, zeros):
    x = np.zeros((N, hi.size))
    x[0] = hi
    for l in range(1, N):
        x[l] = x[l - 1] * 2.0**-53 * rng.uniform(-1, 1, hi.size)
        if zeros:
            x[l] = np.where(rng.integers(0, 2, hi.size) == 1, x[l], np.where(rng.integers(0, 2, hi.size) == 1, 0.0, -0.0))
    return x


def cases(N, rng, count=4096):
    normal = lambda: rng.standard_normal(count)  # noqa: E731
    whole = lambda: rng.integers(1, 2000, count).astype(np.float64)  # noqa: E731
    yield "ordinary", limbs(rng, normal(), N, False), limbs(rng, normal(), N, False)
    yield "zero limbs", limbs(rng, normal(), N, True), limbs(rng, normal(), N, True)
    d = whole()
    yield "exact quotients", limbs(rng, d * whole(), N, True) * (np.arange(N) == 0)[:, None], limbs(rng, d, N, True) * (np.arange(N) == 0)[:, None]
    for e in (-1000, -600, 600, 1000):
        yield f"2^{e}", limbs(rng, np.ldexp(rng.uniform(1, 2, count), e), N, False), limbs(rng, normal(), N, False)
        yield f"by 2^{e}", limbs(rng, normal(), N, False), limbs(rng, np.ldexp(rng.uniform(1, 2, count), e), N, False)
    # one wave holds ordinary, huge, tiny, zero and non-finite operands
    hi = normal()
    hi[::7] = np.ldexp(1.0, rng.integers(-1000, 1000, hi[::7].size))
    hi[::31] = 0.0
    hi[::97] = np.inf
    hi[::101] = np.nan
    yield "mixed", limbs(rng, hi, N, False), limbs(rng, normal(), N, False)
    yield "by mixed", limbs(rng, normal(), N, False), limbs(rng, hi, N, False)


def same(got, ref):
    both = np.isnan(got) & np.isnan(ref)
    return np.array_equal(np.where(both, 0.0, got).view(np.uint64), np.where(both, 0.0, ref).view(np.uint64))


@pytest.mark.parametrize("N", [2, 3, 4])
def test_division_and_sqrt_bitwise_over_ranges(N):
    import torch

    import mfla

    rng = np.random.default_rng(40 + N)
    for name, a, b in cases(N, rng):
        x, y = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
        with np.errstate(all="ignore"):
            assert same(mfla.arith("div", x, y).cpu().numpy(), oracle.arith("div", a, b)), f"x{N} div {name}"
            p = a * np.where(a[0] < 0, -1.0, 1.0)
            assert same(mfla.arith("sqrt", torch.from_numpy(p).cuda()).cpu().numpy(), oracle.arith("sqrt", p)), f"x{N} sqrt {name}"
