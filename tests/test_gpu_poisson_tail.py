"""The far tail of the mixed-precision Poisson sampler, the FP64 search that
decides it and where that search ends; the FP64 sums that decide draws next to a
value of the CDF (marked gpu)."""
import math
import zlib

import numpy as np
import pytest
from scipy import special

pytestmark = pytest.mark.gpu

LAM = np.float32([10.0, 10.5, 17.0, 25.0, 29.5, 33.0, 48.0, 59.0, 100.0, 400.0, 700.0, 707.5])
LAM_UNDER = np.float32([708.5, 745.0, 1000.0, 40000.0, 65535.0])  # e^-lambda taken as 0
U_ONE, U_BELOW = 0xFFFFFFFF, 0xFFFFFE00


def _search(lam, u, p):
    """The plain search from p(0) = p, counted to its end."""
    S, k = p, 0
    while u > S and k < 100000:
        k += 1
        p = p * lam / k
        S += p
    return k


@pytest.mark.parametrize("lam", LAM)
def test_uniform_one_ends_as_the_plain_search_does(native, lam):
    k, path = native.poisson_probe_mixed(np.float32([lam]), np.uint32([U_ONE]))
    l = float(lam)
    p0 = math.exp(-l)
    # e^-lambda of the sampler and of the C library may differ in the last bits
    ends = {_search(l, 1.0, p0 * (1.0 + d * 2.0 ** -52)) for d in range(-4, 5)}
    assert path[0] == 3 and int(k[0]) in ends, (k[0], ends)


def test_uniform_one_with_an_underflowed_start(native):
    k, path = native.poisson_probe_mixed(LAM_UNDER, np.full(LAM_UNDER.size, U_ONE, np.uint32))
    assert (path == 3).all() and (k == 100000).all()


def test_uniform_just_below_one_is_the_exact_inverse(native):
    lam = np.concatenate([LAM, LAM_UNDER])
    k, _ = native.poisson_probe_mixed(lam, np.full(lam.size, U_BELOW, np.uint32))
    for l, n in zip(lam.astype(np.float64), k):
        assert special.pdtrc(n, l) <= 2.0 ** -24 * (1 + 1e-6) and special.pdtrc(n - 1, l) > 2.0 ** -24 * (1 - 1e-6), (l, n)


# crc32 of the draws (int32) as the term-by-term FP64 sums alone decide them
TERM_BY_TERM = {10.0: 2101785422, 11.5: 2358396442, 57.25: 1646697598, 300.0: 1699955642, 900.5: 2218100682,
                5000.0: 3973358506, 30000.75: 3706015999, 65535.0: 2201492289}


def _draws(native, lam):
    words = np.random.default_rng(int(lam)).integers(0, 2 ** 32, 1 << 19, dtype=np.uint32)
    return native.poisson_probe_mixed(np.full(words.size, lam, np.float32), words)


@pytest.mark.parametrize("lam", TERM_BY_TERM)
def test_decisions_are_those_of_the_term_by_term_sums(native, lam):
    k, path = _draws(native, lam)
    assert (path == 3).sum() > 20
    assert zlib.crc32(k.astype("<i4").tobytes()) == TERM_BY_TERM[lam]
