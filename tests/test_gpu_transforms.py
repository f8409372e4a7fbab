"""Products whose transforms take every length of the register kernels, and the
first ones past them, against the oracle: operands that fill the length, leave one
word or three quarters of it, more and fewer entries than a workgroup holds
transforms, both radices (configurations 2 and 5 against 3 and 4), both word sizes,
lazy and strict butterflies (t-mul_geometric.c:24-80 checks equality at random
sizes)."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

P30, P60 = 998244353, 1152921504556515329
P62 = 4611686018326724609  # strict butterflies


@pytest.fixture(scope="module")
def pml():
    import pml_amd
    return pml_amd


_ctxs = {}


def ctx_for(pml, p):
    if p not in _ctxs:
        _ctxs[p] = pml.Context(p)
    return _ctxs[p]


def lengths(log):
    """(lenA, lenB) with products of 2^log, 3/4 2^log and just above 2^(log - 1) words"""
    n = 1 << log
    out = {(max(1, n // 2), n - max(1, n // 2) + 1), (max(1, n // 2 + 1 - n // 8), max(1, n // 8)),
           (max(1, 3 * n // 8), 3 * n // 4 - max(1, 3 * n // 8) + 1)}
    return sorted((a, b) for a, b in out if a + b - 1 <= n)


@pytest.mark.parametrize("p", [P30, P60, P62])
@pytest.mark.parametrize("log", range(1, 18))
def test_every_length(pml, p, log):
    rng = np.random.default_rng(log)
    m, k, n = (5, 3, 7) if log < 9 else (2, 3, 1) if log < 13 else (1, 2, 1)
    for la, lb in lengths(log):
        A = rng.integers(0, p, (m, k, la), dtype=np.uint64)
        B = rng.integers(0, p, (k, n, lb), dtype=np.uint64)
        A[..., -1] = p - 1  # extreme words at the ragged end
        B[0] = p - 1
        assert np.array_equal(ctx_for(pml, p).mul(A, B), O.polmat_mul(A, B, p)), (la, lb)


@pytest.mark.parametrize("p", [P30, P60])
@pytest.mark.parametrize("log", [4, 7, 9, 10, 11, 12, 13, 14, 15])
def test_radices_agree(pml, p, log):
    """every configuration of a batch against the oracle"""
    rng = np.random.default_rng(100 + log)
    la, lb = lengths(log)[-1]
    A = rng.integers(0, p, (2, 2, la), dtype=np.uint64)
    B = rng.integers(0, p, (2, 2, lb), dtype=np.uint64)
    want = O.polmat_mul(A, B, p)
    ctx = ctx_for(pml, p)
    for c in range(1, pml.num_configs()):
        if pml.config_valid(ctx, 2, 2, 2, la, lb, c):
            got = pml.mul_batch([(ctx, A, B), (ctx, A[::-1].copy(), B)], config=c)
            assert np.array_equal(got[0], want), c
            assert np.array_equal(got[1], want[::-1]), c


@pytest.mark.parametrize("p", [P30, P60, P62])
@pytest.mark.parametrize("m,k,n", [
    (1, 1, 1), (3, 17, 2), (15, 16, 17), (16, 31, 32), (33, 33, 5), (49, 63, 47),
    (64, 64, 64), (89, 20, 90), (130, 100, 1), (1, 300, 129),
])
def test_pointwise_tiles(pml, p, m, k, n):
    """dimensions around the 16 x 16 tiles, inner dimensions around the MFMA steps
    and past the old limit of 88 rows, by each kernel that takes them"""
    rng = np.random.default_rng(m + 7 * n)
    A = rng.integers(0, p, (m, k, 5), dtype=np.uint64)
    B = rng.integers(0, p, (k, n, 4), dtype=np.uint64)
    A[0], B[:, 0] = p - 1, p - 1
    want = O.polmat_mul(A, B, p)
    ctx = ctx_for(pml, p)
    assert np.array_equal(ctx.mul(A, B), want)
    assert np.array_equal(ctx.mul(A, B, method="plain"), want)
    if pml.config_valid(ctx, m, k, n, 5, 4, 2):
        assert np.array_equal(ctx.mul(A, B, method="mfma"), want)
