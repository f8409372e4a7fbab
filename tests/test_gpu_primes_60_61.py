"""Products modulo 64-bit primes in [2^60, 2^61) against the oracle: the only moduli
that combine the MFMA pointwise kernel with the strict butterflies, whose inputs have
to lie below 2p.  Operands at the extremes (-1, small negatives) as well as uniform
ones, inner dimensions on both sides of where a sum of products passes (p - 1) 2^64,
every transform length of the register kernels and the first split one, single calls
and every batch configuration (t-mul_geometric.c:24-80 checks equality at random
sizes)."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

# just above 2^60, 1.5 2^60, just below 2^61
PRIMES = [1152921504618381313, 1729382256876716033, 2305843009211596801]


@pytest.fixture(scope="module")
def pml():
    import pml_amd
    return pml_amd


_ctxs = {}


def ctx_for(pml, p):
    if p not in _ctxs:
        _ctxs[p] = pml.Context(p)
    return _ctxs[p]


def operands(rng, kind, p, m, k, n, la, lb):
    if kind == "minus_one":  # constant matrices of -1, stored at length la, lb
        A, B = np.zeros((m, k, la), dtype=np.uint64), np.zeros((k, n, lb), dtype=np.uint64)
        A[..., 0] = p - 1
        B[..., 0] = p - 1
    elif kind == "small":  # small negatives, constant, by small coefficients
        A, B = np.zeros((m, k, la), dtype=np.uint64), rng.integers(0, 4, (k, n, lb), dtype=np.uint64)
        A[..., 0] = p - rng.integers(1, 9, (m, k), dtype=np.uint64)
    else:
        A = rng.integers(0, p, (m, k, la), dtype=np.uint64)
        B = rng.integers(0, p, (k, n, lb), dtype=np.uint64)
    return A, B


def lengths(log):
    """(lenA, lenB) of a product of 2^log words, and of one of at most 3/4 of them"""
    n = 1 << log
    return [(n // 2, n // 2 + 1)] + ([(n // 2, n // 8)] if log >= 5 else [])


@pytest.mark.parametrize("kind", ["minus_one", "small", "uniform"])
@pytest.mark.parametrize("p", PRIMES)
@pytest.mark.parametrize("log", range(1, 15))
def test_single_products(pml, p, log, kind):
    rng = np.random.default_rng(log)
    ctx = ctx_for(pml, p)
    for k in (7, 12, 16, 17, 20, 23, 24, 32, 47) if log < 11 else (9, 16, 24):
        m, n = (3, 2) if log < 9 else (1, 1)
        for la, lb in lengths(log):
            A, B = operands(rng, kind, p, m, k, n, la, lb)
            assert pml.config_valid(ctx, m, k, n, la, lb, 2)
            assert np.array_equal(ctx.mul(A, B, method="mfma"), O.polmat_mul(A, B, p)), (k, la, lb)


@pytest.mark.parametrize("kind", ["minus_one", "small"])
@pytest.mark.parametrize("p", PRIMES)
def test_automatic_choice(pml, p, kind):
    rng = np.random.default_rng(5)
    ctx = ctx_for(pml, p)
    for m, k, n in ((16, 23, 16), (16, 12, 16), (32, 20, 32)):
        for log in (2, 4, 7, 11):
            la, lb = lengths(log)[0]
            A, B = operands(rng, kind, p, m, k, n, la, lb)
            assert np.array_equal(ctx.mul(A, B), O.polmat_mul(A, B, p)), (m, k, n, la, lb)
            assert np.array_equal(ctx.mul(A, B, method="plain"), O.polmat_mul(A, B, p)), (m, k, n, la, lb)


@pytest.mark.parametrize("kind", ["minus_one", "small"])
@pytest.mark.parametrize("p", PRIMES)
@pytest.mark.parametrize("config", [1, 2, 3, 4, 5, 6, 7])
def test_batch_configurations(pml, p, config, kind):
    rng = np.random.default_rng(config)
    ctx = ctx_for(pml, p)
    items, want = [], []
    for log in (2, 3, 4, 6, 8, 10, 11, 12, 13, 14):
        for k in (16, 23):
            for la, lb in lengths(log):
                A, B = operands(rng, kind, p, 2, k, 1, la, lb)
                assert pml.config_valid(ctx, 2, k, 1, la, lb, config)
                items.append((ctx, A, B))
                want.append(O.polmat_mul(A, B, p))
    for g, w, (_, A, B) in zip(pml.mul_batch(items, config=config), want, items):
        assert np.array_equal(g, w), (A.shape, B.shape)
