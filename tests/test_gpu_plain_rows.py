"""The plain pointwise kernel's tiles of two and of four rows against the oracle: sizes
on both sides of the line between them (6 rows, 2048 waves), ragged rows and columns,
inner dimensions around the folds after 15 products, every word size; in batches the
line is at 6 rows alone (t-mul_geometric.c:24-80 checks equality at random sizes)."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

P30, P60, P62 = 998244353, 1152921504556515329, 4611686018326724609


@pytest.fixture(scope="module")
def pml():
    import pml_amd
    return pml_amd


def operands(p, m, k, n, la, lb):
    rng = np.random.default_rng(m + 31 * k + n)
    A = rng.integers(0, p, (m, k, la), dtype=np.uint64)
    B = rng.integers(0, p, (k, n, lb), dtype=np.uint64)
    A[0], B[:, 0] = p - 1, p - 1
    return A, B


@pytest.mark.parametrize("p", [P30, P60, P62])
@pytest.mark.parametrize("m,k,n,length", [
    (6, 3, 9, 16000), (7, 3, 9, 16000), (7, 15, 5, 16000), (9, 2, 5, 16384), (65, 16, 66, 60),
    (65, 17, 66, 200), (129, 31, 61, 100), (1, 40, 3, 300), (2, 15, 1, 5), (3, 1, 2, 7),
])
def test_single_products(pml, p, m, k, n, length):
    A, B = operands(p, m, k, n, length, length - length // 3)
    with pml.Context(p) as ctx:
        assert np.array_equal(ctx.mul(A, B, method="plain"), O.polmat_mul(A, B, p))


@pytest.mark.parametrize("p", [P30, P60, P62])
def test_batches(pml, p):
    shapes = [(m, k, n, la) for m in (1, 2, 5, 6, 7, 8, 17) for k, n, la in ((1, 4, 3), (15, 5, 40), (33, 2, 700))]
    with pml.Context(p) as ctx:
        items = [(ctx,) + operands(p, m, k, n, la, la + 1) for m, k, n, la in shapes]
        want = [O.polmat_mul(A, B, p) for _, A, B in items]
        for config in (1, 3, 7):
            for g, w, s in zip(pml.mul_batch(items, config=config, graph=True), want, shapes):
                assert np.array_equal(g, w), (config, s)
