"""M-Basis in windows of orders against the oracle, bit for bit (the reference's
t-pmbasis.c:70-109 pins the certificate; the basis itself is exact here): orders
around the window (4) and the update tile (12 to 15 coefficients written), rows and
columns around the kernels' lane splits, residuals that need the pivot search,
full rank inside a window, vectors too large for LDS."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

P30, P60, PBIG = 998244353, 1152921504556515329, 18446744073709551557

# (m, n, orders)
SHAPES = [
    (1, 1, (1, 2, 5)), (2, 1, (3, 4, 5, 8, 9, 13)), (4, 2, (11, 12, 13, 16, 25)), (9, 5, (7, 15)),
    (16, 8, (5,)), (20, 11, (6,)), (33, 16, (5,)), (35, 17, (9,)), (50, 32, (14,)), (50, 33, (6,)),
    (70, 3, (10,)), (66, 64, (5,)), (67, 65, (5,)), (140, 20, (6,)), (256, 30, (5,)),
]
KINDS = ["uniform", "lowrank", "sparse", "wide"]


def residual(rng, kind, m, n, order, p):
    hi = p - 1
    F = rng.integers(0, hi, (m, n, order), dtype=np.uint64)
    if kind == "lowrank":  # equal columns: panels with columns that take no pivot
        F[:, n // 2:, :] = F[:, :1, :]
        F[: m // 3, :, ::2] = 0
    elif kind == "sparse":
        F *= (rng.random(F.shape) < 0.1).astype(np.uint64)
    return F


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("p", [P30, P60, PBIG])
@pytest.mark.parametrize("m,n,orders", SHAPES)
def test_mbasis_windows(m, n, orders, p, kind):
    import pml_amd
    rng = np.random.default_rng(1000 * m + n)
    if kind == "wide":  # n >= m: the residual reaches full rank within a window
        if n > 20:
            pytest.skip("m rows suffice")
        m = n
    ctx = pml_amd.Context(p)
    for order in orders:
        F = residual(rng, kind, m, n, order, p)
        if kind == "wide":
            F[:, :, 0] = 0  # not at its first order
        shift = rng.integers(0, 3, m).astype(np.int64)
        P_ref, s_ref = O.mbasis(F, order, shift, p)
        P_dev, s_dev = ctx.mbasis(F, order, shift)
        assert np.array_equal(O.normalise(P_dev), O.normalise(P_ref))
        assert np.array_equal(s_dev, s_ref)
