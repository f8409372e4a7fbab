"""M-Basis by single orders (the shapes where windows of orders do not pay) against the
oracle, bit for bit, as test_gpu_mbasis_window.py does for the windows: rows around the
row list's and the waves' splits, one residual column, residuals too large for the step
kernel to hold, zero residuals at whole orders, full rank at the first and at a later
order, vanishing columns."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

P30, P60, PBIG = 998244353, 1152921504556515329, 18446744073709551557

# (p, m, n, orders): shapes that the rule gives to single orders
SHAPES = [
    (P30, 200, 26, (5,)), (P30, 256, 33, (4,)), (P30, 256, 128, (3,)),
    (P60, 64, 48, (1, 2, 6)), (P60, 100, 12, (7,)), (P60, 128, 1, (9, 18)), (P60, 130, 33, (5,)),
    (P60, 201, 5, (11,)), (P60, 256, 60, (3,)), (P60, 67, 65, (5,)), (P60, 128, 128, (3,)),
    (PBIG, 48, 12, (9,)), (PBIG, 64, 16, (1, 8)), (PBIG, 100, 1, (17,)), (PBIG, 70, 66, (4,)),
    (PBIG, 256, 3, (6,)),
]
KINDS = ["uniform", "lowrank", "sparse", "zero_orders", "full"]


def residual(rng, kind, m, n, order, p):
    F = rng.integers(0, p - 1, (m, n, order), dtype=np.uint64)
    if kind == "lowrank":  # equal columns, zero rows at every other order
        F[:, n // 2:, :] = F[:, :1, :]
        F[: m // 3, :, ::2] = 0
    elif kind == "sparse":
        F *= (rng.random(F.shape) < 0.1).astype(np.uint64)
    elif kind == "zero_orders":  # nothing to do at the first orders, then at later ones too
        F[:, :, : (order + 1) // 2] = 0
        F[m // 2:] = 0
    return F


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("p,m,n,orders", SHAPES)
def test_mbasis_single_orders(p, m, n, orders, kind):
    import pml_amd
    rng = np.random.default_rng(1000 * m + n)
    if kind == "full":  # as many columns as rows: full rank at the first order
        if m > 70:
            pytest.skip("smaller shapes suffice")
        n = m
    ctx = pml_amd.Context(p)
    for order in orders:
        F = residual(rng, kind, m, n, order, p)
        if kind == "full" and order > 2:
            F[:, :, 0] = 0  # at the second order
        shift = rng.integers(0, 3, m).astype(np.int64)
        P_ref, s_ref = O.mbasis(F, order, shift, p)
        P_dev, s_dev = ctx.mbasis(F, order, shift)
        assert np.array_equal(O.normalise(P_dev), O.normalise(P_ref))
        assert np.array_equal(s_dev, s_ref)
