"""Products of constant matrices (lenA = lenB = 1): one-point transforms, by every method
and configuration, against the oracle; and the sizes that the no-allocation entry point
takes, whose scratch holds one evaluation of every entry."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

P30, P60, P62 = 998244353, 1152921504556515329, 4611686018326724609
P61 = 2305843009211596801  # MFMA kernel and strict butterflies


@pytest.fixture(scope="module")
def pml():
    import pml_amd
    return pml_amd


@pytest.mark.parametrize("p", [2, 3, P30, P60, P61, P62])
@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (3, 5, 2), (16, 16, 16), (17, 33, 18), (40, 60, 257)])
def test_constant_products(pml, p, m, k, n):
    rng = np.random.default_rng(m + n)
    A = rng.integers(0, p, (m, k, 1), dtype=np.uint64)
    B = rng.integers(0, p, (k, n, 1), dtype=np.uint64)
    A[0], B[:, 0] = p - 1, p - 1
    want = O.polmat_mul(A, B, p)
    with pml.Context(p) as ctx:
        for method in ("auto", "plain"):
            assert np.array_equal(ctx.mul(A, B, method=method), want), method
        # the constant coefficient of a longer product
        A2 = np.concatenate([A, rng.integers(0, p, (m, k, 4), dtype=np.uint64)], axis=2)
        assert np.array_equal(ctx.mulmid(A2, B, 0, 1), want)
        for c in range(pml.num_configs()):
            if pml.config_valid(ctx, m, k, n, 1, 1, c):
                got = pml.mul_batch([(ctx, A, B), (ctx, A[::-1].copy(), B)], config=c)
                assert np.array_equal(got[0], want), c
                assert np.array_equal(got[1], want[::-1]), c


def test_noalloc_holds_one_point_per_entry(pml):
    """4200 x 4 by 4 x 4200: 141 MB of evaluations at one point, more than the 256 MiB
    at two"""
    L = pml.lib()
    p, m, k = P60, 4200, 4
    rng = np.random.default_rng(1)
    A = rng.integers(0, p, (m, k, 1), dtype=np.uint64)
    B = rng.integers(0, p, (k, m, 1), dtype=np.uint64)
    with pml.Context(p) as ctx:
        dA, dB = pml.DeviceArray(ctx, A.nbytes), pml.DeviceArray(ctx, B.nbytes)
        dC = pml.DeviceArray(ctx, m * m * 8)
        dA.upload(A)
        dB.upload(B)
        # root tables of one point, by a small product
        assert L.pmlg_polmat_mul_dev(ctx.handle, dC.ptr, dA.ptr, dB.ptr, 2, 2, 2, 1, 1, 0, None) == 0
        st = L.pmlg_polmat_mul_dev_noalloc(ctx.handle, dC.ptr, dA.ptr, dB.ptr, m, k, m, 1, 1, 0, None)
        assert st == 0, L.pmlg_last_error()
        ctx.sync()
        C = np.zeros((m, m), dtype=np.uint64)
        dC.download(C)
        for d in (dA, dB, dC):
            d.free()
    a, b = A[..., 0].astype(object), B[..., 0].astype(object)
    for i in (0, 1, 2099, m - 1):
        assert np.array_equal(C[i].astype(object), a[i].dot(b) % p), i
