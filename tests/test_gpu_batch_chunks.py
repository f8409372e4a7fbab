"""Batches whose evaluations exceed one chunk (200 MB): the same products against
the oracle, eager, as a graph and stage by stage, and a batch in which one
product's output is another's input, which sees that input as it was."""
import ctypes

import numpy as np
import pytest

import pml_amd
from oracle import oracle as O

pytestmark = pytest.mark.gpu

P60 = 1152921504556515329
K, LEN = 200, 12000  # 401 transforms of 2^15 points: 105 MB a product


@pytest.fixture(scope="module")
def ctx():
    return pml_amd.Context(P60)


def operands(count, seed):
    rng = np.random.default_rng(seed)
    return [(rng.integers(0, P60, (1, K, LEN), dtype=np.uint64),
             rng.integers(0, P60, (K, 1, LEN), dtype=np.uint64)) for _ in range(count)]


def test_chunks_match_oracle(ctx):
    data = operands(3, 1)
    rng = np.random.default_rng(2)
    data.append((rng.integers(0, P60, (3, 2, 40), dtype=np.uint64),
                 rng.integers(0, P60, (2, 5, 7), dtype=np.uint64)))
    want = [O.polmat_mul(A, B, P60, method="ntt") for A, B in data]
    items = [(ctx, A, B) for A, B in data]
    for graph in (False, True):
        with pml_amd.BatchPlan(items, graph=graph) as plan:
            if graph:
                plan.time_stages(2)
            for _ in range(3):
                plan.run(None)
            plan.sync()
            for got, ref in zip(plan.results(), want):
                assert np.array_equal(got, ref)


def test_output_over_input(ctx):
    (A0, B0), (A1, B1) = operands(2, 3)
    lc = 2 * LEN - 1
    bufs = []
    for x in (A0, B0, A1, B1):
        d = pml_amd.DeviceArray(ctx, x.nbytes)
        d.upload(x)
        bufs.append(d)
    out = pml_amd.DeviceArray(ctx, lc * 8)
    descs = (pml_amd.MulDesc * 2)()
    # product 0 writes where product 1's A lies
    for d, a, b, c in ((descs[0], bufs[0], bufs[1], bufs[2]), (descs[1], bufs[2], bufs[3], out)):
        d.ctx, d.A, d.B, d.C = ctx.handle, a.ptr, b.ptr, c.ptr
        d.m, d.k, d.n, d.lenA, d.lenB = 1, K, 1, LEN, LEN
        d.method, d.config = 0, 2
    assert pml_amd.lib().pmlg_polmat_mul_batch(descs, 2, None) == 0
    got = np.empty(lc, dtype=np.uint64)
    out.download(got)
    assert np.array_equal(got, O.polmat_mul(A1, B1, P60, method="ntt")[0, 0])
