"""What the MFMA pointwise kernel hands to the inverse transform, on the CPU.

The kernel leaves the REDC of a dot product of k residues, V 2^-64 mod p, as it is
where host_redc_small says so and after a Barrett step otherwise.  The lazy
butterflies (p < 2^60) take inputs below 8p, the strict ones hold values below 2p and
let sums pass 2^64 on larger ones.  host_redc_small is compiled from the library's
header; the largest outputs and the strict inverse stages are restated in Python
integers (the device's words: any sum past 2^64 is caught)."""
import ctypes
import os
import subprocess

import pytest

from pml_amd import build

M64 = (1 << 64) - 1
STRICT = [1152921504618381313, 1729382256876716033, 2305843009211596801]
LAZY = [1152921504556515329, 1125899915231233, 1085276161]


@pytest.fixture(scope="module")
def redc_small(tmp_path_factory):
    d = tmp_path_factory.mktemp("redc")
    src = d / "redc.cpp"
    src.write_text('#include "host_arith.hpp"\n'
                   'extern "C" int redc_small(uint64_t p, int64_t k) { return pmlg::host_redc_small(p, k); }\n')
    so = d / "redc.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", build.CSRC, str(src), "-o", str(so)],
                   check=True)
    f = ctypes.CDLL(str(so)).redc_small
    f.argtypes, f.restype = [ctypes.c_uint64, ctypes.c_int64], ctypes.c_int
    return f


def redc(V, p):
    m = (-V * pow(p, -1, 1 << 64)) & M64
    return (V + m * p) >> 64


def output(V, p, small):
    """the kernel's word for a dot product V"""
    u = redc(V, p)
    assert u <= M64
    return u if small else u - ((u * ((1 << 64) // p)) >> 64) * p


def kmax(p):
    """largest k of the MFMA kernel (k (p - 1)^2 + (p + 1) 2^64 < 2^128)"""
    return min(4064, ((1 << 128) - 1 - ((p + 1) << 64)) // (p - 1) ** 2)


@pytest.mark.parametrize("p", STRICT + LAZY)
def test_largest_output_is_within_the_inverse_range(redc_small, p):
    limit = 2 * p if p >= 1 << 60 else 8 * p
    for k in range(1, kmax(p) + 1):
        if redc_small(p, k):
            # (V + m p) >> 64 at the largest V and any m
            assert (k * (p - 1) ** 2 + M64 * p) >> 64 < limit, k
        # (otherwise the Barrett step's result is below 2p)


def strict_inverse(x, p, w):
    """The device's strict decimation in time: bit-reversed in, natural out, unscaled"""
    def word(v):
        assert 0 <= v <= M64, "a word overflows"
        return v

    def add_2p(a, b):
        s = word(a + b)
        return s - 2 * p if s >= 2 * p else s

    def shoup(v, c):
        q = (v * ((c << 64) // p)) >> 64
        return word(v * c - q * p)

    x, n, h = list(x), len(x), 1
    wi = pow(w, -1, p)
    while h < n:
        for i0 in range(0, n, 2 * h):
            for j in range(h):
                a, c = x[i0 + j], x[i0 + j + h]
                v = c if j == 0 else shoup(c, pow(wi, j * (n // (2 * h)), p))
                x[i0 + j] = add_2p(a, v)
                d = word(a + 2 * p - v)
                x[i0 + j + h] = d - 2 * p if d >= 2 * p else d
        h *= 2
    return x


@pytest.mark.parametrize("p", STRICT)
@pytest.mark.parametrize("n", [4, 8, 16])
def test_strict_inverse_of_minus_one_matrices(redc_small, p, n):
    """Constant matrices of -1: every evaluation of every entry is p - 1"""
    g = next(g for g in range(2, 100) if pow(g, (p - 1) // 2, p) == p - 1)
    w = pow(g, (p - 1) // n, p)
    for k in range(1, kmax(p) + 1):
        u = output(k * (p - 1) ** 2, p, redc_small(p, k))
        x = strict_inverse([u] * n, p, w)
        assert x[0] % p == k * n * pow(1 << 64, -1, p) % p
        assert all(v % p == 0 for v in x[1:]), k
