"""Work that a user of the library has it do, as timed cases.

    listed()             the cases, each a dict of plain values
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what a program holds before the call, on the GPU
    run(state)           one pass through the public entry points; its outputs
    work(case)           bytes and operations one pass cannot do without
    exact(case, seed)    the outputs in Python integers, where that is quick

Operands are uniform residues, as the coefficients of the intermediate
matrices of approximant and kernel computations are.  Four moduli stand for
the word sizes and paths in use: 998244353 (32-bit words on the device),
2^60 - 3 2^24 + 1 (64-bit words, transforms modulo p) and two 60-bit primes of
the reference's published benchmarks without the roots of unity that a
transform needs (products through the multi-prime path).

Every family reads device memory that the program owns and writes device
memory that it owns; the calls run on the context's (the plan's) own stream.
"""
import ctypes
import math
import random

import numpy as np
import torch

import pml_amd

P30 = 998244353
P60 = 1152921504556515329
PNF = 723501827743829161   # the published product benchmark's prime
PNK = 820293421056153991   # the published kernel-basis benchmark's prime

_i64p = ctypes.POINTER(ctypes.c_int64)


def _mul(name, m, k, n, la, lb, p):
    return {"name": name} | _mul_of(m, k, n, la, lb, p)


def _mul_of(m, k, n, la, lb, p):
    return {"family": "mul", "m": m, "k": k, "n": n, "la": la, "lb": lb, "p": p}


def listed():
    return [
        # the smallest calls: latency, launches and host work are everything
        _mul("mul_4x4_len16_p60", 4, 4, 4, 16, 16, P60),
        # an ordinary small product modulo a 30-bit prime
        _mul("mul_16x16_len256_p30", 16, 16, 16, 256, 256, P30),
        # the library's headline product, one call at a time
        _mul("mul_32x32_len4096_p60", 32, 32, 32, 4096, 4096, P60),
        # odd dimensions, operands of different lengths
        _mul("mul_37x21x50_len3001x1200_p60", 37, 21, 50, 3001, 1200, P60),
        # large dimensions at moderate length: the pointwise products dominate
        _mul("mul_128x128_len500_p60", 128, 128, 128, 500, 500, P60),
        # few long entries: transforms longer than one workgroup's memory
        _mul("mul_4x4_len200000_p60", 4, 4, 4, 200000, 200000, P60),
        # the headline shape modulo a 60-bit prime without roots of unity
        _mul("mul_32x32_len4096_nonfft", 32, 32, 32, 4096, 4096, PNF),
        # the middle product at the top of a PM-Basis of order 2048
        {"name": "mulmid_64x64x32_order2048_p30", "family": "mulmid", "m": 64, "n": 32,
         "order": 2048, "p": P30},
        # the headline product in batches: one plan, replayed
        {"name": "batch_16_32x32_len4096_p60", "family": "batch", "count": 16, "dim": 32,
         "len": 4096, "shapes": 0, "p": P60},
        # many products of uneven shapes, lengths and word sizes in one plan
        {"name": "batch_48_uneven", "family": "batch", "count": 48, "dim": 64, "len": 4096,
         "shapes": 4, "p": 0},
        # PM-Basis of the golden fixture's shape (order 2048)
        {"name": "pmbasis_64x32_order2048_p30", "family": "pmbasis", "m": 64, "n": 32,
         "order": 2048, "p": P30, "shifted": False},
        # kernel basis of the published table's shape, at half its degree
        {"name": "kernel_32x17_deg512_nonfft", "family": "kernel", "m": 32, "n": 17, "deg": 512,
         "p": PNK},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["mul", "mul", "mul", "mulmid", "batch", "pmbasis", "kernel"])
    if family == "mul":
        p = rng.choice([P30, P60, P60, PNF])
        m, k, n = (_log(rng, 2, 128) for _ in range(3))
        la = _log(rng, 4, 200000)
        lb = max(2, int(la * rng.uniform(0.2, 1.0)))
        # within the listed cases' cost: points times entries and products
        while (m * k + k * n + m * n) * (la + lb) > 3 * 2 ** 23 or m * k * n * (la + lb) > 2 ** 30:
            la, lb = max(4, la * 3 // 4), max(2, lb * 3 // 4)
        return _mul_of(m, k, n, la, lb, p)
    if family == "mulmid":
        m = _log(rng, 4, 64)
        return {"family": "mulmid", "m": m, "n": rng.randint((m + 3) // 4, m),
                "order": _log(rng, 33, 2048), "p": rng.choice([P30, P60])}
    if family == "batch":
        return {"family": "batch", "count": rng.randint(8, 32),
                "dim": rng.randint(16, 64), "len": _log(rng, 256, 4096),
                "shapes": rng.randint(1, 10 ** 6), "p": rng.choice([0, P30, P60])}
    if family == "pmbasis":
        m = rng.randint(8, 64)
        return {"family": "pmbasis", "m": m, "n": rng.randint(m // 4, m * 3 // 4),
                "order": _log(rng, 40, 900), "p": rng.choice([P30, P60, PNK]),
                "shifted": rng.random() < 0.5}
    m = rng.randint(8, 32)
    return {"family": "kernel", "m": m, "n": rng.randint(m // 4, m // 2 + 1),
            "deg": _log(rng, 32, 400), "p": rng.choice([P30, P60, PNK])}


# ---------------------------------------------------------------------------
# what a program holds
# ---------------------------------------------------------------------------
_CONTEXTS = {}


def _context(p):
    """One context per modulus for the life of the process, as programs keep it."""
    if p not in _CONTEXTS:
        _CONTEXTS[p] = pml_amd.Context(p)
    return _CONTEXTS[p]


def _shapes(case):
    """(p, m, k, n, la, lb) of every product of a batch (shapes 0: all alike)."""
    if case["shapes"] == 0:
        d = case["dim"]
        return [(case["p"], d, d, d, case["len"], case["len"])] * case["count"]
    rng = random.Random(case["shapes"])
    out = []
    for _ in range(case["count"]):
        p = case["p"] or rng.choice([P30, P60])
        m, k, n = (rng.randint(2, case["dim"]) for _ in range(3))
        out.append((p, m, k, n, _log(rng, 16, case["len"]), _log(rng, 16, case["len"])))
    return out


class _Residues:
    """Uniform residues from one seeded generator on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def __call__(self, p, *shape):
        return torch.randint(0, p, shape, generator=self.g, device="cuda", dtype=torch.int64)


class _Plan:
    """A planned batch on the program's own tensors (pmlg_batch_plan)."""

    def __init__(self, shapes, rand):
        self.keep, self.out = [], []
        descs = (pml_amd.MulDesc * len(shapes))()
        for d, (p, m, k, n, la, lb) in zip(descs, shapes):
            A, B = rand(p, m, k, la), rand(p, k, n, lb)
            C = torch.zeros(m, n, la + lb - 1, device="cuda", dtype=torch.int64)
            self.keep += [A, B]
            self.out.append(C)
            d.ctx, d.A, d.B, d.C = _context(p).handle, A.data_ptr(), B.data_ptr(), C.data_ptr()
            d.m, d.k, d.n, d.lenA, d.lenB = m, k, n, la, lb
            d.method, d.config = pml_amd.METHOD_AUTO, -1
        torch.cuda.synchronize()  # the inputs are ready before the plan's stream reads them
        h = ctypes.c_void_p()
        _check(pml_amd.lib().pmlg_batch_plan_create(ctypes.byref(h), descs, len(shapes),
                                                    pml_amd.BATCH_GRAPH))
        self.handle = h.value

    def run(self):
        _check(pml_amd.lib().pmlg_batch_plan_run(self.handle, None))

    def __del__(self):
        if getattr(self, "handle", None):
            torch.cuda.synchronize()
            pml_amd.lib().pmlg_batch_plan_destroy(self.handle)
            self.handle = None


def _check(status):
    if status != 0:
        raise pml_amd.PmlgError(status, pml_amd.lib().pmlg_last_error().decode())


def prepare(case, seed):
    rand = _Residues(seed)
    s = {"case": case}
    family = case["family"]
    if family == "batch":
        s["plan"] = _Plan(_shapes(case), rand)
        return s
    p = case["p"]
    s["ctx"] = _context(p)
    if family == "mul":
        m, k, n, la, lb = (case[x] for x in ("m", "k", "n", "la", "lb"))
        s["A"], s["B"] = rand(p, m, k, la), rand(p, k, n, lb)
        s["C"] = torch.zeros(m, n, la + lb - 1, device="cuda", dtype=torch.int64)
    elif family == "mulmid":
        m, n, order = case["m"], case["n"], case["order"]
        half = order // 2
        s["A"], s["B"] = rand(p, m, m, half + 1), rand(p, m, n, order)
        s["C"] = torch.zeros(m, n, order - half, device="cuda", dtype=torch.int64)
    elif family == "pmbasis":
        m, n, order = case["m"], case["n"], case["order"]
        s["F"] = rand(p, m, n, order)
        s["P"] = torch.zeros(m, m, order + 1, device="cuda", dtype=torch.int64)
        s["shift"] = np.zeros(m, dtype=np.int64)
        if case["shifted"]:
            s["shift"] = np.random.default_rng(int(seed)).integers(0, order // 4 + 1, m)
    else:
        m, n, deg = case["m"], case["n"], case["deg"]
        s["F"] = rand(p, m, n, deg + 1)
        # room for the generic degree n deg / (m - n) twice over
        s["cap"] = 2 * (n * (deg + 1) // (m - n)) + 64
        s["K"] = torch.zeros(m, m, s["cap"], device="cuda", dtype=torch.int64)
    torch.cuda.synchronize()  # the context's stream may read the inputs from here on
    return s


def run(s):
    case = s["case"]
    family = case["family"]
    if family == "mul":
        s["ctx"].mul_dev(s["C"].data_ptr(), s["A"].data_ptr(), s["B"].data_ptr(), case["m"],
                         case["k"], case["n"], case["la"], case["lb"])
        return s["C"]
    if family == "mulmid":
        m, n, order = case["m"], case["n"], case["order"]
        half = order // 2
        _check(pml_amd.lib().pmlg_polmat_mulmid_dev(
            s["ctx"].handle, s["C"].data_ptr(), s["A"].data_ptr(), s["B"].data_ptr(), m, m, n,
            half + 1, order, half, order, pml_amd.METHOD_AUTO, None))
        return s["C"]
    if family == "batch":
        s["plan"].run()
        return s["plan"].out
    if family == "pmbasis":
        m, n, order = case["m"], case["n"], case["order"]
        shift = s["shift"].copy()
        # coefficients past the basis's length stay the zeros of the program's buffer
        s["ctx"].pmbasis_dev(s["P"].data_ptr(), order + 1, shift, s["F"].data_ptr(), m, n, order,
                             order)
        return {"basis": s["P"], "shift": shift}
    m, n = case["m"], case["n"]
    shift, piv = np.zeros(m, dtype=np.int64), np.zeros(m, dtype=np.int64)
    length, nullity = ctypes.c_int64(0), ctypes.c_int64(0)
    _check(pml_amd.lib().pmlg_kernel_basis_dev(
        s["ctx"].handle, s["K"].data_ptr(), s["cap"], ctypes.byref(length), ctypes.byref(nullity),
        piv.ctypes.data_as(_i64p), shift.ctypes.data_as(_i64p), s["F"].data_ptr(), m, n,
        case["deg"] + 1, pml_amd.KERNEL_ZLS, pml_amd.METHOD_AUTO, None))
    k = nullity.value
    return {"kernel": s["K"], "length": length.value, "nullity": k, "pivots": piv[:k],
            "degrees": shift[:k]}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _product_ops(m, k, n, la, lb, lc):
    """Modular operations of a product by evaluation at lc points: two per
    multiply-add of the pointwise products, three per butterfly."""
    lg = max(1.0, math.log2(lc))
    return 2.0 * m * k * n * lc + 1.5 * (m * k + k * n + m * n) * lc * lg


def work(case):
    family = case["family"]
    if family == "batch":
        b = f = 0.0
        for _, m, k, n, la, lb in _shapes(case):
            b += 8.0 * (m * k * la + k * n * lb + m * n * (la + lb - 1))
            f += _product_ops(m, k, n, la, lb, la + lb - 1)
        return {"bytes": b, "flops": f}
    if family == "mul":
        m, k, n, la, lb = (case[x] for x in ("m", "k", "n", "la", "lb"))
        return {"bytes": 8.0 * (m * k * la + k * n * lb + m * n * (la + lb - 1)),
                "flops": _product_ops(m, k, n, la, lb, la + lb - 1)}
    if family == "mulmid":
        m, n, order = case["m"], case["n"], case["order"]
        half = order // 2
        return {"bytes": 8.0 * (m * m * (half + 1) + m * n * (order + order - half)),
                "flops": _product_ops(m, m, n, half + 1, order, order)}
    # bases: the input once, the basis once; a middle product and a product
    # at every node of the divide and conquer on the order
    m, n = case["m"], case["n"]
    order = case["order"] if family == "pmbasis" else 2 * (case["deg"] * n // (m - n) + case["deg"])
    deg = order * n // m + 1  # generic degree of the basis
    f, half = 0.0, order // 2
    nodes = 1
    while half >= 1:
        h = max(1, half * n // m)
        f += nodes * (_product_ops(m, m, n, h, 2 * half, 2 * half) + _product_ops(m, m, m, h, h, 2 * h))
        half //= 2
        nodes *= 2
    read = order if family == "pmbasis" else case["deg"] + 1
    out = m * m * deg if family == "pmbasis" else (m - n) * m * (case["deg"] * n // (m - n) + 1)
    return {"bytes": 8.0 * (m * n * read + out), "flops": f}


# ---------------------------------------------------------------------------
# the same in Python integers
# ---------------------------------------------------------------------------
def _pack(row, width):
    return int.from_bytes(b"".join(int(x).to_bytes(width, "little") for x in row), "little")


def _product(A, B, p):
    """A * B mod p by Kronecker substitution (arrays m x k x la, k x n x lb)."""
    m, k, la = A.shape
    n, lb = B.shape[1:]
    bits = 2 * (p - 1).bit_length() + (k * min(la, lb)).bit_length() + 1
    width = (bits + 7) // 8
    PA = [[_pack(A[i, t], width) for t in range(k)] for i in range(m)]
    PB = [[_pack(B[t, j], width) for j in range(n)] for t in range(k)]
    lc = la + lb - 1
    out = np.zeros((m, n, lc), dtype=np.int64)
    for i in range(m):
        for j in range(n):
            v = sum(PA[i][t] * PB[t][j] for t in range(k)).to_bytes(width * (lc + 1), "little")
            out[i, j] = [int.from_bytes(v[d * width:(d + 1) * width], "little") % p for d in range(lc)]
    return out


def exact(case, seed):
    if case["family"] not in ("mul", "mulmid"):
        return None
    if case["family"] == "mul":
        m, k, n, lc = case["m"], case["k"], case["n"], case["la"] + case["lb"]
    else:
        m, k, n, lc = case["m"], case["m"], case["n"], 2 * case["order"]
    if m * k * n * lc ** 1.6 > 1e8 or m * n * lc > 2e6:
        return None
    s = prepare(case, seed)
    C = _product(s["A"].cpu().numpy(), s["B"].cpu().numpy(), case["p"])
    if case["family"] == "mulmid":
        half = case["order"] // 2
        C = np.ascontiguousarray(C[:, :, half:case["order"]])
    return C
