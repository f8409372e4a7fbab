"""Every transform kernel launched with more than 64 KiB of dynamic LDS has a once-only
flag of its own for raising its limit (CPU: the symbols of the built library).  Many of
the kernels share one function type, and a flag per type raised the limit of whichever
was launched first only."""
import os
import re
import subprocess

import pytest

from pml_amd import build

# <Win, W, ...> and <W, Wout, ...>: the word type is m (64 bits, 2^13 points: 67,584
# bytes) or j (32 bits, 2^14 points: the same)
KERNEL = re.compile(r"ntt_(fwd|inv)_regI([jm])([jm])Lb[01]ELi(\d+)E(?:Li\dE)+(?:Lb[01]E)?E")


def symbols():
    if not os.path.exists(build.LIB):
        pytest.fail("libpmlgpu.so is not built (python -m pml_amd.build)")
    out = subprocess.run(["nm", build.LIB], stdout=subprocess.PIPE, text=True, check=True).stdout
    return [line.split()[-1] for line in out.splitlines()]


def test_one_flag_per_kernel_above_the_default_limit():
    syms = symbols()
    large = set()
    for s in syms:
        k = KERNEL.search(s)
        if k and "__device_stub__" in s:
            word = k.group(3) if k.group(1) == "fwd" else k.group(2)
            if int(k.group(4)) >= (13 if word == "m" else 14):
                large.add(k.group(0))
    assert len(large) == 36  # 10 forward kernels x {32-bit, strict, lazy}, 2 inverse ones x the same
    flags = [KERNEL.search(s) for s in syms if "launch_xform" in s and s.endswith("6raised")]
    assert all(flags)
    names = sorted(k.group(0) for k in flags)
    assert names == sorted(large)
