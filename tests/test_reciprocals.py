"""The reference typing's reciprocals (p2z-tests_amd/csrc/p2z_lane.hpp) stand for
the reference's double divisions rounded to float (OMP:521, 628, 637).

ref_inv_det: 1/det through two Newton steps is rounded to double from a value
within 2^-86 of it, then to float.  That differs from the division's float only
if the double division and it fall on two sides of a rounding boundary next to
the middle of two floats, that is if 1/det lies within 2^-86 of one of the 2^25
points half a double's step on either side of a 25-bit odd mantissa.  The
enumeration here takes the double nearest to each point's reciprocal, exactly."""
from __future__ import annotations

import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CHECK = os.path.join(HERE, "..", "p2z-tests_amd", "bin", "p2z_reciprocal_check")


def nearest_double_reciprocal(lo: int, hi: int) -> float:
    """Smallest |d b - 2^106| / 2^106 over the doubles d and the points b of the
    middles lo .. hi - 1.  A point is the 54-bit integer b = 2^29 m +- 1 (m a
    25-bit odd integer), and d a 53-bit integer with d b next to 2^106.  The
    difference is below b, so that 64 bits hold it."""
    best = 1 << 62
    m = np.arange(lo, hi, dtype=np.uint64) * np.uint64(2) + np.uint64(1)
    for s in (-1, 1):
        b = (m << np.uint64(29)).astype(np.int64) + s
        d = np.rint(2.0 ** 106 / b.astype(np.float64)).astype(np.int64).view(np.uint64)
        for k in (-2, -1, 0, 1, 2):
            with np.errstate(over="ignore"):
                r = ((d + np.uint64(k % (1 << 64))) * b.view(np.uint64)).view(np.int64)  # 2^106 is 0 mod 2^64
            best = min(best, int(np.abs(r).min()))
    return best / 2.0 ** 106


def test_enumeration_against_exact_integers():
    rng = np.random.default_rng(1)
    for m in rng.integers(1 << 23, 1 << 24, 50).tolist():
        exact = min(abs(d * b - (1 << 106)) for s in (-1, 1) for b in [(2 * m + 1 << 29) + s]
                    for d in [(1 << 106) // b, (1 << 106) // b + 1])
        assert nearest_double_reciprocal(m, m + 1) == exact / 2.0 ** 106


def test_no_double_has_a_reciprocal_next_to_a_boundary():
    step = 1 << 20
    best = min(nearest_double_reciprocal(lo, lo + step) for lo in range(1 << 23, 1 << 24, step))
    print(f"nearest: 2^{np.log2(best):.2f}", flush=True)
    assert best > 2.0 ** -86


@pytest.mark.gpu
def test_on_the_gpu():
    run = subprocess.run([CHECK], capture_output=True, text=True, timeout=100)
    print(run.stdout, run.stderr, flush=True)
    assert run.returncode == 0
    res = {ln.split()[0]: ln.split() for ln in run.stdout.splitlines()}
    assert int(res["ref_rcp"][2]) == 1 << 32
    assert int(res["fast_rcp"][2]) == 2 * (200 * (1 << 23) - 1)  # |x| in (2^-100, 2^100), both signs
    for name in ("fast_rcp", "ref_rcp", "ref_inv_det"):
        assert int(res[name][4]) == 0, name
    # one Newton step squares the hardware's error, two bring 2^-24 below 2^-86
    assert float(res["rcp_f64"][6]) < 2.0 ** -24
