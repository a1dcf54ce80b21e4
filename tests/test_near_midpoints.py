"""The quantizer's check for values whose E2M1 code the conversion instruction may get wrong (csrc/quantize_kernel.h,
``e2m1_try8``), restated on the CPU: it has to find every value for which rounding to nearest, ties to even, is not what the
reference's biased comparison gives."""
import numpy as np
import torch

import oracle as O

GRID = np.array([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0])
MIDPOINTS = np.array([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], dtype=np.float32)


def flagged(x):
    low = (x.view(np.uint32) << np.uint32(11)) + np.uint32(128 << 11)
    return low < np.uint32(256 << 11)


def nearest_even(x):
    a = np.abs(x.astype(np.float64))
    i = np.searchsorted(GRID, a, side="right") - 1
    lo, hi = GRID[i], GRID[np.minimum(i + 1, 7)]
    up = (a - lo > hi - a) | ((a - lo == hi - a) & (i % 2 == 1))
    code = np.where((i < 7) & up, i + 1, i)
    return code


def rule(x):
    return (O.encode_e2m1(torch.from_numpy(x)).numpy() & 7).astype(np.int64)


def test_every_value_that_rounds_otherwise_is_found():
    rng = np.random.default_rng(0)
    around = (MIDPOINTS.view(np.uint32)[:, None] + np.arange(-4000, 4001, dtype=np.int64)[None, :]).astype(np.uint32).ravel().view(np.float32)
    zeros = np.zeros(1, dtype=np.float32)
    x = np.concatenate([around, rng.uniform(0, 8, 1 << 20).astype(np.float32), np.exp2(rng.uniform(-30, 3, 1 << 18)).astype(np.float32), GRID.astype(np.float32), zeros])
    x = np.concatenate([x, -x])
    other = nearest_even(x) != rule(x)
    assert other.any() and flagged(x)[other].all()
    assert flagged(x[len(around):len(around) + (1 << 20)]).mean() < 0.001
    # a power of two in front changes nothing: the check looks at the mantissa
    for e in (-99, -20, 7, 100):
        assert (flagged(np.ldexp(around, e)) == flagged(around)).all()


def test_ties_themselves_are_found():
    assert flagged(MIDPOINTS).all() and flagged(-MIDPOINTS).all()
