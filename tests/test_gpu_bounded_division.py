"""FP64 two-step tiles divide without the operand scaling where their values
allow it and march again with IEEE divisions where they do not: fields with one
value of 2^299, 2^300 or more, an infinity, a NaN or a zero divisor (a
difference of exactly -1e-6) somewhere in a tile, and material constants at
and past the limit, bit for bit against the oracle."""
import numpy as np
import pytest

import golden_data as gd
import le2d_amd
from oracle import Oracle

pytestmark = pytest.mark.gpu
ARGS = (0.2, (1.0, 0.9), (2.0, 1.0, 1.5))


def _run(g0, args, lanes, seg, steps):
    ny, nx = g0.shape[:2]
    with le2d_amd.Task(nx, ny, *args) as t:
        t.load(g0)
        t.set_step_pairs(seg)
        t.set_step_pair_window(lanes)
        t.step_n(steps)
        return t.grid().copy()


@pytest.mark.parametrize("lanes", [64, 128])
@pytest.mark.parametrize("value", [2.0**299, -(2.0**300), 2.0**900, np.inf, np.nan, 1e-310])
@pytest.mark.parametrize("at", [(0, 0, 0), (40, 118, 2), (24, 60, 4), (63, 200, 1)])
def test_one_value_outside_the_bounds(lanes, value, at):
    g0 = np.random.default_rng(5).standard_normal((64, 201, 5))
    g0[at] = value
    got = _run(g0, ARGS, lanes, 24, 4)
    ref = g0.copy()
    with np.errstate(all="ignore"):
        Oracle(np.float64).run(ref, *ARGS, 4)
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan)
    assert gd.same_bits(got[~nan], ref[~nan])


@pytest.mark.parametrize("lanes", [64, 128])
def test_zero_divisors(lanes):
    rng = np.random.default_rng(6)
    g0 = np.zeros((50, 130, 5))
    g0[..., :2] = rng.choice([0.0, -1e-6, 1e-6, 1.0], size=(50, 130, 2))
    got = _run(g0, ARGS, lanes, 16, 4)
    ref = g0.copy()
    Oracle(np.float64).run(ref, *ARGS, 4)
    assert gd.same_bits(got, ref)


@pytest.mark.parametrize("rho", [1e-300, 2.0**-62, 2.0**-58, 2.0**58, 2.0**62, 1e300])
def test_constants_outside_the_bounds(rho):
    g0 = np.random.default_rng(7).standard_normal((40, 130, 5))
    args = (0.2, (1.0, 0.9), (2.0, 1.0, rho))
    got = _run(g0, args, 128, 16, 2)
    ref = g0.copy()
    with np.errstate(all="ignore"):
        Oracle(np.float64).run(ref, *args, 2)
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan)
    assert gd.same_bits(got[~nan], ref[~nan])
