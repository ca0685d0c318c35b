"""The two-step pass in blocks held in registers, the default of grids that do not
fill the device (each size below gets another block height): sizes at and one
past a block's 56 columns and its rows, grids smaller than a wavefront's rows,
values and divisors out of the bounded division's range; FP64 bit for bit
against the oracle, FP32 bit for bit against single steps."""
import numpy as np
import pytest

import golden_data as gd
import le2d_amd
from oracle import Oracle

pytestmark = pytest.mark.gpu
ARGS = (0.2, (1.0, 0.9), (2.0, 1.0, 1.5))
SIZES = [(3, 3), (4, 5), (56, 8), (57, 9), (113, 4), (3, 1000), (250, 296), (250, 297), (392, 400),
         (393, 401), (505, 504), (504, 505), (616, 640), (617, 641), (727, 720), (728, 721),
         (1031, 517), (890, 896)]


def _run(g0, dtype, steps, pairs=None):
    ny, nx = g0.shape[:2]
    with le2d_amd.Task(nx, ny, *ARGS, dtype=dtype) as t:
        t.load(g0)
        if pairs is not None:
            t.set_step_pairs(pairs)
        t.step_n(steps)  # fewer than 8: the default shape
        return t.grid().copy()


@pytest.mark.parametrize("nx,ny", SIZES)
def test_blocks_match_oracle(nx, ny):
    g0 = np.random.default_rng(nx * ny).standard_normal((ny, nx, 5))
    ref = g0.copy()
    Oracle(np.float64).run(ref, *ARGS, 4)
    assert gd.same_bits(_run(g0, np.float64, 4), ref)


@pytest.mark.parametrize("nx,ny", SIZES)
def test_fp32_blocks_equal_single_steps(nx, ny):
    g0 = np.random.default_rng(nx * ny).standard_normal((ny, nx, 5)).astype(np.float32)
    assert gd.same_bits(_run(g0, np.float32, 4), _run(g0, np.float32, 4, pairs=0))


@pytest.mark.parametrize("value", [2.0**900, np.inf, np.nan, 1e-310])
def test_values_outside_the_bounds(value):
    g0 = np.random.default_rng(8).standard_normal((70, 130, 5))
    g0[31, 57, 3] = value
    g0[10, 100:104, 0] = [0.0, -1e-6, -2e-6, 1e-6]
    ref = g0.copy()
    with np.errstate(all="ignore"):
        Oracle(np.float64).run(ref, *ARGS, 4)
    got = _run(g0, np.float64, 4)
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan)
    assert gd.same_bits(got[~nan], ref[~nan])


@pytest.mark.parametrize("nx,ny", [(1201, 1161), (1960, 1400), (1961, 1441), (3501, 2521)])
def test_fp32_blocks_that_share_units(nx, ny):
    g0 = np.random.default_rng(nx * ny).standard_normal((ny, nx, 5)).astype(np.float32)
    assert gd.same_bits(_run(g0, np.float32, 2), _run(g0, np.float32, 2, pairs=0))
