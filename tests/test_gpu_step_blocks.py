"""Single steps of each launch form (register blocks of every height, the march
in 64-column windows) with both y-edges: sizes at and one past a block's 60
columns and its rows, grids smaller than a wavefront's rows, values out of the
bounded division's range; FP64 bit for bit against the oracle (clamped edges) and
against the two sweeps one by one (ring edge), FP32 bit for bit against the march."""
import numpy as np
import pytest

import golden_data as gd
import le2d_amd
from oracle import Oracle

pytestmark = pytest.mark.gpu
ARGS = (0.2, (1.0, 0.9), (2.0, 1.0, 1.5))
SIZES = [(3, 3), (4, 5), (5, 6), (60, 4), (61, 5), (119, 121), (300, 256), (301, 257), (540, 600),
         (541, 601), (301, 1021), (600, 500), (601, 501), (3, 5000), (1300, 701), (1000, 1000),
         (2041, 2161)]


def _task(g0, dtype, soa):
    ny, nx = g0.shape[:2]
    t = le2d_amd.Task(nx, ny, *ARGS, le2d_amd.ST_SOA if soa else le2d_amd.ST_AOS, dtype=dtype)
    t.load(np.ascontiguousarray(np.moveaxis(g0, -1, 0)) if soa else g0)
    return t


def _step(g0, dtype, soa, march=False):
    with _task(g0, dtype, soa) as t:
        if march:
            t.set_tiles(xy_seg=11, xy_block=128)
        t.step_n(1)
        return t.grid().copy()


def _two_sweeps(g0, dtype, soa):
    with _task(g0, dtype, soa) as t:
        t.step_x()
        t.step_y()
        return t.grid().copy()


def _field(nx, ny, dtype):
    return np.random.default_rng(nx * ny).standard_normal((ny, nx, 5)).astype(dtype)


@pytest.mark.parametrize("nx,ny", SIZES)
def test_fp64_clamped_edges(nx, ny):
    g0 = _field(nx, ny, np.float64)
    ref = g0.copy()
    Oracle(np.float64).run(ref, *ARGS, 1)
    assert gd.same_bits(_step(g0, np.float64, False), ref)


@pytest.mark.parametrize("nx,ny", SIZES)
def test_fp64_ring_edge(nx, ny):
    g0 = _field(nx, ny, np.float64)
    assert gd.same_bits(_step(g0, np.float64, True), _two_sweeps(g0, np.float64, True))


@pytest.mark.parametrize("soa", [False, True])
@pytest.mark.parametrize("nx,ny", SIZES + [(4101, 4003)])
def test_fp32_equals_march(nx, ny, soa):
    g0 = _field(nx, ny, np.float32)
    assert gd.same_bits(_step(g0, np.float32, soa), _step(g0, np.float32, soa, march=True))


@pytest.mark.parametrize("nx,ny", [(130, 70), (1300, 701)])  # block and march
@pytest.mark.parametrize("value", [2.0**900, np.inf, np.nan, 1e-310])
def test_values_outside_the_bounds(value, nx, ny):
    g0 = _field(nx, ny, np.float64)
    g0[31, 57, 3] = value
    g0[10, 100:104, 0] = [0.0, -1e-6, -2e-6, 1e-6]
    ref = g0.copy()
    with np.errstate(all="ignore"):
        Oracle(np.float64).run(ref, *ARGS, 1)
    got = _step(g0, np.float64, False)
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan)
    assert gd.same_bits(got[~nan], ref[~nan])
