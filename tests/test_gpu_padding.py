"""The columns that pad a grid's rows are never initialised.  Whatever they hold
(zeros, NaN, infinities, 2^1000), FP64 passes give the oracle's bits, and a pass
over a grid of one 128-column strip, whose every tile reads a padding column,
takes the time that it takes with zeros there.  A tile marched a second time
would double it; 1.4 is midway."""
import ctypes

import numpy as np
import pytest

import golden_data as gd
import le2d_amd
from oracle import Oracle

pytestmark = pytest.mark.gpu
ARGS = (0.2, (1.0, 0.9), (2.0, 1.0, 1.5))
_hip = ctypes.CDLL("libamdhip64.so")
_hip.hipMemcpy2D.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p, ctypes.c_size_t,
                             ctypes.c_size_t, ctypes.c_size_t, ctypes.c_int]
_hip.hipMemcpy2D.restype = ctypes.c_int


def _fill(views, value):
    """Writes `value` into the padding of each state (field rows of `plane` values)."""
    for v in views:
        pad, rows, e = v.plane - v.nx, v.ny * v.pitch // v.plane, v.elem
        assert pad > 0 and v.pitch == 5 * v.plane and e == 8
        src = np.full((rows, pad), value)
        assert _hip.hipMemcpy2D(v.base + v.nx * e, v.plane * e, src.ctypes.data, pad * e, pad * e, rows,
                                1) == 0  # host to device


def _task(g0, seg, lanes):
    t = le2d_amd.Task(g0.shape[1], g0.shape[0], *ARGS)
    t.load(g0)
    t.set_step_pairs(seg)
    t.set_step_pair_window(lanes)
    return t


@pytest.mark.parametrize("value", [0.0, np.nan, -np.inf, 2.0**1000])
@pytest.mark.parametrize("nx,ny", [(3, 3), (119, 40), (121, 33), (241, 50), (301, 65)])
def test_values_do_not_matter(nx, ny, value):
    g0 = np.random.default_rng(nx * ny).standard_normal((ny, nx, 5))
    ref = g0.copy()
    Oracle(np.float64).run(ref, *ARGS, 4)
    with _task(g0, 16, 128) as t:
        current = t.device_view()
        t.step_n(2)
        t.wait()
        _fill((current, t.device_view()), value)  # both buffers
        t.step_n(2)
        assert gd.same_bits(t.grid(), ref)


def test_time_does_not_depend_on_them():
    nx, ny = 119, 30000
    g0 = np.random.default_rng(1).standard_normal((ny, nx, 5))
    with _task(g0, 37, 128) as t:  # 811 tiles, fewer than run at once
        buffers = [t.device_view()]
        t.time_pairs(1)
        buffers.append(t.device_view())
        ms = {}
        for value in (0.0, np.nan):
            _fill(buffers, value)
            t.time_pairs(20)
            ms[value] = min(t.time_pairs(20) for _ in range(9))
    assert ms[np.nan] < 1.4 * ms[0.0], ms
