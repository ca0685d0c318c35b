"""The separate sweeps at the edges of their forms: widths at and one past a
window's 60 columns, one and a few rows, heights around the y-sweep's group of 4
rows, and a grid on each side of the size that stays in the last-level cache;
FP64 bit for bit against the oracle with both y-edges, FP32 bit for bit against
other launch shapes."""
import numpy as np
import pytest

import golden_data as gd
import le2d_amd
from oracle import EDGE_CLAMP, EDGE_RING, Oracle

pytestmark = pytest.mark.gpu
ARGS = (0.2, (1.0, 0.9), (2.0, 1.0, 1.5))
SIZES = [(3, 3), (4, 4), (5, 5), (59, 6), (60, 7), (61, 8), (62, 9), (121, 3), (257, 13), (2050, 1701)]


def _task(g0, dtype):
    ny, nx = g0.shape[:2]
    t = le2d_amd.Task(nx, ny, *ARGS, dtype=dtype)
    t.load(g0)
    return t


@pytest.mark.parametrize("edge", [EDGE_CLAMP, EDGE_RING])
@pytest.mark.parametrize("nx,ny", SIZES)
def test_fp64_sweeps_match_oracle(nx, ny, edge):
    g0 = np.random.default_rng(nx * ny).standard_normal((ny, nx, 5))
    o = Oracle(np.float64)
    rx = g0.copy()
    o.sweep_x(rx, ARGS[0], ARGS[1][0], ARGS[2], soa=False)
    ry = rx.copy()
    o.sweep_y(ry, ARGS[0], ARGS[1][1], ARGS[2], edge=edge, soa=False)
    with _task(g0, np.float64) as t:
        t.step_x()
        assert gd.same_bits(t.grid(), rx)
        t.step_y() if edge == EDGE_CLAMP else t.step_y_cf(1)
        assert gd.same_bits(t.grid(), ry)


@pytest.mark.parametrize("shape", [(1, 1, 64), (3, 6, 128), (2, 1000, 256)])
@pytest.mark.parametrize("nx,ny", SIZES + [(2900, 2500)])
def test_fp32_shapes_agree(nx, ny, shape):
    g0 = np.random.default_rng(nx * ny).standard_normal((ny, nx, 5)).astype(np.float32)
    out = []
    for s in (None, shape):
        with _task(g0, np.float32) as t:
            if s:
                t.set_tiles(x_rows=s[0], y_seg=s[1], y_block=s[2])
            t.step_x()
            t.step_y()
            t.step_y_cf(1)
            out.append(t.grid().copy())
    assert gd.same_bits(*out)
