"""Interface tiles of the two-step pass as blocks (k_step2_mat_block): sizes at
and one past a block's 56 columns and 8 rows, interfaces on every edge of a
block and of the grid, runs of single-material bands between them; FP64 bit for
bit against the oracle's node-local scheme, FP32 within the tier's bound of it
(relative L2 1e-5)."""
import numpy as np
import pytest

import golden_data as gd
import le2d_amd
from oracle import Oracle

pytestmark = pytest.mark.gpu
MATS = [(2.0, 1.0, 1.0), (2.6, 1.4, 2.2), (1.7, 0.8, 0.7)]


def _ids(kind, nx, ny):
    ids = np.zeros((ny, nx), np.uint8)
    if kind == "edges":
        ids[0], ids[-1] = 1, 2
        ids[:, 0], ids[:, -1] = 2, 1
    elif kind == "row":  # one node row in the middle of its bands
        ids[ny // 2] = 1
    elif kind == "column":
        ids[:, nx // 2] = 2
    elif kind == "dot":
        ids[ny // 3, nx // 3] = 1
    return ids


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["edges", "row", "column", "dot"])
@pytest.mark.parametrize("nx,ny,seg", [(3, 3, 2), (56, 8, 8), (57, 9, 9), (121, 17, 16),
                                       (249, 41, 24), (130, 200, 80)])
def test_blocks_match_oracle(nx, ny, seg, kind, dtype):
    rng = np.random.default_rng(nx + ny)
    g0 = rng.standard_normal((ny, nx, 5))
    ids = _ids(kind, nx, ny)
    dt, h = 0.25, (1.0, 0.9)
    ref = g0.astype(dtype).astype(np.float64)
    Oracle(np.float64).run_mat(ref, dt, h, MATS, ids, 6)
    for lanes in (64, 128, 256):
        with le2d_amd.Task(nx, ny, dt, h, MATS[0], dtype=dtype) as t:
            t.load(g0.astype(dtype))
            t.set_materials(MATS, ids)
            t.set_step_pairs(seg)
            t.set_step_pair_window(lanes)
            t.step_n(6)
            got = t.grid().copy()
        if dtype == np.float64:
            assert gd.same_bits(got, ref), lanes
        else:
            assert np.linalg.norm(got - ref) < 1e-5 * np.linalg.norm(ref), lanes
