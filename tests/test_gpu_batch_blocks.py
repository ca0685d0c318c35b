"""Two-step batches whose default launch is in blocks, one set of sizes for each
block height (8, 16, 24 and the highest), among them single-block instances and
sizes one past a block's 56 columns and its rows, and one set past the limit; an
odd step count with graph replays.  FP64 bit for bit against the oracle, FP32 bit
for bit against a marched launch shape."""
import numpy as np
import pytest

import golden_data as gd
import le2d_amd
from oracle import Oracle

pytestmark = pytest.mark.gpu
ARGS = (0.2, (1.0, 0.9), (2.0, 1.0, 1.5))
# 256 compute units: the set's blocks of the height below fill at most one each
SETS = {8: [(3, 3), (57, 9), (56, 8), (200, 170), (113, 121)],
        16: [(57, 17), (400, 300), (300, 257)],
        24: [(57, 25), (3, 24), (500, 400), (301, 241)],
        40: [(640, 512), (57, 41)],
        0: [(900, 700), (57, 41), (3, 3)]}


def _states(sizes, dtype):
    return [np.random.default_rng(k).standard_normal((ny, nx, 5)).astype(dtype)
            for k, (nx, ny) in enumerate(sizes)]


def _run(states, dtype, steps, march=False):
    b = le2d_amd.Batch(dtype)
    for g in states:
        b.add(g.shape[1], g.shape[0], *ARGS)
    b.commit()
    with b:
        if march:
            b.set_shape(128, 7)
        for k, g in enumerate(states):
            b.load(k, g)
        b.step(steps)
        b.wait()
        return [b.read(k) for k in range(len(states))]


@pytest.mark.parametrize("rows", SETS)
def test_fp64_matches_oracle(rows):
    states = _states(SETS[rows], np.float64)
    for g, got in zip(states, _run(states, np.float64, 9)):
        ref = g.copy()
        Oracle(np.float64).run(ref, *ARGS, 9)
        assert gd.same_bits(got, ref), got.shape


@pytest.mark.parametrize("rows", SETS)
def test_fp32_equals_march(rows):
    states = _states(SETS[rows], np.float32)
    for got, ref in zip(_run(states, np.float32, 9), _run(states, np.float32, 9, march=True)):
        assert gd.same_bits(got, ref), got.shape
