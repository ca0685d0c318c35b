"""FP64 values out of the bounded division's range (2^300 and more, infinities,
NaN).  Where only some wavefronts of a tile meet one, in each block height and in
the marches, every finite result has the oracle's bits.  A field of them (a run
that has blown up) takes the IEEE divisions, which cost up to about a tenth, and
part of the bounded march; marching every tile twice in full would cost 1.8 to
1.9 times a finite field's pass."""
import numpy as np
import pytest

import golden_data as gd
import le2d_amd
from oracle import Oracle

pytestmark = pytest.mark.gpu
ARGS = (0.2, (1.0, 0.9), (2.0, 1.0, 1.5))
N = 2048


@pytest.mark.parametrize("value", [np.inf, 2.0**400])
@pytest.mark.parametrize("nx,ny,steps", [
    (90, 70, 2), (250, 300, 2), (512, 512, 2), (620, 600, 2), (724, 724, 2), (900, 900, 2),
    (130, 70, 1), (512, 512, 1), (900, 900, 1), (2400, 1930, 1)])
def test_some_rows(nx, ny, steps, value):
    g0 = np.random.default_rng(nx).standard_normal((ny, nx, 5))
    for k, j in enumerate(range(0, ny, 37)):  # other rows of a tile each time
        g0[j, (53 * k) % nx, k % 5] = value
    ref = g0.copy()
    with np.errstate(all="ignore"):
        Oracle(np.float64).run(ref, *ARGS, steps)
    with le2d_amd.Task(nx, ny, *ARGS) as t:
        t.load(g0)
        t.step_n(steps)
        got = t.grid().copy()
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan)
    assert gd.same_bits(got[~nan], ref[~nan])


@pytest.mark.parametrize("value", [np.nan, 2.0**400])
@pytest.mark.parametrize("what", ["time_pairs", "time_steps"])
def test_time_of_a_whole_field(what, value):
    ms = []
    for field in (np.random.default_rng(1).standard_normal((N, N, 5)), value):
        with le2d_amd.Task(N, N, *ARGS) as t:
            t.load(field)
            time = getattr(t, what)
            time(20)
            ms.append(min(time(20) for _ in range(9)))
    assert ms[1] < 1.4 * ms[0], ms
