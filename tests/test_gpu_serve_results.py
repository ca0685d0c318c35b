"""Results of the serving loop at the edges of their copy's pieces: below, at and one
value past the bytes a thread, a piece and a stage take (256 KB, 1 MB, 8 MB), and more
concurrent callers than there are stages; every byte as the oracle's."""
import threading

import numpy as np
import pytest

import golden_data as gd
import le2d_amd
from oracle import Oracle

pytestmark = pytest.mark.gpu
ARGS = (0.2, (1.0, 1.0), (2.0, 1.0, 1.5))
# nodes of 40 bytes; 26214 x 40 is 16 bytes short of 1 MB
SIZES = [(3, 3), (64, 103), (127, 103), (3, 8738), (5, 5243), (3, 69905), (401, 523), (601, 701)]


def _ref(nx, ny):
    g = np.zeros((ny, nx, 5))
    with le2d_amd.Task(nx, ny, *ARGS) as t:
        t.set_ball((nx / 2, ny / 2), 5.0, 1.0)
        g = t.grid().copy()
    Oracle(np.float64).run(g, *ARGS, 2)
    return g


def _submit(s, nx, ny):
    return s.submit(nx, ny, 2, np.float64, *ARGS, disk=(nx / 2, ny / 2, 5.0, 1.0), keep=True)


@pytest.mark.parametrize("nx,ny", SIZES)
def test_sizes(nx, ny):
    with le2d_amd.Server(1 << 30, 8) as s:
        i = _submit(s, nx, ny)
        s.drain(60)
        assert gd.same_bits(s.result(i), _ref(nx, ny))


def test_more_callers_than_stages():
    with le2d_amd.Server(1 << 30, 32) as s:
        ids = [_submit(s, *SIZES[-1 - k % 2]) for k in range(12)]
        s.drain(60)
        out = {}
        th = [threading.Thread(target=lambda i=i: out.update({i: s.result(i)})) for i in ids]
        for t in th:
            t.start()
        for t in th:
            t.join()
        for k, i in enumerate(ids):
            assert gd.same_bits(out[i], _ref(*SIZES[-1 - k % 2]))
