"""A launch shape that was read and is set again, on the same task or on another of
its grid, runs in the form it ran in: register blocks or a march, as the default
or the tuner chose.  The forms expected of each grid assume 256 compute units."""
import numpy as np
import pytest

import golden_data as gd
import le2d_amd

pytestmark = pytest.mark.gpu
ARGS = (0.2, (1.0, 0.9), (2.0, 1.0, 1.5))
F8, F4 = np.float64, np.float32
# grid -> rows of the default two-step blocks (0: a march)
PAIRS = {(F8, 96, 80): 4, (F8, 250, 300): 8, (F8, 400, 500): 16, (F8, 512, 512): 24,
         (F8, 620, 640): 32, (F8, 724, 724): 40, (F8, 900, 900): 0, (F8, 2048, 1000): 0,
         (F4, 96, 80): 4, (F4, 250, 300): 8, (F4, 400, 500): 16, (F4, 512, 512): 24,
         (F4, 1031, 517): 40, (F4, 900, 900): 64, (F4, 1500, 1001): 40, (F4, 4200, 3000): 0}


def _task(dtype, nx, ny):
    return le2d_amd.Task(nx, ny, *ARGS, dtype=dtype)


def _pairs(t):
    return t.get_step_pairs(), t.get_step_pair_window(), t.get_step_blocks()[1]


@pytest.mark.parametrize("dtype,nx,ny", PAIRS)
def test_default_pair_shape(dtype, nx, ny):
    rows = PAIRS[dtype, nx, ny]
    with _task(dtype, nx, ny) as t:
        shape = _pairs(t)
        assert shape[2] == rows
        assert not rows or shape[:2] == (rows, 64)
        t.set_step_pairs(shape[0])
        t.set_step_pair_window(shape[1])
        assert _pairs(t) == shape


@pytest.mark.parametrize("dtype,nx,ny", [(F8, 512, 512), (F8, 900, 900), (F4, 1031, 517)])
def test_tuned_pair_shape(dtype, nx, ny):
    with _task(dtype, nx, ny) as t:
        assert t.tune_step_pairs() == t.get_step_pairs()
        shape = _pairs(t)
    with _task(dtype, nx, ny) as t:
        t.set_step_pair_window(shape[1])
        t.set_step_pairs(shape[0])
        assert _pairs(t) == shape


@pytest.mark.parametrize("dtype,heights", [(F8, (4, 8, 16, 24, 32, 40)), (F4, (4, 8, 16, 24, 40, 64))])
def test_heights_name_blocks(dtype, heights):
    """Every block height set by hand, a march one row higher and one in another window."""
    g0 = np.random.default_rng(4).standard_normal((150, 313, 5)).astype(dtype)
    out = []
    for seg, window, rows in [(h, 64, h) for h in heights] + [(17, 64, 0), (16, 128, 0)]:
        with _task(dtype, 313, 150) as t:
            t.load(g0)
            t.set_step_pairs(seg)
            t.set_step_pair_window(window)
            assert _pairs(t) == (seg, window, rows)
            t.step_n(4)
            out.append(t.grid().copy())
    assert all(gd.same_bits(g, out[0]) for g in out[1:])


@pytest.mark.parametrize("dtype,nx,ny,rows", [
    (F8, 96, 80, 4), (F8, 300, 250, 12), (F8, 512, 512, 20), (F8, 900, 900, 0), (F8, 2400, 1930, 24),
    (F4, 512, 512, 20), (F4, 1500, 1001, 20), (F4, 8192, 2049, 44)])
def test_tiles(dtype, nx, ny, rows):
    with _task(dtype, nx, ny) as t:
        tiles = t.get_tiles()
        assert t.get_step_blocks()[0] == rows
        t.set_tiles(xy_seg=tiles[3] + 1)
        assert t.get_step_blocks()[0] == 0
        t.set_tiles(*tiles)
        assert t.get_tiles() == tiles and t.get_step_blocks()[0] == rows


def test_x_sweep_form():
    """The default rows keep the wavefront form (FP64 512^2: 8.3 us a sweep, 12.6 in
    whole workgroups; 1.25 is midway)."""
    with _task(F8, 512, 512) as t:
        t.time_sweeps(50)
        before = min(t.time_sweeps(20)[0] for _ in range(9))
        t.set_tiles(*t.get_tiles())
        after = min(t.time_sweeps(20)[0] for _ in range(9))
    assert after < 1.25 * before


def _batch(dtype, sizes):
    b = le2d_amd.Batch(dtype)
    for nx, ny in sizes:
        b.add(nx, ny, *ARGS)
    b.commit()
    return b


@pytest.mark.parametrize("dtype,rows,sizes", [
    (F8, 8, [(200, 170), (113, 121), (57, 9)]), (F8, 24, [(500, 400), (301, 241)]),
    (F4, 40, [(640, 512), (57, 41)]), (F8, 0, [(900, 700), (57, 41)])])
def test_batch_shape(dtype, rows, sizes):
    with _batch(dtype, sizes) as b:
        shape, form = b.get_shape(), b.form()
        assert b.get_blocks() == rows
        b.set_shape(128, 16, "tiles")
        assert b.get_blocks() == 0
        b.set_shape(shape[0], shape[1], form)
        assert b.get_shape() == shape and b.get_blocks() == rows
        b.set_shape(shape[0], shape[1])
        assert b.get_shape() == shape and b.get_blocks() == rows


@pytest.mark.parametrize("dtype", [F8, F4])
def test_tuned_blocks_stay_with_such_batches(dtype):
    """Three small grids tuned to blocks leave the default of three larger
    ones of the same count alone, with a total in the same class too."""
    small, large = [(200, 170), (113, 121), (57, 9)], [(500, 500), (500, 490), (490, 500)]
    thin = [(3, 5000), (3, 5000), (3, 5900)]  # as many nodes, three times the blocks
    want = []
    for sizes in (large, thin):
        with _batch(dtype, sizes) as b:
            want.append((b.get_shape(), b.get_blocks()))
    with _batch(dtype, small) as b:
        b.autotune(1)
        assert b.get_blocks() > 0
    for sizes, shape in zip((large, thin), want):
        with _batch(dtype, sizes) as b:
            assert (b.get_shape(), b.get_blocks()) == shape


def test_short_segments_of_fp32_sets():
    """FP32 sets that one round of 64-column workgroups would hold take two or three
    of shorter segments, with the results of another shape."""
    rng = np.random.default_rng(16)
    sizes = [tuple(int(v) for v in np.exp(rng.uniform(np.log(96), np.log(500), 2)))
             for _ in range(16)]
    states = [np.random.default_rng(k).standard_normal((ny, nx, 5)).astype(F4)
              for k, (nx, ny) in enumerate(sizes)]
    out = []
    for march in (False, True):
        with _batch(F4, sizes) as b:
            if march:
                b.set_shape(128, 37)
            else:
                width, seg = b.get_shape()[:2]
                strips = sum(-(-nx // 56) * -(-ny // seg) for nx, ny in sizes)
                assert width == 64 and b.get_blocks() == 0 and 1024 < strips <= 3 * 1024
            for k, g in enumerate(states):
                b.load(k, g)
            b.step(9)
            b.wait()
            out.append([b.read(k) for k in range(len(sizes))])
    assert all(gd.same_bits(x, y) for x, y in zip(*out))


@pytest.mark.parametrize("dtype,nx,ny,kernels", [
    (F8, 96, 80, ("k_step2_block", "k_step_block")), (F8, 900, 900, ("k_step2_split", "k_step_xy")),
    (F8, 2048, 2048, ("k_step2_xy", "k_step_xy")), (F4, 1500, 1001, ("k_step2_block", "k_step_block"))])
def test_bench_names_the_kernels_that_run(dtype, nx, ny, kernels):
    import bench
    with _task(dtype, nx, ny) as t:
        assert bench.step_kernels(t) == kernels
