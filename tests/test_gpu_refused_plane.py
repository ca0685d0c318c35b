"""A material plane that is refused (an id past the table, a material constant of
zero, no device memory) leaves the task as it was: its launch shape, the plane
that was in force, and its results."""
import ctypes

import numpy as np
import pytest

import golden_data as gd
import le2d_amd
from oracle import Oracle

pytestmark = pytest.mark.gpu
MATS = [(2.0, 1.0, 1.0), (2.6, 1.4, 2.2)]
NX, NY = 130, 97
ARGS = (0.25, (1.0, 0.9), MATS[0])


def _ids(column):
    ids = np.zeros((NY, NX), np.uint8)
    ids[:, column:] = 1
    return ids


def _state():
    return np.random.default_rng(3).standard_normal((NY, NX, 5))


@pytest.mark.parametrize("mats,ids", [(MATS[:1], _ids(60)), ([(2.0, 0.0, 1.0)], None)])
def test_bad_plane(mats, ids):
    ref = _state()
    Oracle(np.float64).run(ref, *ARGS, 6)
    with le2d_amd.Task(NX, NY, *ARGS) as t:
        t.load(_state())
        shape = t.get_step_pairs(), t.get_step_pair_window(), t.get_step_blocks()
        assert shape[2][1] > 0  # blocks
        with pytest.raises(le2d_amd.LE2DError):
            t.set_materials(mats, ids)
        assert (t.get_step_pairs(), t.get_step_pair_window(), t.get_step_blocks()) == shape
        t.step_n(6)
        assert gd.same_bits(t.grid(), ref)


@pytest.mark.parametrize("granted", range(4))  # id plane, two constant tables, energy table
def test_no_memory_for_a_second_plane(granted):
    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    hip.hipFree.argtypes = [ctypes.c_void_p]
    left = [None]

    def alloc(ptr, nbytes, ctx):
        if left[0] is not None:
            if left[0] == 0:
                return 1
            left[0] -= 1
        return hip.hipMalloc(ptr, nbytes)

    fns = le2d_amd.ALLOC_FN(alloc), le2d_amd.FREE_FN(lambda p, ctx: hip.hipFree(p) and None)
    ref = _state()
    Oracle(np.float64).run_mat(ref, ARGS[0], ARGS[1], MATS, _ids(60), 6)
    le2d_amd.set_device_allocator(*fns)
    try:
        with le2d_amd.Task(NX, NY, *ARGS) as t:
            t.load(_state())
            t.set_materials(MATS, _ids(60))
            t.step_n(4)
            left[0] = granted
            with pytest.raises(le2d_amd.LE2DError):
                t.set_materials(MATS, _ids(20))
            left[0] = None
            t.step_n(2)
            got = t.grid().copy()
    finally:
        le2d_amd.set_device_allocator(None, None)
    assert gd.same_bits(got, ref)


@pytest.mark.parametrize("count", [8, 9])
def test_plane_set_after_the_tuner_ran_and_taken_away(count):
    """What the tuner found without a plane is not the plane's shape: it has the
    default of grids with one, and the tuned shape is back when the plane goes."""
    ref = _state()
    o = Oracle(np.float64)
    o.run(ref, *ARGS, count)
    o.run_mat(ref, ARGS[0], ARGS[1], MATS, _ids(60), count)
    o.run(ref, *ARGS, count)
    with le2d_amd.Task(NX, NY, *ARGS) as t:
        t.set_materials(MATS, _ids(60))
        default = t.get_step_pairs(), t.get_step_pair_window()
    with le2d_amd.Task(NX, NY, *ARGS) as t:
        t.load(_state())
        t.step_n(count)
        shape = t.get_step_pairs(), t.get_step_pair_window(), t.get_step_blocks()
        assert shape[2][1] > 0  # blocks
        t.set_materials(MATS, _ids(60))
        assert (t.get_step_pairs(), t.get_step_pair_window()) == default
        t.step_n(count)
        t._check(t.lib.le2d_set_material_plane(t.ref, 0, None, None), "remove the plane")
        assert (t.get_step_pairs(), t.get_step_pair_window(), t.get_step_blocks()) == shape
        t.step_n(count)
        assert gd.same_bits(t.grid(), ref)
