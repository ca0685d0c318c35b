"""Registers and occupancy of the register blocks and of the kernels that share
their sweeps, from the compiler's resource report (see test_kernel_resources).

A block holds its rows in registers for a whole pass: nothing may spill, and its
wavefronts must all be resident, WV / 4 for each SIMD, twice that where the
launch rules count on two blocks a compute unit."""
import pytest

from test_kernel_resources import _kernels, table  # noqa: F401 (fixture)


@pytest.mark.parametrize("prefix", ["k_step2_block", "k_step_block", "k_step_batch_blocks",
                                    "k_step2_mat_block", "k_sweep_x_row"])
def test_no_spills(table, prefix):  # noqa: F811
    for name, r in _kernels(table, prefix).items():
        assert r["spill"] == 0 and r["scratch"] == 0, (name, r)


def test_single_step_marches(table):  # noqa: F811
    """The 64-column march, the default's, keeps everything in registers; the wider
    ones and those with a material plane, held to three waves, spill at most two in
    FP64."""
    for prefix in ("k_step_xy", "k_step_mat_homog"):
        for name, r in _kernels(table, prefix).items():
            most = 0 if name.startswith("k_step_xy") and name.endswith("64>") else 2
            most = most if "double" in name else 0
            assert r["spill"] <= most and r["scratch"] <= 12, (name, r)
            assert r["waves"] >= 3, (name, r)


def _args(name):
    return [a.strip() for a in name[name.index("<") + 1:-1].split(",")]


@pytest.mark.parametrize("prefix", ["k_step2_block", "k_step_block", "k_step_batch_blocks"])
def test_blocks_are_resident(table, prefix):  # noqa: F811
    for name, r in _kernels(table, prefix).items():
        real, wavefronts = _args(name)[0], int(_args(name)[-1])
        rows = int(_args(name)[-2])
        need = (wavefronts + 3) // 4
        # FP32 blocks of 40 rows (two steps) and of 20 and 44 (one) share compute units, as do
        # the FP64 ones of 24 rows on four wavefronts
        if real == "float" and (rows, wavefronts) in ((4, 12), (3, 8)) or (rows, wavefronts) == (7, 4):
            need *= 2
        assert r["waves"] >= need, (name, r)
