"""Launches of direct convolutions planned on the host (tests/cpp/test_direct_plan.cpp):
what the entry point accepts, it launches."""
import subprocess

import pytest

from host_cpp import program

F32, F64, C128, I32 = 0, 1, 3, 6   # ndconv.h


@pytest.fixture(scope="module")
def exe():
    return program("test_direct_plan")


def launches(exe, dtype, *axes):
    """(LDS bytes, grid, block, form) of each launch; axes are (n, k, dilation, stride)."""
    r = subprocess.run([exe, str(dtype)] + [str(v) for a in axes for v in a], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
    rows = [line.split()[1:] for line in r.stdout.splitlines() if line.startswith("launch")]
    return [tuple(int(v) for v in row[:3]) + (row[3],) for row in rows]


@pytest.mark.parametrize("dtype", [F32, F64, I32])
@pytest.mark.parametrize("axes", [[(100, 3, 0, 1)], [(100, 3, 1, 1), (100, 3, 0, 1)], [(100, 3, 0, 1), (100, 3, 1, 1)],
                                  [(5, 2, 0, 1), (40, 3, 1, 1), (50, 3, 1, 1)],
                                  # dilations of a single tap, past every offset the kernels form
                                  [(100, 1, 1 << 16, 1), (100, 3, 1, 1)], [(100, 1, 1 << 31, 1)],
                                  [(100, 1, 1 << 50, 1), (100, 3, 1, 1)], [(100, 1, 1 << 49, 1)]])
def test_any_dilation_is_planned(exe, dtype, axes):
    """conv takes dilation 0 (every tap meets the same sample) and any dilation of one tap."""
    assert len(launches(exe, dtype, *axes)) == 1


@pytest.mark.parametrize("dtype,axes", [(C128, [(20, 3, 1, 1), (700, 3, 1, 10)]), (F32, [(1024, 3, 1, 1), (20480, 3, 1, 20)]),
                                        (F64, [(1026, 3, 1, 1), (20480, 3, 1, 10)]), (C128, [(700, 3, 1, 1), (700, 1, 1, 10)])])
def test_strides_up_to_the_lds_limit(exe, dtype, axes):
    """Regions that fill LDS but for a few hundred bytes leave no room for the offset tables."""
    (smem, _, _, _), = launches(exe, dtype, *axes)
    assert 155 * 1024 < smem <= 159 * 1024


@pytest.mark.parametrize("dtype", [F32, I32])
@pytest.mark.parametrize("shape,taps,dil,matrix", [
    ((62500, 256), (9, 1), 3, False), ((250000, 64), (3, 3), 3, False), ((666666, 24), (1, 7), 3, False),   # d phases, few taps
    ((333333, 12), (3, 3), 1, False),                                                                         # a narrow tile
    ((4000, 4000), (3, 3), 1, True), ((4000, 4000), (31, 31), 1, True), ((4000, 4000), (31, 31), 3, True),
    ((300, 300), (5, 5), 1, True), ((60, 300), (9, 9), 2, True)])                                            # few workgroups
def test_matrix_form_where_its_tiles_are_filled(exe, dtype, shape, taps, dil, matrix):
    (_, _, _, form), = launches(exe, dtype, *[(n, k, dil, 1) for n, k in zip(shape, taps)])
    assert form == ("matrix" if matrix else "vector")
