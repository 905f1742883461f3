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
    """(LDS bytes, grid, block) of each launch; axes are (n, k, dilation, stride)."""
    r = subprocess.run([exe, str(dtype)] + [str(v) for a in axes for v in a], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
    return [tuple(int(v) for v in line.split()[1:]) for line in r.stdout.splitlines() if line.startswith("launch")]


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
    (smem, _, _), = launches(exe, dtype, *axes)
    assert 155 * 1024 < smem <= 159 * 1024
