"""The rules by which a call picks its kernels, asked of the built library
(without a GPU they assume 256 compute units)."""
import ctypes

import pytest

import mind_amd as M

MAX_DIM = (1 << 31) - 1


def _rule(mangled, *args):
    f = M.lib()[mangled]
    f.restype = ctypes.c_bool
    f.argtypes = [ctypes.c_bool if isinstance(a, bool) else ctypes.c_int for a in args]
    return f(*args)


def _i8_mid(m, k, n, panels=False):
    return _rule("_ZN3det6i8_midEiiib", m, n, k, panels)


@pytest.mark.parametrize("m,n", [(1, (1 << 30) + 77), (1, MAX_DIM), (64, MAX_DIM - 40), (65, 1 << 29),
                                 (1 << 20, 1 << 16)])
def test_mid_kernel_leaves_grids_a_launch_cannot_hold(m, n):
    # 64 x 64 tiles of 256 threads: 2^24 of them are 2^32 threads
    assert not _i8_mid(m, 8, n)


def test_mid_kernel_takes_the_largest_grid_a_launch_holds():
    assert _i8_mid(1, 8, ((1 << 24) - 8) * 64)
