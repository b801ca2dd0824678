"""The rules by which a call picks its kernels, asked of the built library
(without a GPU they assume 256 compute units)."""
import pytest

import routes as R

MAX_DIM = (1 << 31) - 1


@pytest.mark.parametrize("m,n", [(1, (1 << 30) + 77), (1, MAX_DIM), (64, MAX_DIM - 40), (65, 1 << 29),
                                 (1 << 20, 1 << 16)])
def test_mid_kernel_leaves_grids_a_launch_cannot_hold(m, n):
    # 64 x 64 tiles of 256 threads: 2^24 of them are 2^32 threads
    assert not R.i8_mid(m, 8, n)


def test_mid_kernel_takes_the_largest_grid_a_launch_holds():
    assert R.i8_mid(1, 8, ((1 << 24) - 8) * 64)


@pytest.mark.parametrize("m,k,n,offs,ws,route", R.I8_ROUTES)
def test_i8_route(m, k, n, offs, ws, route):
    assert R.i8(m, k, n, *offs, ws) == route


@pytest.mark.parametrize("m,k,n,offs,route", R.I16_ROUTES)
def test_i16_route(m, k, n, offs, route):
    assert R.i16(m, k, n, *offs) == route


@pytest.mark.parametrize("fill,k,nb", R.GEMV_MFMA)
def test_gemv_mfma_groups(fill, k, nb):
    m = R.gemv_rows(fill)
    assert all(R.gemv_mfma(m, k, g) for g in {min(nb, 8), nb % 8 or 8})
