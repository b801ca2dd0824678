"""Every route that a shape can take through the int8 and int16 GEMMs and the
batched Q16 GEMV (tests/routes.py), full outputs against the oracle: operands
at odd addresses, workspaces of exactly the size asked for and full of
garbage, poisoned outputs, nothing written past them."""
import sys

import numpy as np
import pytest

import mind_amd as M
import oracle as O
import routes as R

pytestmark = pytest.mark.gpu

POISON = np.int32(-1515870811)   # 0xA5 bytes


def note(msg):
    print(f"[gpu-case] {msg}", file=sys.stderr, flush=True)


def _at(a, off):
    buf = M.DeviceBuffer(a.nbytes + 64)
    M.check(M.lib().det_memcpy_htod(buf.ptr + off, a.ctypes.data, a.nbytes))
    return buf


def _gemm(op, a, b, m, k, n, offs, ws_bytes, route):
    L, s = M.lib(), M.Stream()
    want = np.empty(m * n, np.int32)
    cpu = O.lib().det_cpu_gemm_i8 if op == M.DET_OP_I8 else O.lib().det_cpu_gemm_i16
    assert cpu(a.ctypes.data, b.ctypes.data, want.ctypes.data, m, k, n) == 0
    da, db, dc = _at(a, offs[0]), _at(b, offs[1]), M.DeviceBuffer(m * n * 4 + 256)
    ws = M.DeviceBuffer(max(ws_bytes, 256))
    for rep in range(2):
        ws.fill(0x5B + rep), dc.fill(0xA5)
        note(f"op={op} {m}x{k}x{n} offsets={offs} ws={ws_bytes} {route} rep={rep}")
        M.check(L.det_matmul_ws_dev(op, da.ptr + offs[0], db.ptr + offs[1], dc.ptr, m, k, n,
                                    ws.ptr if ws_bytes else None, ws_bytes, s.ptr))
        s.sync()
        got = dc.to_array(np.int32, (m * n + 64,))
        np.testing.assert_array_equal(got[:m * n], want)
        assert (got[m * n:] == POISON).all()
    for buf in (da, db, dc, ws):
        buf.free()
    s.destroy()


@pytest.mark.parametrize("m,k,n,offs,ws,route", R.I8_ROUTES)
def test_gemm_i8_routes(m, k, n, offs, ws, route):
    assert R.i8(m, k, n, *offs, ws) == route
    a, b = O.gen_i8(0x2077 ^ (m * 1000003 + k * 1009 + n), m * k, k * n)
    a[:: max(1, a.size // 97)], b[:: max(1, b.size // 89)] = -128, -128
    need = R.i8_workspace(m, k, n, not any(offs)) if ws else 0
    assert need > 0 or not route.startswith("panels")
    _gemm(M.DET_OP_I8, a, b, m, k, n, offs, need, route)


@pytest.mark.parametrize("m,k,n,offs,route", R.I16_ROUTES)
def test_gemm_i16_routes(m, k, n, offs, route):
    assert R.i16(m, k, n, *offs) == route
    a, b = O.gen_i16(0x2077 ^ (m * 1000003 + k * 1009 + n), m * k, k * n)
    a[:: max(1, a.size // 97)], b[:: max(1, b.size // 89)] = -32768, -32768
    _gemm(M.DET_OP_I16, a, b, m, k, n, offs, M.lib().det_workspace_bytes(M.DET_OP_I16, m, k, n), route)


@pytest.mark.parametrize("fam", ["full", "extreme"])
@pytest.mark.parametrize("fill,k,nb", R.GEMV_MFMA)
def test_gemv_q16_mfma(fill, k, nb, fam):
    """Groups of 3 to 8 vectors on the MFMA kernel up to its largest K (32768):
    full-range W and x, or every limb of W and every digit of x at its extremes
    (x near 2^31 - 1 needs the fifth digit; the rows of one sign hold the
    largest sums).  A workspace of exactly the size asked for takes it; one
    byte less, or none, takes the VALU kernel: the same integers."""
    m = R.gemv_rows(fill)
    assert all(R.gemv_mfma(m, k, g) for g in {min(nb, 8), nb % 8 or 8})
    assert m % 64 and m * k * 4 < 1 << 31
    rng = np.random.default_rng(m + k * 31 + nb)
    ext = np.array([2147483647, -2147483648, -2147483647, 2139062144, 2139062143, 0, 1, -1, 65535, -65536,
                    -8421505, 8421504], np.int32)
    if fam == "full":
        draw = lambda size: rng.integers(-(1 << 31), 1 << 31, size).astype(np.int32)
    else:
        draw = lambda size: ext[rng.integers(0, len(ext), size)]
    # (a long random run, repeated: every row starts elsewhere in it)
    W, X = np.resize(draw((1 << 20) + 7), m * k), draw(nb * k)
    if fam == "extreme":   # sums of products of one sign: the accumulators' limits
        for r, v in ((0, -2147483648), (1, 2147483647), (m - 1, -2147483648), (m - 2, 2139062143)):
            W[r * k:(r + 1) * k] = v
        X[:k], X[k:2 * k] = 2147483647, -2147483648
        X[2 * k:3 * k] = 2139062144
    rows = np.unique(np.r_[0:5, 62:67, m - 70:m, rng.integers(0, m, 40)])
    want = O.gemv_q16_rows(W, X, m, k, nb, rows)
    L, s = M.lib(), M.Stream()
    need = L.det_gemv_workspace_bytes(m, k, nb)
    assert need > 0
    dW, dX, dY = M.DeviceBuffer.from_array(W), M.DeviceBuffer.from_array(X), M.DeviceBuffer(nb * m * 4)
    ws, first = M.DeviceBuffer(need), None
    for ws_ptr, ws_bytes in ((ws.ptr, need), (ws.ptr, need - 1), (None, 0)):
        note(f"gemv q16 {m}x{k} nb={nb} {fam} ws_bytes={ws_bytes}")
        ws.fill(0x3C), dY.fill(0xA5)
        M.check(L.det_gemv_q16_ws_dev(dW.ptr, dX.ptr, dY.ptr, m, k, nb, ws_ptr, ws_bytes, s.ptr))
        s.sync()
        got = dY.to_array(np.int32, (nb, m))
        np.testing.assert_array_equal(got[:, rows], want)
        first = got if first is None else first
        np.testing.assert_array_equal(got, first)
        # the vectors' operands are written there by the MFMA kernel's prep alone
        touched = bool((ws.to_array(np.uint8, (need,)) != 0x3C).any())
        assert touched == (ws_bytes == need)
    for buf in (dW, dX, dY, ws):
        buf.free()
    s.destroy()
