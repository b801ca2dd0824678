"""The rules by which a call picks its kernels, asked of the built library
(without a GPU they assume 256 compute units), and shapes that take each of
them: a change of a rule that moves such a shape to another route shows here
and not as a test that quietly covers less."""
import ctypes

import mind_amd as M

I8 = ("rows", "small", "mid", "on_grid", "panels_b", "panels", "bytes")
I16 = ("mid", "small", "interleaved", "limb")


def rule(mangled, *args, restype=ctypes.c_bool):
    f = M.lib()[mangled]
    f.restype = restype
    f.argtypes = [ctypes.c_bool if isinstance(a, bool) else ctypes.c_int for a in args]
    return f(*args)


def _route(mangled, m, k, n, a, b, *ws):
    f = M.lib()[mangled]
    f.restype = ctypes.c_int
    f.argtypes = [ctypes.c_void_p] * 2 + [ctypes.c_int] * 3 + [ctypes.c_bool] * len(ws)
    return f(a, b, m, n, k, *ws)


def i8(m, k, n, a=0, b=0, ws=True):
    """Operands at addresses a, b; ws: a workspace of the size such operands ask for."""
    return I8[_route("_ZN3det8i8_routeEPKaS1_iiib", m, k, n, a, b, ws)]


def i16(m, k, n, a=0, b=0):
    return I16[_route("_ZN3det9i16_routeEPKsS1_iii", m, k, n, a, b)]


def i8_workspace(m, k, n, aligned):
    return rule("_ZN3det18i8_workspace_bytesEiiib", m, n, k, aligned, restype=ctypes.c_size_t)


def i8_mid(m, k, n, panels=False, on_grid=False):
    return rule("_ZN3det6i8_midEiiibb", m, n, k, panels, on_grid)


def q16_direct(m, k, n):
    return rule("_ZN3det10q16_directEiii", m, n, k)


def gemv_mfma(m, k, nb):
    """Whether a group of nb vectors takes the MFMA kernel (given a workspace)."""
    return rule("_ZN3det10gemv8_paysEiii", m, k, nb)


def compute_units():
    return rule("_ZN3det8cu_countEv", restype=ctypes.c_int)


# (m, k, n, offsets of A and B in bytes, workspace given, route)
I8_ROUTES = [
    # both operands repacked: no size on the 16-byte grid; on it, misaligned; on
    # it, a grid that the edge kernel would underfill; fewer columns than a tile
    (2111, 650, 1999, (0, 0), True, "panels"), (2048, 768, 2064, (1, 3), True, "panels"),
    (2000, 2000, 2000, (0, 0), True, "panels"), (5000, 300, 50, (0, 0), True, "panels"),
    (4097, 1025, 1030, (8, 4), True, "panels"),
    # B alone: ragged, misaligned, underfilled
    (2048, 1024, 4100, (0, 0), True, "panels_b"), (2048, 768, 2064, (0, 4), True, "panels_b"),
    (2048, 1024, 2000, (0, 0), True, "panels_b"),
    # as they are, on the range-checked 256 x 256 tiles (K or M off 128)
    (3000, 1008, 3008, (0, 0), False, "on_grid"), (2000, 2000, 2000, (0, 0), False, "on_grid"),
    (2100, 1056, 4112, (0, 0), True, "on_grid"),
    # byte loads: off the grid, fewer than 64 columns, no workspace
    (5000, 300, 50, (0, 0), False, "bytes"), (4100, 1037, 63, (1, 3), False, "bytes"),
    (70000, 3, 17, (0, 0), False, "bytes"), (65, 5000, 33, (0, 0), False, "bytes"),
    # 64 x 64 tiles against one round of larger tiles: few steps and rounds; on
    # the grid; rows on the 4-byte grid; much padding; several rounds there
    (2001, 350, 2001, (0, 0), True, "mid"), (2001, 490, 2001, (0, 0), True, "panels"),
    (2304, 112, 2304, (0, 0), True, "mid"), (2304, 304, 2304, (0, 0), True, "on_grid"),
    (3008, 112, 3008, (0, 0), True, "on_grid"), (3008, 48, 3008, (0, 0), True, "mid"),
    (2000, 500, 2000, (0, 0), True, "mid"), (2000, 600, 2000, (0, 0), True, "panels"),
    (209, 431, 16001, (0, 0), True, "mid"), (3009, 250, 3009, (0, 0), True, "mid"),
    (3159, 521, 1376, (0, 0), True, "mid"), (2513, 367, 2513, (0, 0), True, "panels"),
    # (no K remainder; two rounds of tiles here)
    (2512, 384, 2512, (0, 0), True, "mid"), (1869, 1673, 676, (0, 0), True, "mid"),
    # and without a workspace: any size off the grid
    (2111, 650, 1999, (0, 0), False, "mid"), (2048, 768, 2064, (1, 3), False, "mid"),
]
# int16 as interleaved limbs: off the grid (by size, by address), on it, few rows
I16_ROUTES = [(2100, 1601, 1400, (0, 0), "interleaved"), (1000, 5000, 1200, (2, 2), "interleaved"),
              (700, 6000, 1000, (0, 0), "interleaved"), (64, 20000, 3000, (0, 2), "interleaved"),
              (2048, 640, 1664, (0, 0), "interleaved")]
# rows, K, vectors, whether each group takes the MFMA kernel: rows that fill
# just over 7/10 (9/10) of a round of 64-row blocks, the last block partly
GEMV_MFMA = [(0.7, 1024, 13), (0.7, 32768, 5), (0.7, 32768, 8), (0.9, 8704, 3), (0.9, 8704, 4), (0.9, 32768, 12)]


def gemv_rows(fill):
    return -int(-fill * compute_units() // 1) * 64 - 13
