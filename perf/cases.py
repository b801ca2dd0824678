"""What this library's users run, as measurable cases.

A case is one call of a public entry point with its sizes.  ``listed()`` gives
one case for each way the library is used, ``draw(rng)`` further cases of the
same ranges: round and odd sizes, the smallest calls, where a launch is most
of the time, and the largest, where memory or the matrix cores are.  Every
output is exact by contract (integer arithmetic, and a fixed schedule for
f32), so every tolerance is "exact".

Device cases pass tensors of the current torch stream to the ``*_dev`` entry
points, with the workspace a serving program keeps; host cases pass numpy
arrays to the synchronous host-pointer calls.
"""
import math

import numpy as np
import torch

import mind_amd as M

F32_OPS = {"dot": M.DET_F32_DOT, "l1": M.DET_F32_L1, "linf": M.DET_F32_LINF}
GEMM_OPS = {"i8": M.DET_OP_I8, "i16": M.DET_OP_I16, "q16": M.DET_OP_Q16}
ELEM_BYTES = {"i8": 1, "i16": 2, "q16": 4}


def listed():
    return [
        # int8 layer over a full batch of tokens: the headline shape, the largest product
        dict(name="i8_square", kind="gemm", op="i8", m=4096, k=4096, n=4096),
        # the same MLP layer at decode: a few token rows against the whole weight matrix
        dict(name="i8_few_rows", kind="gemm", op="i8", m=16, k=4096, n=11008),
        # int8 operands with no size on the 16-byte grid
        dict(name="i8_ragged", kind="gemm", op="i8", m=2047, k=2047, n=2047),
        # int16 product of ordinary size, not a multiple of any tile
        dict(name="i16_gemm", kind="gemm", op="i16", m=1500, k=1500, n=1500),
        # Q16.16 product of the reference bench's layer size
        dict(name="q16_gemm", kind="gemm", op="q16", m=1024, k=1024, n=1024),
        # one query scored against the routing catalog
        dict(name="gemv_catalog", kind="gemv_q16", m=11922, k=384, nb=1),
        # a large Q16.16 matrix applied to a batch of eight vectors: the largest read
        dict(name="gemv_batch", kind="gemv_q16", m=16384, k=16384, nb=8),
        # int16 matrix-vector product whose rows are not whole 16-byte vectors
        dict(name="gemv_i16", kind="gemv_i16", m=8192, k=8190),
        # strict f32 distances of one query to many rows
        dict(name="rows_f32", kind="rows_f32", metric="l1", rows=65536, cols=1024),
        # many short transforms: frames of 256 samples
        dict(name="fft_frames", kind="fft", logn=8, batch=65536, wide=False),
        # long transforms
        dict(name="fft_long", kind="fft", logn=16, batch=16, wide=False),
        # the smallest calls, as the reference makes them: one small product from host memory
        dict(name="host_small", kind="host", op="q16", m=64, k=64, n=64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, grid):
    """A size in [lo, hi], spread over its logarithm; half of them on a grid."""
    v = _log_int(rng, lo, hi)
    if rng.random() < 0.5:
        v = max(grid, v // grid * grid)
    return min(max(v, lo), hi)


def draw(rng):
    what = rng.choice(["i8", "i8_few_rows", "i16", "q16", "gemv_q16", "gemv_batch", "gemv_i16", "rows_f32",
                       "fft_frames", "fft_long", "host"])
    if what == "i8":
        return dict(kind="gemm", op="i8", m=_size(rng, 256, 4096, 128), k=_size(rng, 256, 4096, 128),
                    n=_size(rng, 256, 4096, 128))
    if what == "i8_few_rows":
        return dict(kind="gemm", op="i8", m=_log_int(rng, 1, 64), k=_size(rng, 1024, 8192, 256),
                    n=_size(rng, 1024, 16384, 256))
    if what == "i16":
        return dict(kind="gemm", op="i16", m=_size(rng, 64, 2048, 64), k=_size(rng, 128, 2048, 64),
                    n=_size(rng, 128, 2048, 64))
    if what == "q16":
        return dict(kind="gemm", op="q16", m=_size(rng, 16, 1024, 64), k=_size(rng, 128, 1024, 64),
                    n=_size(rng, 128, 1024, 64))
    if what == "gemv_q16":
        return dict(kind="gemv_q16", m=_size(rng, 256, 16384, 64), k=_size(rng, 64, 16384, 64), nb=1)
    if what == "gemv_batch":
        return dict(kind="gemv_q16", m=_size(rng, 256, 16384, 64), k=_size(rng, 64, 8192, 64),
                    nb=_log_int(rng, 2, 16))
    if what == "gemv_i16":
        return dict(kind="gemv_i16", m=_size(rng, 256, 16384, 64), k=_size(rng, 64, 16384, 64))
    if what == "rows_f32":
        return dict(kind="rows_f32", metric=rng.choice(["dot", "l1", "linf"]), rows=_size(rng, 1024, 65536, 64),
                    cols=_size(rng, 64, 2048, 64))
    if what == "fft_frames":
        logn = rng.randint(6, 11)
        return dict(kind="fft", logn=logn, batch=_log_int(rng, 16, (1 << 24) >> logn), wide=rng.random() < 0.25)
    if what == "fft_long":
        logn = rng.randint(12, 18)
        return dict(kind="fft", logn=logn, batch=_log_int(rng, 1, (1 << 21) >> logn), wide=rng.random() < 0.25)
    op = rng.choice(["i8", "q16", "gemv", "dot"])
    if op in ("i8", "q16"):
        return dict(kind="host", op=op, m=_log_int(rng, 16, 256), k=_log_int(rng, 16, 256), n=_log_int(rng, 16, 256))
    if op == "gemv":
        return dict(kind="host", op=op, m=_log_int(rng, 64, 512), k=_log_int(rng, 64, 512), n=1)
    return dict(kind="host", op=op, m=1, k=_log_int(rng, 256, 65536), n=1)


# ------------------------------------------------------------------ inputs

def _randint(g, lo, hi, shape, dtype):
    return torch.randint(lo, hi, shape, generator=g, dtype=dtype, device="cuda")


def _gemm_operand(g, op, shape):
    if op == "i8":
        return _randint(g, -128, 128, shape, torch.int8)
    if op == "i16":
        return _randint(g, -32768, 32768, shape, torch.int16)
    # Q16.16 reals in [-4, 4), one in a hundred at the type's limits
    x = _randint(g, -(4 << 16), 4 << 16, shape, torch.int32)
    top = torch.where(_randint(g, 0, 2, shape, torch.int8) == 0, 2**31 - 1, 1 - 2**31).to(torch.int32)
    return torch.where(_randint(g, 0, 100, shape, torch.int8) == 0, top, x)


def _workspace(nbytes):
    return torch.empty(max(int(M.check(nbytes)), 1), dtype=torch.uint8, device="cuda")


def prepare(case, seed):
    L, kind = M.lib(), case["kind"]
    if kind == "host":
        r = np.random.default_rng(seed)
        m, k, n = case["m"], case["k"], case["n"]
        if case["op"] == "i8":
            return dict(case=case, a=r.integers(-128, 128, (m, k), np.int8), b=r.integers(-128, 128, (k, n), np.int8))
        lim = 4 << 16
        a = r.integers(-lim, lim, (m, k), np.int32)
        return dict(case=case, a=a[0] if case["op"] == "dot" else a,
                    b=r.integers(-lim, lim, (k, n), np.int32) if case["op"] == "q16"
                    else r.integers(-lim, lim, k, np.int32))
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    s = dict(case=case)
    if kind == "gemm":
        op, m, k, n = case["op"], case["m"], case["k"], case["n"]
        s["a"], s["b"] = _gemm_operand(g, op, (m, k)), _gemm_operand(g, op, (k, n))
        s["c"] = torch.empty((m, n), dtype=torch.int32, device="cuda")
        s["ws"] = _workspace(L.det_workspace_bytes(GEMM_OPS[op], m, k, n))
    elif kind in ("gemv_q16", "gemv_i16"):
        m, k, nb = case["m"], case["k"], case.get("nb", 1)
        q = kind == "gemv_q16"
        lim, dtype = (1 << 16, torch.int32) if q else (1 << 15, torch.int16)
        s["w"], s["x"] = _randint(g, -lim, lim, (m, k), dtype), _randint(g, -lim, lim, (nb, k), dtype)
        s["y"] = torch.empty((nb, m), dtype=torch.int32, device="cuda")
        if q:
            s["ws"] = _workspace(L.det_gemv_workspace_bytes(m, k, nb))
    elif kind == "rows_f32":
        rows, cols = case["rows"], case["cols"]
        s["w"] = torch.rand((rows, cols), generator=g, device="cuda") * 2 - 1
        s["x"] = torch.rand(cols, generator=g, device="cuda") * 2 - 1
        s["y"] = torch.empty(rows, device="cuda")
    else:
        n, batch = 1 << case["logn"], case["batch"]
        lim = 1 << (40 if case["wide"] else 16)
        s["re"], s["im"] = (_randint(g, -lim, lim, (batch, n), torch.int64) for _ in range(2))
        s["ore"], s["oim"] = torch.empty_like(s["re"]), torch.empty_like(s["im"])
        s["tw"] = torch.from_numpy(M.fft_twiddles(n)).cuda()
    return s


# ------------------------------------------------------------------ one pass

def run(s):
    case, L = s["case"], M.lib()
    kind = case["kind"]
    if kind == "host":
        if case["op"] == "i8":
            return M.det_matmul_i8(s["a"], s["b"])
        if case["op"] == "q16":
            return M.det_matmul_q16(s["a"], s["b"])
        return M.det_gemv_q16(s["a"], s["b"]) if case["op"] == "gemv" else M.dot_q16(s["a"], s["b"])
    st = torch.cuda.current_stream().cuda_stream
    if kind == "gemm":
        a, b, c, ws = s["a"], s["b"], s["c"], s["ws"]
        M.check(L.det_matmul_ws_dev(GEMM_OPS[case["op"]], a.data_ptr(), b.data_ptr(), c.data_ptr(), case["m"],
                                    case["k"], case["n"], ws.data_ptr(), ws.numel(), st))
        return c
    if kind == "gemv_q16":
        w, x, y, ws = s["w"], s["x"], s["y"], s["ws"]
        M.check(L.det_gemv_q16_ws_dev(w.data_ptr(), x.data_ptr(), y.data_ptr(), case["m"], case["k"], case["nb"],
                                      ws.data_ptr(), ws.numel(), st))
        return y
    if kind == "gemv_i16":
        w, x, y = s["w"], s["x"], s["y"]
        M.check(L.det_gemv_i16_dev(w.data_ptr(), x.data_ptr(), y.data_ptr(), case["m"], case["k"], st))
        return y
    if kind == "rows_f32":
        w, x, y = s["w"], s["x"], s["y"]
        M.check(L.det_rows_metric_f32_dev(F32_OPS[case["metric"]], w.data_ptr(), x.data_ptr(), y.data_ptr(),
                                          case["rows"], case["cols"], st))
        return y
    re, im, ore, oim, tw = s["re"], s["im"], s["ore"], s["oim"], s["tw"]
    M.check(L.det_fft_q16_oop_dev(re.data_ptr(), im.data_ptr(), ore.data_ptr(), oim.data_ptr(), tw.data_ptr(),
                                  case["logn"], 1 << case["logn"], case["batch"], st))
    return ore, oim


# ------------------------------------------------------------------ what it cannot do without

def work(case):
    kind = case["kind"]
    if kind == "fft":
        pts = case["batch"] << case["logn"]
        return dict(bytes=32 * pts + (8 << case["logn"]), flops=5 * pts * case["logn"])
    if kind == "rows_f32":
        r, c = case["rows"], case["cols"]
        return dict(bytes=4 * (r * c + c + r), flops=2 * r * c)
    if kind in ("gemv_q16", "gemv_i16"):
        m, k, nb, e = case["m"], case["k"], case.get("nb", 1), 4 if kind == "gemv_q16" else 2
        return dict(bytes=e * (m * k + nb * k) + 4 * nb * m, flops=2 * m * k * nb)
    m, k, n = case["m"], case["k"], case["n"]
    e = ELEM_BYTES.get(case["op"], 4)
    return dict(bytes=e * (m * k + k * n) + 4 * m * n, flops=2 * m * k * n)


def tolerance(case):
    return "exact"


# ------------------------------------------------------------------ the same results in plain 64-bit arithmetic

def _wrap32(x):
    return (((x + 2**31) & (2**32 - 1)) - 2**31).to(torch.int32)


def _exact_product(a, b):
    """Integer product whose float64 sums are exact (below 2^53)."""
    return _wrap32((a.double() @ b.double()).to(torch.int64))


def _q16_product(a, b):
    """sum_k floor(a[i, k] * b[k, j] / 2^16), a slice of rows at a time."""
    bt = b.to(torch.int64).T.contiguous()
    step = max(1, (1 << 27) // max(1, bt.numel()))
    rows = [((a[i:i + step, None, :].to(torch.int64) * bt[None]) >> 16).sum(-1) for i in range(0, a.shape[0], step)]
    return _wrap32(torch.cat(rows))


def _fft(re, im, tw, logn):
    n = 1 << logn
    pos = torch.arange(n, device=re.device)
    rev = torch.zeros_like(pos)
    for b in range(logn):
        rev |= ((pos >> b) & 1) << (logn - 1 - b)
    re, im = re[:, rev], im[:, rev]
    for b in range(logn):
        h = 1 << b
        r, i = re.reshape(-1, n // (2 * h), 2, h), im.reshape(-1, n // (2 * h), 2, h)
        ar, br, ai, bi = r[:, :, 0], r[:, :, 1], i[:, :, 0], i[:, :, 1]
        if b:
            k = torch.arange(h, device=re.device) << (logn - 1 - b)
            wr, wi = tw[2 * k], tw[2 * k + 1]
            br, bi = ((wr * br) >> 16) - ((wi * bi) >> 16), ((wr * bi) >> 16) + ((wi * br) >> 16)
        re = torch.stack((ar + br, ar - br), 2).reshape(-1, n)
        im = torch.stack((ai + bi, ai - bi), 2).reshape(-1, n)
    return re, im


def exact(case, seed):
    s, kind = prepare(case, seed), case["kind"]
    if kind == "host":
        a, b = s["a"].astype(np.int64), s["b"].astype(np.int64)
        if case["op"] == "i8":
            return (a @ b).astype(np.int32)
        if case["op"] == "dot":
            return int(np.int64(((a * b) >> 16).sum()).astype(np.int32))
        if case["op"] == "gemv":
            return ((a * b) >> 16).sum(-1).astype(np.int32)
        return ((a[:, :, None] * b[None]) >> 16).sum(1).astype(np.int32)
    if kind == "gemm":
        return (_q16_product if case["op"] == "q16" else _exact_product)(s["a"], s["b"])
    if kind == "gemv_q16":
        return _q16_product(s["x"], s["w"].T)
    if kind == "gemv_i16":
        return _exact_product(s["x"], s["w"].T)
    if kind == "rows_f32":
        w, x = s["w"].double(), s["x"].double()
        if case["metric"] == "dot":
            return w @ x
        d = (w - x).abs()
        return d.sum(-1) if case["metric"] == "l1" else d.amax(-1)
    return _fft(s["re"], s["im"], s["tw"], case["logn"])
