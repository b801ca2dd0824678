"""Checks on the gfx950 assembly of every HIP source, compiled on the CPU with
the library's own device flags (hipcc cross-compiles; no GPU needed).

1. M0: the LDS-DMA helpers (dma16 / dma16s in mind_amd/csrc/det_common.h)
   set M0 in inline assembly.  The compiler treats M0 as a reserved register
   and ignores it in an asm clobber list (it warns so), so the helpers are
   safe only while the compiler itself keeps no value in M0 across them:
   every M0 access must be one of the helpers' three-instruction sequences
   (s_mov_b32 m0 / s_nop 0 / buffer_load_dwordx4 ... lds).
2. Scalar memory is only read: every scalar instruction is an arithmetic or
   control one, or a scalar load.  Stores go through the vector memory path
   only.
3. Sums that have to wrap are unsigned in the source: signed overflow is
   undefined and the build has no -fwrapv.

It is a CPU test: it never needs a GPU."""
import concurrent.futures as cf
import glob
import os
import re
import shutil
import subprocess

import pytest

import mind_amd.build as B

SRCS = sorted(glob.glob(os.path.join(B.CSRC, "*.hip")))

pytestmark = pytest.mark.skipif(not os.path.exists(B.HIPCC) and shutil.which("hipcc") is None,
                                reason="hipcc not installed")


def _asm(src, out_dir):
    out = os.path.join(out_dir, os.path.basename(src)[:-4] + ".s")
    r = subprocess.run([B.HIPCC, *B.DEVICE_FLAGS, "--cuda-device-only", "-S", src, "-o", out],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    return out


@pytest.fixture(scope="module")
def instructions(tmp_path_factory):
    """{file: [instruction lines]} (comments, labels and directives dropped)."""
    d = str(tmp_path_factory.mktemp("asm"))
    with cf.ThreadPoolExecutor(max_workers=8) as ex:
        outs = list(ex.map(lambda s: _asm(s, d), SRCS))
    res = {}
    for path in outs:
        ins = []
        for line in open(path):
            t = line.split(";")[0].strip()
            if t and not t.startswith(".") and not t.endswith(":"):
                ins.append(t)
        res[os.path.basename(path)] = ins
    return res


def test_m0_only_in_the_lds_dma_sequences(instructions):
    m0 = re.compile(r"\bm0\b")
    sequences = 0
    for name, ins in instructions.items():
        for i, t in enumerate(ins):
            if not m0.search(t):
                continue
            where = f"{name}: {t!r}"
            assert re.fullmatch(r"s_mov_b32 m0, s\d+", t), "M0 used outside the DMA helpers: " + where
            assert ins[i + 1] == "s_nop 0", where
            assert ins[i + 2].startswith("buffer_load_dwordx4") and ins[i + 2].endswith(" lds"), where
            sequences += 1
    assert sequences > 0   # the DMA kernels are in the build


# scalar instructions: arithmetic on registers, control, loads
SCALAR = re.compile(r"s_(\w+_[biu](32|64)|(addk|cmpk_\w+|mulk|movk)_[iu]32|nop|waitcnt|barrier|endpgm|branch|"
                    r"cbranch_\w+|setprio|sleep|(buffer_)?load_dword(x(2|4|8|16))?)")


def test_no_scalar_cache_writes(instructions):
    found = {t.split()[0] for ins in instructions.values() for t in ins
             if t.startswith("s_") and not SCALAR.fullmatch(t.split()[0])}
    assert not found, found
    assert sum(len(v) for v in instructions.values()) > 10000   # the kernels were really compiled


# file: (mangled) functions with 64-bit sums that may leave int64's range, or
# that compare any int64 with a bound
WRAPPING = {"det_gemv.hip": "_ZN3det4gemv3Q16",
            "det_fft.hip": r"_Z\w*(?:load_tw32|run_pass|butterfly|in_range)"}


@pytest.mark.parametrize("src", sorted(WRAPPING))
def test_wrapping_sums_are_unsigned(src, tmp_path):
    """In the unoptimised IR, where clang marks signed sums `nsw`."""
    out = str(tmp_path / "x.ll")
    r = subprocess.run([B.HIPCC, *B.DEVICE_FLAGS, "--cuda-device-only", "-S", "-emit-llvm", "-Xclang",
                        "-disable-llvm-passes", os.path.join(B.CSRC, src), "-o", out],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    seen, inside = set(), None
    for line in open(out):
        if line.startswith("define "):
            m = re.search(r"@(" + WRAPPING[src] + r"\w*)\(", line)
            inside = m and m.group(1)
            seen |= {inside} - {None}
        elif inside:
            assert not re.search(r"= (add|sub) nsw i64 (?!0, )", line), (inside, line)   # (0 - x: a bound's sign)
    assert seen
