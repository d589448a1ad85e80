"""CPU checks of how the split-KV P.V launch shares out rows
(fmha_amd/csrc/fmha_decode_pieces.hpp).  The host sizes the workspace, the
counts and the grid from the longest row allowed; the device then picks the
size of a piece from the lengths that are there.  Whatever the lengths, the
pieces it makes must fit what the host set aside, and a batch that is as full
as the host assumed keeps the host's size."""
import ctypes
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "fmha_amd", "csrc")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("pieces") / "libpv_pieces.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Werror", "-fsanitize=signed-integer-overflow",
                    "-fsanitize-undefined-trap-on-error", "-I" + CSRC, "-o", out,
                    os.path.join(HERE, "native", "pv_pieces_shim.cpp")], check=True)
    return ctypes.CDLL(out)


def _plan(lib, batch, units, g, max_rows, d, forced=0, scattered=0):
    out = (ctypes.c_int64 * 6)()
    lib.pv_plan(ctypes.c_int64(batch), units, g, max_rows, d, scattered, forced, out)
    return dict(zip(("shift", "fine", "parts", "npv", "total", "full"), out))


def _take(lib, batch, units, g, max_rows, d, lens, forced=0, uniform=0, scattered=0):
    got = [ctypes.c_int64() for _ in range(3)]
    lib.pv_take(ctypes.c_int64(batch), units, g, max_rows, d, scattered, forced, uniform, (ctypes.c_int32 * len(lens))(*lens),
                *(ctypes.byref(x) for x in got))
    return [x.value for x in got]


def _lengths(rng, batch, max_rows):
    kind = rng.randrange(6)
    if kind == 0:
        return [max_rows] * batch
    if kind == 1:
        return [rng.choice((0, -1, max_rows + 1, 2 ** 31 - 1, -(2 ** 31))) for _ in range(batch)]
    if kind == 2:
        return [rng.randint(0, max_rows) for _ in range(batch)]
    if kind == 3:  # one long row among short ones
        return [max_rows] + [rng.randint(0, min(20, max_rows)) for _ in range(batch - 1)]
    if kind == 4:  # next to the edges of a piece
        return [min(max_rows, max(0, (1 << rng.randint(7, 13)) * rng.randint(0, 40) + rng.randint(-1, 1)))
                for _ in range(batch)]
    return [int(max_rows ** rng.random()) for _ in range(batch)]


def test_pieces_fit_what_the_host_set_aside(lib):
    rng = random.Random(1)
    finer = 0
    for i in range(20000):
        batch = rng.choice((1, 1, 2, 3, rng.randint(1, 64), rng.randint(65, 300)))
        units = rng.choice((1, 2, 3, 4, 8, 16, 32, 64))
        g = rng.choice((1, 4, 8, 16, 32))
        d = rng.choice((64, 128, 256))
        max_rows = rng.choice((rng.randint(17, 300), rng.randint(17, 9000), int(2 ** rng.uniform(5, 28))))
        forced = rng.choice((0, 0, 0, 128, 512, 4096))
        uniform = int(rng.random() < 0.1)
        scattered = rng.randrange(2)
        lens = _lengths(rng, batch, max_rows)
        p = _plan(lib, batch, units, g, max_rows, d, forced, scattered)
        shift, pieces, most = _take(lib, batch, units, g, max_rows, d, lens, forced, uniform, scattered)
        case = (batch, units, g, max_rows, d, scattered, forced, uniform, lens[:8], p, shift, pieces, most)
        assert p["fine"] <= shift <= p["shift"], case
        assert pieces <= p["total"] and most <= p["npv"], case
        assert shift == p["shift"] or not (forced or uniform or batch > 256), case
        assert p["parts"] == 1 or d == 256, case
        finer += shift < p["shift"]
    assert finer > 1000  # the device's own choice is among what is checked


def test_full_batches_keep_the_planned_size(lib):
    for batch, units, max_rows, d in ((3, 4, 66558, 256), (1, 8, 108751, 256), (8, 8, 32768, 128), (57, 8, 2233, 64)):
        p = _plan(lib, batch, units, 4, max_rows, d)
        assert p["shift"] == 12  # few, long pieces
        assert _take(lib, batch, units, 4, max_rows, d, [max_rows] * batch)[0] == 12
        short = [max_rows // 20] * batch
        assert _take(lib, batch, units, 4, max_rows, d, short)[0] < 12
