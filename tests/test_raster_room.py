"""Scratch memory of the device raster (csrc/raster_room.hpp), compiled for the
host: scenes whose tile lists do not fit are drawn in two passes, whose list is
one word per triangle, and the lists hold whatever comes where they say so."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "dynamicradiancevolume_amd" / "csrc"
NO_MEMORY, OTHER = -3, -2


@pytest.fixture(scope="module")
def rr(tmp_path_factory):
    d = tmp_path_factory.mktemp("raster_room")
    src = d / "rr.cpp"
    src.write_text('#include "raster_room.hpp"\nextern "C" {\n'
                   "uint64_t words(int w, int h, uint32_t n) { return drvk::raster_work_words(w, h, n); }\n"
                   "uint64_t least(uint32_t n) { return drvk::raster_least_words(n); }\n"
                   "void room(int w, int h, uint32_t n, uint64_t* o) { const auto r = drvk::tile_room(w, h, n);"
                   " o[0] = r.pairs; o[1] = r.wide; o[2] = r.cut; o[3] = r.all; }\n"
                   "int reserve(uint64_t words, uint64_t least, size_t* refused, int no_memory, int (*f)(uint64_t))"
                   "{ return drvk::reserve_raster_words(words, least, refused, no_memory, f); }\n"
                   "}\n")
    so = d / "librr.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", str(CSRC), str(src), "-o", str(so)],
                   check=True)
    lib = C.CDLL(str(so))
    lib.words.restype = lib.least.restype = C.c_uint64
    lib.words.argtypes = [C.c_int, C.c_int, C.c_uint32]
    lib.least.argtypes = [C.c_uint32]
    return lib


def _reserve(lib, words, least, refused, fits):
    """The sizes tried and the result; `fits` maps a size to a return code."""
    tried = []

    @C.CFUNCTYPE(C.c_int, C.c_uint64)
    def f(n):
        tried.append(n)
        return fits(n)

    rc = lib.reserve(C.c_uint64(words), C.c_uint64(least), C.byref(refused), NO_MEMORY, f)
    return tried, rc


def test_lists_that_do_not_fit_leave_the_two_passes(rr):
    big = rr.words(1920, 1080, 1 << 24)
    least = rr.least(1 << 24)
    assert least == (1 << 24) + 1 and big > 16 * least
    small = rr.words(1920, 1080, 1000)
    refused = C.c_size_t(2 ** 64 - 1)
    def room(n):
        return 0 if n < big else NO_MEMORY
    assert _reserve(rr, big, least, refused, room) == ([big, least], 0)
    assert _reserve(rr, big, least, refused, room) == ([least], 0)  # not tried again
    assert _reserve(rr, small, 1001, refused, room) == ([small], 0)  # less may still fit
    # nothing fits, or something else fails
    refused = C.c_size_t(2 ** 64 - 1)
    assert _reserve(rr, big, least, refused, lambda n: NO_MEMORY) == ([big, least], NO_MEMORY)
    refused = C.c_size_t(2 ** 64 - 1)
    assert _reserve(rr, big, least, refused, lambda n: OTHER) == ([big], OTHER)
    assert refused.value == 2 ** 64 - 1
    # a window that takes the two passes anyway is tried once, also after a refusal
    refused = C.c_size_t(5)
    assert _reserve(rr, least, least, refused, lambda n: NO_MEMORY) == ([least], NO_MEMORY)
    assert refused.value == 5


@pytest.mark.parametrize("w,h", [(384, 256), (1920, 1080), (3840, 2160), (65536, 16), (16384, 16384)])
def test_room_holds_what_it_promises(rr, w, h):
    o = (C.c_uint64 * 4)()
    tiles = -(-w // 16) * -(-h // 16)
    for n in (0, 1, 2, 1000, 16000, 32768, 33825, 33826, 70000, 1 << 20, 1 << 24):
        rr.room(w, h, n, o)
        pairs, wide, cut, everything = o
        # a triangle has at most two pieces of at most 64 tiles, each in a list or a record
        if everything:
            assert pairs >= 128 * n and wide >= 2 * n and cut >= 2 * n
        assert pairs <= 4 * n + (1 << 22) and wide <= 65536 and cut <= 65536
        assert wide * tiles <= max(1 << 30, 256 * tiles)
        assert pairs + 2 * 64 * n < 2 ** 32  # claimed in 32 bits
        assert rr.words(w, h, n) == 8 + 2 * n + 2 * tiles + 4 * (pairs + wide + cut)
        assert rr.words(w, h, n) >= rr.least(n) and 4 * rr.words(w, h, n) <= 72 * n + (70 << 20) + 8 * tiles
    assert rr.words(256, 256, 1000) == rr.words(w, h, (1 << 24) + 1) - (1 << 24) - 1 + 1000 == 1001
