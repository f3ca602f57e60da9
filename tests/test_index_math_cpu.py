"""The kernels' integer formulas (csrc/index_math.hpp) over the whole range the
entry points accept, compiled for the host from the text the kernels use."""
import ctypes
import subprocess

import pytest

from conftest import PKG_DIR

CSRC = PKG_DIR / "attnkernels" / "csrc"
WRAPPERS = """
#include <cmath>

#include "index_math.hpp"
extern "C" {
size_t page_row_offset(int t, int bs, int d) { return ak::page_row_offset(t, bs, d); }

int split_count(int c, int size, float reciprocal) { return ak::split_count(c, size, reciprocal); }

// Contexts just below, at and just above every multiple of size, with the
// reciprocal a unit low, right and a unit high: the first wrong one, or -1.
int first_wrong(int size) {
    for (int u = -1; u <= 1; ++u) {
        float r = 1.f / (float)size;
        if (u) r = std::nextafter(r, u > 0 ? 2.f : 0.f);
        for (int m = 0; m < (1 << 24); m += size)
            for (int c = m - 2; c <= m + 2; ++c)
                if (c >= 0 && c < (1 << 24) && ak::split_count(c, size, r) != (c + size - 1) / size) return c;
    }
    return -1;
}
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("index_math")
    (d / "w.cpp").write_text(WRAPPERS)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", str(CSRC), str(d / "w.cpp"), "-o",
                    str(d / "w.so")], check=True)
    L = ctypes.CDLL(str(d / "w.so"))
    L.page_row_offset.argtypes, L.page_row_offset.restype = [ctypes.c_int] * 3, ctypes.c_size_t
    L.split_count.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_float]
    L.first_wrong.argtypes = [ctypes.c_int]
    return L


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("shift", [4, 5, 12, 23, 24, 25, 30])
def test_row_offsets_of_pages_of_any_size(lib, d, shift):
    """Up to one page of 2^30 tokens (block tables hold at most 2^31 - 1 tokens), past
    the 2^24 rows whose offsets in elements fit 32 bits."""
    bs, last = 1 << shift, (1 << 31) - 1
    for t in (0, 15, 16, bs - 16, bs - 1, bs, bs + 17, (1 << 24) - 16, 1 << 24, (1 << 25) + 48, last - 16, last):
        if 0 <= t <= last:
            assert lib.page_row_offset(t, bs, d) == t % bs * d, (t, bs)


def test_the_whole_chunk_loops_use_it():
    """Both grouped-query kernels read pages of 16, 32, ... tokens from a chunk's first row."""
    text = (CSRC / "decode.hip").read_text()
    assert text.count("page_stride + page_row_offset(t, bs, D)") == 2
    assert "page_stride + (t & (bs - 1))" not in text


def test_split_counts_are_exact_up_to_2_24_tokens(lib):
    """Every multiple of a split size, and its neighbours, with a reciprocal off by a unit either way."""
    for size in [*range(32, 4097, 32), *range(4096 + 64, 1 << 17, 4096 + 64), 29216, 33152, 1 << 20, (1 << 24) - 64, 1 << 24]:
        assert lib.first_wrong(size) == -1, size
