"""Index arithmetic of packed canvas reads (kernels/k44_pack_index.hpp, what the kernel and its
launch use) on the host, around 2^31 and 2^32 elements, against Python's integers."""
import ctypes
import subprocess
from pathlib import Path

import pytest

KERNELS = Path(__file__).resolve().parents[1] / "snntome_amd" / "csrc" / "kernels"
SOURCE = r"""
#include "k44_pack_index.hpp"
extern "C" unsigned at(uint64_t first, uint64_t n, uint64_t cols, uint64_t q, uint64_t *rc) {
    unsigned bits = 0;
    k44dev::with_pack_index(first, n, cols, [&](auto f, auto k, auto w) {
        using I = decltype(f);
        static_assert(sizeof(f) == sizeof(k) && sizeof(f) == sizeof(w), "one index type");
        const auto p = k44dev::row_col<I>((I)(f + (I)q), w);
        rc[0] = p.r;
        rc[1] = p.c;
        bits = 8u * sizeof(I);
    });
    return bits;
}
"""


@pytest.fixture(scope="module")
def at(tmp_path_factory):
    d = tmp_path_factory.mktemp("pack")
    (d / "at.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC",
                    f"-I{KERNELS}", str(d / "at.cpp"), "-o", str(d / "at.so")], check=True)
    fn = ctypes.CDLL(str(d / "at.so")).at
    fn.argtypes = [ctypes.c_uint64] * 4 + [ctypes.POINTER(ctypes.c_uint64)]
    fn.restype = ctypes.c_uint

    def call(first, n, cols, q):
        rc = (ctypes.c_uint64 * 2)()
        bits = fn(first, n, cols, q, rc)
        return bits, (rc[0], rc[1])

    return call


PART = 1 << 19  # elements of a pageable read's parts


@pytest.mark.parametrize("cols", [1, 7, 64, 2**19 + 1, 2**31 - 1, 2**31, 2**32 - 1, 2**32, 2**32 + 64,
                                  2**33 + 2**20, 10_200_000_000])
def test_rows_and_columns(at, cols):
    """Every part of a read around the limits, first to last element of the part."""
    for edge in (0, PART, 2**31 - PART, 2**31, 2**32 - PART, 2**32, cols - cols % PART):
        for first in {max(0, edge - PART), edge}:
            for q in (0, 8, 64, PART - 8, PART - 1):
                bits, got = at(first, PART, cols, q)
                assert got == divmod(first + q, cols), (first, q)
                assert bits == (32 if first + PART < 2**31 and cols < 2**32 else 64)
