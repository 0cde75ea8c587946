"""Where the few-row GEMM keeps its bf16 activation (csrc/fragment_layout.h, plain
C++ on the host): every element has a place of its own, also in rows of more than
2^30 elements, whose byte and word offsets leave 32 bits (CPU only)."""

import ctypes
import subprocess

import pytest

from conftest import PKG_ROOT

SRC = r"""
#include "fragment_layout.h"
extern "C" uint64_t word(int64_t tile, int64_t steps, int64_t step, int half, int lane) {
  return hif8::fragment_word(tile, steps, step, half, lane);
}
extern "C" uint64_t word_of_k(int k0) { return hif8::fragment_word(0, 0, k0 / hif8::kStepK, 0, 0); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("frag")
    (d / "frag.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{PKG_ROOT / 'csrc'}", str(d / "frag.cpp"),
                    "-o", str(d / "libfrag.so")], check=True)
    lib = ctypes.CDLL(str(d / "libfrag.so"))
    lib.word.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int] * 2
    lib.word.restype = lib.word_of_k.restype = ctypes.c_uint64
    return lib


def test_fragments_tile_the_operand(lib):
    steps = 3
    words = [lib.word(t, steps, s, h, lane) for t in range(2) for s in range(steps) for h in range(2)
             for lane in range(64)]
    assert words == list(range(2 * steps * 128))


@pytest.mark.parametrize("k", [2 ** 20, 2 ** 30 - 64, 2 ** 30, 2 ** 30 + 64, 2 ** 31 - 64])
def test_offsets_of_long_rows(lib, k):
    assert lib.word_of_k(k) == 2 * k
    steps = k // 64
    assert lib.word(1, steps, steps - 1, 1, 63) == 4 * k - 1
