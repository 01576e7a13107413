"""How the quantisation of contiguous rows is dealt to workgroups (csrc/row_work_split.h, whole-number arithmetic shared by
the kernels, their launches and this test): every element once, no position outside its row, at the ends of the range."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vecops_amd", "csrc")
INT32_MAX = 2 ** 31 - 1

SOURCE = """
#include "row_work_split.h"
using namespace vecops_hip;
extern "C" {
int64_t pieces(int64_t k) { return quantize_pieces(k); }
// first elements of the quads of one piece, [lane][i], and which of them lie whole in a row of k
void piece_quads(int64_t piece, int64_t k, int64_t* first, uint8_t* whole) {
  for (int lane = 0; lane < 256; ++lane)
    for (int i = 0; i < kQuantizeQuads; ++i) {
      *first = quantize_quad(piece, lane, i);
      *whole++ = quantize_quad_is_whole(*first++, k);
    }
}
}
"""


@pytest.fixture(scope="module")
def split(tmp_path_factory):
    where = tmp_path_factory.mktemp("row_work_split")
    source, out = where / "split.cpp", where / "split.so"
    source.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=undefined", "-fno-sanitize-recover=all", "-shared", "-fPIC", "-Wall",
                    "-Werror", "-I", CSRC, "-o", str(out), str(source)], check=True)
    lib = C.CDLL(str(out))
    lib.pieces.restype = C.c_int64
    lib.pieces.argtypes = [C.c_int64]
    lib.piece_quads.argtypes = [C.c_int64, C.c_int64, C.c_void_p, C.c_void_p]
    return lib


@pytest.mark.parametrize("k", [1, 4, 1023, 2047, 2048, 2049, 4097, INT32_MAX - 2048, INT32_MAX - 2047, INT32_MAX - 255, INT32_MAX])
def test_a_row_s_last_piece_covers_its_end_and_nothing_before_it(split, k):
    last = split.pieces(k) - 1
    quads, whole = np.zeros(512, np.int64), np.zeros(512, np.uint8)
    split.piece_quads(last, k, quads.ctypes.data, whole.ctypes.data)
    assert np.array_equal(np.sort(quads), last * 2048 + 4 * np.arange(512))
    assert np.array_equal(whole.astype(bool), quads <= k - 4)        # no lane reads or writes four past the row's end
    assert last * 2048 < k <= (last + 1) * 2048
