"""How the quantisation of contiguous rows is dealt to workgroups (csrc/row_work_split.h, whole-number arithmetic shared by
the kernels, their launches and this test): every element once, no position outside its row, launches that the device takes,
at the ends of the range."""
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
static int elements(int left) { return left >= 4 ? 4 : left > 0 ? left : 0; }
extern "C" {
int32_t by_pieces(int64_t rows, int64_t k) { return quantize_by_pieces(rows, k); }
int64_t blocks(int64_t rows, int64_t k) { return quantize_blocks(rows, k); }
int64_t sum_blocks(int64_t n, int64_t k) { return packed_sums_blocks(n, k); }
// What a workgroup takes: row, first element, elements (0: none).  By pieces [lane][i], 512 entries; by quads the first
// `most` of each lane, [lane][step], rows past the end among them.
void by_pieces_of(int64_t k, uint32_t block, int64_t* row, int64_t* first, int32_t* length) {
  const uint32_t pieces = static_cast<uint32_t>(quantize_pieces(k)), piece = block % pieces;
  for (int lane = 0; lane < 256; ++lane)
    for (int i = 0; i < kQuantizeQuads; ++i) {
      *row++ = block / pieces;
      const int begin = quantize_quad(piece, lane, i);
      *first++ = begin;
      *length++ = elements(static_cast<int>(k) - begin);
    }
}
void by_quads_of(int64_t k, uint32_t block, uint32_t blocks, int64_t most, int64_t* row, int64_t* first, int32_t* length) {
  const QuantizeWalk walk = quantize_walk(k, blocks);
  for (int lane = 0; lane < 256; ++lane) {
    QuantizeQuad at = quantize_first(walk, block * 256 + lane);
    for (int64_t step = 0; step < most; ++step, at = quantize_next(walk, at)) {
      const int begin = static_cast<int>(at.quad) * 4;
      *row++ = at.row;
      *first++ = begin;
      *length++ = elements(static_cast<int>(k) - begin);
    }
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
    lib.blocks.restype = lib.sum_blocks.restype = C.c_int64
    lib.blocks.argtypes = lib.sum_blocks.argtypes = lib.by_pieces.argtypes = [C.c_int64, C.c_int64]
    lib.by_pieces_of.argtypes = [C.c_int64, C.c_uint32] + [C.c_void_p] * 3
    lib.by_quads_of.argtypes = [C.c_int64, C.c_uint32, C.c_uint32, C.c_int64] + [C.c_void_p] * 3
    return lib


def _taken(split, by_pieces, rows, k, block, blocks, most=1):
    """Row, first element and number of elements of everything the workgroup takes."""
    count = 512 if by_pieces else 256 * most
    row, first, length = np.zeros(count, np.int64), np.zeros(count, np.int64), np.zeros(count, np.int32)
    where = [x.ctypes.data for x in (row, first, length)]
    if by_pieces:
        split.by_pieces_of(k, block, *where)
    else:
        split.by_quads_of(k, block, blocks, most, *where)
    assert (first >= 0).all() and (length >= 0).all() and (length <= 4).all()
    mine = (row < rows) & (length > 0)
    return row[mine], first[mine], length[mine]


@pytest.mark.parametrize("by_pieces", [True, False])
@pytest.mark.parametrize("k", [1, 4, 1023, 2047, 2048, 2049, 4097, INT32_MAX - 2048, INT32_MAX - 2047, INT32_MAX - 255, INT32_MAX])
def test_a_row_s_end_is_covered_and_nothing_past_it(split, by_pieces, k):
    blocks = (k + 2047) // 2048 if by_pieces else 8192
    quads = (k + 3) // 4
    most = 1 if by_pieces else (quads + 8192 * 256 - 1) // (8192 * 256)
    row, first, length = _taken(split, by_pieces, 1, k, blocks - 1 if by_pieces else (quads - 1) // 256 % 8192, blocks, most)
    assert (row == 0).all() and np.array_equal(length, np.minimum(k - first, 4))     # no lane goes past the row's end
    assert first.max() == (quads - 1) * 4


@pytest.mark.parametrize("blocks", [None, 1, 2, 3, 7])
@pytest.mark.parametrize("rows,k", [(1, 1), (1100, 3), (520, 4), (519, 5), (300, 69), (37, 512), (7, 513), (5, 1024), (3, 1025),
                                    (5, 2047), (3, 2048), (4, 2049), (9, 9001), (2, 16384)])
def test_every_element_of_every_row_once(split, rows, k, blocks):
    by_pieces = blocks is None
    if by_pieces:
        blocks = rows * ((k + 2047) // 2048)
    most = (rows * ((k + 3) // 4) + blocks * 256 - 1) // (blocks * 256)
    taken = np.zeros((rows, k), np.int64)
    for block in range(blocks):
        row, first, length = _taken(split, by_pieces, rows, k, block, blocks, most)
        for e in range(4):
            np.add.at(taken, (row[length > e], first[length > e] + e), 1)
    assert (taken == 1).all()


@pytest.mark.parametrize("n", [1, 8, 65504, 65505, 2 ** 23 - 32, 2 ** 23, 2 ** 27, 2 ** 27 + 8, 2 ** 30])
@pytest.mark.parametrize("k", [1, 512, 513, 8192])
def test_packed_row_sums_launches_stay_within_what_the_device_takes(split, n, k):
    assert 1 <= split.sum_blocks(n, k) * 256 < 2 ** 32


@pytest.mark.parametrize("rows,k", [(2 ** 24, 16), (2 ** 24 + 1, 1), (17_000_000, 64), (2 ** 23, 2048), (2 ** 23, 2049), (2 ** 25, 2049),
                                    (INT32_MAX, 1), (INT32_MAX, 4096), (1, INT32_MAX)])
def test_launches_stay_within_what_the_device_takes(split, rows, k):
    assert 1 <= split.blocks(rows, k) * 256 < 2 ** 32      # work items of a launch's dimension
    assert split.by_pieces(rows, k) == 0 or split.blocks(rows, k) == rows * ((k + 2047) // 2048)


def test_short_rows_leave_no_lane_idle(split):
    """Up to 1024 elements a row goes by quads: a workgroup's lanes take neighbouring quads across rows."""
    for k in (1, 3, 17, 64, 100, 512, 1000, 1024):
        rows = 1 << 16
        assert split.by_pieces(rows, k) == 0
        assert _taken(split, False, rows, k, 0, split.blocks(rows, k))[0].size == 256
    assert split.by_pieces(1 << 16, 1025) == 1
