"""Which products with a partial last K tile, or with rows that are not 16-byte aligned, the rule table gives the four-stage 128x128
kernel, and which it leaves to 64x64 tiles and slim ones.  The times beside the shapes (us): what the plan runs, and the other way."""
import ctypes as C

import pytest

from test_capi_cpu import _operand
from vecops_amd import capi


def _plan(dtype, m, n, k, cin=False):
    plan, out = capi.Plan(), capi.I32 if dtype == capi.I8 else dtype
    a, b, c = _operand(dtype, (m, k)), _operand(dtype, (n, k)), _operand(out, (m, n))
    assert capi.lib().vecops_hip_plan_matmul(C.byref(a), C.byref(b), C.byref(c) if cin else None, C.byref(c), 0, C.byref(plan)) == 0
    return capi.FAMILY_NAMES[plan.family], plan.split_k, plan.slim_tile


@pytest.mark.parametrize("dtype,m,n,k,cin,family", [
    (capi.BF16, 1256, 1752, 520, False, "tile_64"),      # 11.8, 12.4
    (capi.BF16, 1256, 1752, 1000, False, "tile_128"),    # 16.1, 17.5
    (capi.F16, 1384, 2008, 520, False, "tile_128"),      # 12.3, 12.7
    (capi.I8, 1256, 1752, 1040, False, "tile_64"),       # 13.0, 16.3
    (capi.I8, 1256, 1752, 3088, False, "tile_64"),       # 24.4, 25.0
    (capi.I8, 1256, 1752, 6160, False, "tile_128"),      # 38.5, 42.3
    (capi.I8, 1256, 1752, 6160, True, "tile_64"),        # 45.1, 50.7
    (capi.I8, 1384, 2008, 2064, False, "tile_64"),       # 20.2, 20.8
    (capi.I8, 1384, 2008, 3088, False, "tile_128"),      # 25.3, 26.4
    (capi.I8, 1384, 2008, 4112, True, "tile_64")])       # 35.5, 41.5
def test_a_partial_k_tile(dtype, m, n, k, cin, family):
    assert _plan(dtype, m, n, k, cin)[0] == family


# 128x128 tiles that are a good part padding, more of them than can be split in two: at most two 64x64 ones a unit instead
@pytest.mark.parametrize("dtype,m,n,k", [(capi.F16, 288, 5624, 2008),      # 22.3, 23.7
                                         (capi.I8, 288, 5624, 4016),       # 21.2, 27.4
                                         (capi.BF16, 288, 5624, 4001),     # 43.6, 50.0
                                         (capi.I8, 288, 5624, 8004),       # 36.8, 44.8
                                         (capi.BF16, 390, 4300, 6004),     # 55.3, 59.1
                                         (capi.I8, 513, 3300, 8001)])      # 51.7, 56.0
def test_padded_tiles(dtype, m, n, k):
    assert _plan(dtype, m, n, k)[0] == "tile_64"


# rows of whole words, which slim tiles load faster than rows at odd addresses
@pytest.mark.parametrize("dtype,m,n,k,slim", [(capi.BF16, 744, 1112, 3074, 0x4040),     # 20.1, 21.0
                                              (capi.BF16, 744, 1112, 3073, 0),          # 21.4, 23.4
                                              (capi.BF16, 744, 1112, 6002, 0),          # 27.0, 32.2
                                              (capi.I8, 744, 1112, 6152, 0x4040),       # 19.4, 21.8
                                              (capi.I8, 744, 1112, 12008, 0),           # 28.4, 31.5
                                              (capi.BF16, 488, 4056, 8004, 0x8040),     # 57.4, 65.1
                                              (capi.BF16, 150, 8000, 6004, 0),          # 47.3, 60.3
                                              (capi.I8, 150, 8000, 16004, 0),           # 60.8, 81.4
                                              (capi.BF16, 1000, 1000, 6004, 0),         # 28.1, 30.9
                                              (capi.BF16, 200, 7000, 5004, 0x8040),     # 37.8, 42.9
                                              (capi.I8, 1000, 1300, 6148, 0x8030),      # 26.0, 29.0
                                              (capi.BF16, 488, 4056, 6001, 0),          # 47.1, 53.8
                                              (capi.I8, 488, 4056, 12008, 0x8040),      # 45.1, 53.8
                                              (capi.I8, 488, 4056, 12001, 0)])          # 53.1, 60.1
def test_rows_of_words(dtype, m, n, k, slim):
    family, split, tile = _plan(dtype, m, n, k)
    assert family == "tile_128" and split > 1 and tile == slim
