"""Which tile a prepacked B is multiplied on where K, or A's rows, line up with nothing: not priced for the kernels that such rows
have without a pack, except where those rank the same."""
import ctypes as C

import pytest

from test_capi_cpu import _operand
from vecops_amd import capi


def _family(dtype, m, n, k):
    plan = capi.Plan()
    a, c = _operand(dtype, (m, k)), _operand(capi.I32 if dtype == capi.I8 else dtype, (m, n))
    assert capi.lib().vecops_hip_plan_matmul_packed_b(C.byref(a), dtype, n, None, C.byref(c), C.byref(plan)) == 0
    return capi.FAMILY_NAMES[plan.family]


# short K: 128x128 pairs (us there and on the tile that unpacked rows take: 28.9 and 35.5, 36.4 and 44.0, 38.9 and 46.1, 40 and 49,
# 55 and 62, 71 and 76; 60 and 67)
@pytest.mark.parametrize("m,n,k", [(3039, 6427, 259), (2577, 6815, 475), (3957, 4697, 513), (2869, 5728, 740), (2530, 7053, 869),
                                   (3115, 5506, 1265), (7941, 4575, 389)])
def test_pairs_of_a_short_k(m, n, k):
    for dtype in (capi.BF16, capi.F16):
        assert _family(dtype, m, n, k) == "tile_128"


# a long one: 137 us on 128x128 tiles, 113 here; 390 and 318; and on 256x256 ones, 366 and 306
@pytest.mark.parametrize("m,n,k,family", [(5000, 4000, 2001, "tile_128x256"), (3975, 6055, 6105, "tile_128x256"), (4394, 7607, 3533, "tile_256")])
def test_a_long_k(m, n, k, family):
    for dtype in (capi.BF16, capi.F16):
        assert _family(dtype, m, n, k) == family


# the two rectangles level: 21.0 us on 256x128 tiles, 19.9 on 128x256 ones; 51.4 and 47.7; int8 3 to 4 %
@pytest.mark.parametrize("m,n,k", [(1489, 3724, 751), (2500, 2500, 2501)])
def test_rectangles(m, n, k):
    for dtype in (capi.BF16, capi.F16):
        assert _family(dtype, m, n, k) == "tile_128x256"


def test_aligned_rows_are_priced_as_before():
    assert [_family(capi.BF16, *shape) for shape in ((5000, 4000, 2048), (2500, 2500, 2560), (4096, 4096, 4096))] == ["tile_256x352", "tile_128", "tile_256"]
