"""Where a plan says that a slim tile runs (VecopsHipPlan.slim_tile): in the library's own plans, never for a family that a
caller requires or prefers and gets."""
import ctypes as C

from vecops_amd import capi

import pytest

from test_capi_cpu import _operand, _plan, _plan_family
from test_slim_gpu import BF16, INT8, SHAPES


def _product(dtype, m, n, k, out):
    return _operand(dtype, (m, k)), _operand(dtype, (n, k)), _operand(out, (m, n))


def test_own_plans_name_the_slim_tile_and_requested_families_do_not():
    call = _product(capi.BF16, 64, 2048, 1408, capi.F32)
    rc, own = _plan(*call)
    assert rc == 0 and capi.FAMILY_NAMES[own.family] == "tile_64" and own.slim_tile == 256 * 32 + 16 and own.b_layout == 0
    rc, automatic = _plan_family(*call, "tile_256", capi.SELECT_AUTOMATIC)
    assert rc == 0 and bytes(automatic) == bytes(own)
    for selection in (capi.SELECT_REQUIRE, capi.SELECT_PREFER):
        for split in (0, 1):
            rc, named = _plan_family(*call, "tile_64", selection, split_k=split)
            assert rc == 0 and capi.FAMILY_NAMES[named.family] == "tile_64" and named.slim_tile == 0
    # a preferred family that cannot serve: the library's own choice
    rc, preferred = _plan_family(*call, "skinny", capi.SELECT_PREFER)
    assert rc == 0 and bytes(preferred) == bytes(own)
    # big products, other layouts and operand classes: none
    for a, b, c in (_product(capi.BF16, 4096, 4096, 4096, capi.F32), _product(capi.U8, 64, 2048, 1408, capi.I32),
                    _product(capi.F32, 64, 2048, 1408, capi.F32), _product(capi.F64, 64, 2048, 1408, capi.F64),
                    (call[0], _operand(capi.BF16, (2048, 1408), strides=(1, 2048)), call[2])):
        rc, p = _plan(a, b, c)
        assert rc == 0 and p.slim_tile == 0


def test_the_plan_record_kept_its_size():
    assert C.sizeof(capi.Plan) == 32 and capi.Plan.peeled_columns.offset == 20


@pytest.mark.parametrize("tile", list(SHAPES))
def test_the_tile_of_every_shape(tile):
    want = 0 if tile == "none" else 256 * int(tile.split("x")[0]) + int(tile.split("x")[1])
    for m, n, k in SHAPES[tile]:
        for dtype in (capi.BF16, capi.F16):
            for out in (dtype, capi.F32):        # (the result's type does not enter)
                rc, p = _plan(*_product(dtype, m, n, k, out))
                assert rc == 0 and p.slim_tile == want, (m, n, k, hex(p.slim_tile))
    for (bm, bn), (m, n, k) in BF16.items():
        assert _plan(*_product(capi.BF16, m, n, k, capi.F32))[1].slim_tile == 256 * bm + bn
    for (bm, bn), (m, n, k) in INT8.items():
        assert _plan(*_product(capi.I8, m, n, k, capi.I32))[1].slim_tile == 256 * bm + bn


def test_one_round_and_what_it_replaces():
    """More than one workgroup a compute unit: never (a second round's start and the first one's stores lie between).  128x128
    tiles only in place of the four-stage kernel, whose short K is its own (4384 x 384 x 512: 7.4 us there, 9.0 on a slim tile)."""
    for (m, n, k), dtype in (((4384, 384, 512), capi.BF16), ((736, 2048, 512), capi.BF16), ((2797, 608, 568), capi.BF16),
                             ((5888, 512, 1000), capi.BF16), ((736, 3040, 6464), capi.I8), ((1152, 2040, 2080), capi.BF16),
                             ((256, 7808, 397), capi.BF16)):
        rc, p = _plan(*_product(dtype, m, n, k, capi.I32 if dtype == capi.I8 else capi.F32))
        assert rc == 0 and p.slim_tile == 0, (m, n, k, hex(p.slim_tile))
    batch, m, n, k = 13, 1, 3776, 1340
    rc, p = _plan(_operand(capi.BF16, (batch, m, k)), _operand(capi.BF16, (batch, n, k)), _operand(capi.F32, (batch, m, n)))
    assert rc == 0 and p.slim_tile == 0
    # level or ahead where the vendor grid's and the table's own examples lie
    for (m, n, k), dtype in (((512, 4096, 4096), capi.BF16), ((1024, 2048, 4096), capi.BF16), ((512, 4096, 4096), capi.I8),
                             ((1024, 2048, 4096), capi.I8)):
        rc, p = _plan(*_product(dtype, m, n, k, capi.I32 if dtype == capi.I8 else capi.BF16))
        assert rc == 0 and p.slim_tile == 256 * 128 + 64, (m, n, k)
    rc, p = _plan(*_product(capi.I8, 512, 4096, 11008, capi.I32))      # level: 37.4 us in two parts, 37.8 on a slim tile
    assert rc == 0 and p.slim_tile == 0 and p.split_k == 2
