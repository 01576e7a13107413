"""Where a plan says that a slim tile runs (VecopsHipPlan.slim_tile): in the library's own plans, never for a family that a
caller requires or prefers and gets."""
import ctypes as C

from vecops_amd import capi

from test_capi_cpu import _operand, _plan, _plan_family


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
