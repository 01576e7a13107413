"""How sums leave the tile kernels by whole rows of a wavefront's tile (store_rows in tile_gemm.h): C inputs, bias rows, fused
transforms, the output types, rows of C and of the C input at any alignment, tiles cut off at the edges.

Operands, C inputs, scales and shifts are small integers or powers of two, so that every sum and every step of the transform is
exact in fp32 and only the conversion to C's type rounds: results are compared bit for bit (silu, whose two transcendentals are
the hardware's, to a few units in the last place of an fp32 result rounded once more)."""
import pytest

pytestmark = pytest.mark.gpu

FAMILIES = ["tile_256", "tile_256x128", "tile_128x256", "tile_192", "tile_128", "tile_64"]


def _ints(gen, shape, low, high, dtype, device):
    import torch
    return torch.randint(low, high + 1, shape, generator=gen).to(dtype).to(device)


def _strided(t, pad, offset):
    """The same values in rows `pad` elements longer, `offset` elements into their storage."""
    import torch
    rows, cols = t.shape
    store = torch.zeros(rows * (cols + pad) + offset, dtype=t.dtype, device=t.device)
    view = store[offset:].view(rows, cols + pad)[:, :cols]
    view.copy_(t)
    return view


def _dtypes():
    import torch
    return {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


# n: whole eights, odd, and less than a lane's eight columns in the last tile; k: short enough for the exactness, ragged
@pytest.mark.parametrize("family", FAMILIES)
@pytest.mark.parametrize("m,n,k", [(300, 392, 96), (257, 391, 128), (512, 512, 640), (193, 259, 72)])
@pytest.mark.parametrize("src,out,cin", [("bf16", "bf16", None), ("f16", "f16", None), ("bf16", "f32", None), ("f16", "f16", "f16"),
                                         ("bf16", "bf16", "bf16"), ("bf16", "f32", "f32"), ("bf16", "bf16", "f32"),
                                         ("f16", "f32", "f16"), ("bf16", "bf16", "row bf16"), ("f16", "f32", "row f32"),
                                         ("f16", "f16", "row f32")])
def test_outputs_and_c_inputs(device, family, m, n, k, src, out, cin):
    import torch
    from vecops_amd import capi
    if family == "tile_192" and k % 8 != 0:
        pytest.skip("the 192 x 192 tile takes 16-byte aligned rows")
    t, gen = _dtypes(), torch.Generator().manual_seed(m + n + k)
    a, b = _ints(gen, (m, k), -3, 3, t[src], device), _ints(gen, (n, k), -3, 3, t[src], device)
    sums = a.float() @ b.float().t()
    c_in = None
    if cin is not None:
        row, kind = cin.startswith("row "), t[cin.split()[-1]]
        c_in = _ints(gen, (1 if row else m, n), -9, 9, kind, device)
        sums = sums + c_in.float()
        c_in = c_in.expand(m, n) if row else c_in
    want = sums.to(t[out])
    # C (and a full C input) dense, and in rows and at a base that line up with nothing
    for pad, offset in ((0, 0), (3, 1)):
        c = _strided(torch.full((m, n), 77.0, dtype=t[out], device=device), pad, offset)
        given = _strided(c_in, pad + 2, offset) if c_in is not None and not cin.startswith("row ") else c_in
        capi.matmul_family(a, b, c, capi.family_request(family, capi.SELECT_REQUIRE, split_k=1), c_in=given)
        torch.cuda.synchronize()
        assert torch.equal(c, want), (pad, offset)
    if cin == out:  # accumulated in place: C is its own C input
        c = c_in.clone()
        capi.matmul_family(a, b, c, capi.family_request(family, capi.SELECT_REQUIRE, split_k=1), c_in=c)
        torch.cuda.synchronize()
        assert torch.equal(c, want)


@pytest.mark.parametrize("m,n,k", [(128, 16384, 512), (1000, 4001, 512), (4096, 4096, 512), (2000, 5001, 264), (700, 900, 640)])
@pytest.mark.parametrize("src,out", [("bf16", "bf16"), ("f16", "f16"), ("bf16", "f32"), ("f16", "f32")])
@pytest.mark.parametrize("form", ["relu bias", "clamp scales", "rows only", "full"])
def test_fused_transforms(device, m, n, k, src, out, form):
    import torch
    from vecops_amd import capi
    t, gen = _dtypes(), torch.Generator().manual_seed(m * 3 + n + k)
    a, b = _ints(gen, (m, k), -2, 2, t[src], device), _ints(gen, (n, k), -2, 2, t[src], device)
    x, c_in = a.float() @ b.float().t(), None
    if form == "relu bias":
        bias = _ints(gen, (1, n), -9, 9, t[src], device)
        x, c_in = (x + bias.float()).clamp_min(0.0), bias.expand(m, n)
        ep = capi.epilogue(activation="relu")
    elif form == "clamp scales":
        rows, cols = 2.0 ** _ints(gen, (m,), -2, 1, torch.float32, device), 2.0 ** _ints(gen, (n,), -1, 2, torch.float32, device)
        x = (((x * rows[:, None]) * cols) * 0.5 + 3.0).clamp(-40.0, 50.0)
        ep = capi.epilogue(activation="clamp", scale=0.5, shift=3.0, row_scales=rows, column_scales=cols, clamp=(-40.0, 50.0))
    elif form == "rows only":
        rows = 2.0 ** _ints(gen, (m,), -2, 1, torch.float32, device)
        x = x * rows[:, None]
        ep = capi.epilogue(row_scales=rows)
    else:
        c_in = _ints(gen, (m, n), -9, 9, t[src], device)
        x = (x + c_in.float()) * 0.25
        ep = capi.epilogue(scale=0.25)
    c = torch.full((m, n), 77.0, device=device).to(t[out])
    capi.matmul_fused(a, b, c, ep, c_in=c_in)
    torch.cuda.synchronize()
    assert torch.equal(c, x.to(t[out]))


@pytest.mark.parametrize("m,n,k", [(1000, 4001, 512), (4096, 4096, 512)])
def test_silu(device, m, n, k):
    import torch
    from vecops_amd import capi
    gen = torch.Generator().manual_seed(5)
    a, b = (_ints(gen, (r, k), -2, 2, torch.bfloat16, device) for r in (m, n))
    bias = _ints(gen, (1, n), -9, 9, torch.bfloat16, device)
    x = (a.float() @ b.float().t() + bias.float()).double() / 16
    c = torch.empty((m, n), dtype=torch.float32, device=device)
    capi.matmul_fused(a, b, c, capi.epilogue(activation="silu", scale=1 / 16), c_in=bias.expand(m, n))
    torch.cuda.synchronize()
    want = x * torch.sigmoid(x)
    # the exponential and the reciprocal are each within 1 ulp, the exponential's argument within 1/2 ulp of |x| <= 64: 2^-18
    # relative at most
    assert ((c.double() - want).abs() <= want.abs() * 2.0 ** -17 + 1e-30).all()


@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("out", ["bf16", "f16", "f32"])
def test_values_that_are_no_numbers(device, value, out):
    """In the operands, in a C input and in a bias row: they arrive in the elements they belong to and nowhere else."""
    import torch
    from vecops_amd import capi
    t, gen = _dtypes(), torch.Generator().manual_seed(9)
    src = torch.float16 if out == "f16" else torch.bfloat16
    m, n, k = 520, 777, 320
    a, b = _ints(gen, (m, k), 1, 2, src, device), _ints(gen, (n, k), 1, 2, src, device)
    c_in = torch.zeros((m, n), dtype=t[out], device=device)
    a[17, 5] = value
    c_in[400, 776] = value
    c = torch.empty((m, n), dtype=t[out], device=device)
    capi.matmul(a, b, c, c_in=c_in)
    torch.cuda.synchronize()
    plain = torch.isfinite(c)
    expected = torch.ones_like(plain)
    expected[17, :] = False
    expected[400, 776] = False
    assert torch.equal(plain, expected)


@pytest.mark.parametrize("family", ["tile_256", "tile_128x256", "tile_128", "tile_64"])
@pytest.mark.parametrize("m,n,k", [(300, 391, 96), (257, 259, 640)])
def test_byte_operands_to_rows_that_line_up_with_nothing(device, family, m, n, k):
    import torch
    from vecops_amd import capi
    gen = torch.Generator().manual_seed(3)
    a, b = _ints(gen, (m, k), -127, 127, torch.int8, device), _ints(gen, (n, k), -127, 127, torch.int8, device)
    sums = (a.double() @ b.double().t()).to(torch.int32)
    request = capi.family_request(family, capi.SELECT_REQUIRE, split_k=1)
    for pad, offset in ((0, 0), (1, 1)):
        c = _strided(torch.full((m, n), 77, dtype=torch.int32, device=device), pad, offset)
        capi.matmul_family(a, b, c, request)
        torch.cuda.synchronize()
        assert torch.equal(c, sums)
        c_in = _strided(_ints(gen, (m, n), -1000, 1000, torch.int32, device), pad + 1, offset)
        capi.matmul_family(a, b, c, request, c_in=c_in)
        torch.cuda.synchronize()
        assert torch.equal(c, sums + c_in)


@pytest.mark.parametrize("m,n,k", [(600, 1003, 256), (2000, 4097, 384), (2048, 11007, 512)])
def test_dequantised_rows_that_line_up_with_nothing(device, m, n, k):
    import torch
    from vecops_amd import capi
    gen = torch.Generator().manual_seed(4)
    a, b = _ints(gen, (m, k), -127, 127, torch.int8, device), _ints(gen, (n, k), -127, 127, torch.int8, device)
    rows, cols = 2.0 ** _ints(gen, (m,), -9, -5, torch.float32, device), 2.0 ** _ints(gen, (n,), -9, -5, torch.float32, device)
    c = torch.empty((m, n), dtype=torch.float32, device=device)
    capi.matmul_i8_dequant(a, b, rows, cols, c)
    torch.cuda.synchronize()
    assert torch.equal(c, ((a.double() @ b.double().t()).float() * rows[:, None]) * cols)


# C inputs that go into the sums in LDS (of another width than C's, before a transform, past a lane's whole share): every
# remainder of four columns, fewer than four in all, tiles of every shape cut off anywhere
@pytest.mark.parametrize("family", FAMILIES)
@pytest.mark.parametrize("m,n", [(257, 388), (300, 389), (200, 390), (129, 391), (520, 513), (70, 1), (40, 2), (33, 3), (65, 5)])
@pytest.mark.parametrize("src,out,cin", [("bf16", "bf16", "f32"), ("f16", "f32", "f16"), ("bf16", "f32", "f32"), ("f16", "f16", "f16")])
def test_c_inputs_of_any_width_and_extent(device, family, m, n, src, out, cin):
    import torch
    from vecops_amd import capi
    t, gen, k = _dtypes(), torch.Generator().manual_seed(m * n), 96
    a, b = _ints(gen, (m, k), -3, 3, t[src], device), _ints(gen, (n, k), -3, 3, t[src], device)
    c_in = _ints(gen, (m, n), -9, 9, t[cin], device)
    want = (a.float() @ b.float().t() + c_in.float()).to(t[out])
    request = capi.family_request(family, capi.SELECT_REQUIRE, split_k=1)
    for pad, offset in ((0, 0), (3, 1)):
        c = _strided(torch.full((m, n), 77.0, dtype=t[out], device=device), pad, offset)
        capi.matmul_family(a, b, c, request, c_in=_strided(c_in, pad + 2, offset))
        torch.cuda.synchronize()
        assert torch.equal(c, want), (pad, offset)


@pytest.mark.parametrize("m,n,k", [(70, 3, 640), (1000, 4002, 512), (4096, 4095, 512), (300, 391, 640), (3000, 2999, 256)])
@pytest.mark.parametrize("src,out,cin", [("bf16", "bf16", "bf16"), ("f16", "f32", "f32"), ("f16", "f16", "f32"), ("bf16", "f32", "bf16")])
def test_c_inputs_before_a_transform(device, m, n, k, src, out, cin):
    import torch
    from vecops_amd import capi
    t, gen = _dtypes(), torch.Generator().manual_seed(m + 5 * n + k)
    a, b = _ints(gen, (m, k), -2, 2, t[src], device), _ints(gen, (n, k), -2, 2, t[src], device)
    c_in = _ints(gen, (m, n), -9, 9, t[cin], device)
    rows, cols = 2.0 ** _ints(gen, (m,), -2, 1, torch.float32, device), 2.0 ** _ints(gen, (n,), -1, 2, torch.float32, device)
    want = ((((a.float() @ b.float().t() + c_in.float()) * rows[:, None]) * cols) * 0.5 + 3.0).clamp_min(0.0).to(t[out])
    for pad, offset in ((0, 0), (5, 1)):
        c = _strided(torch.full((m, n), 77.0, device=device).to(t[out]), pad, offset)
        capi.matmul_fused(a, b, c, capi.epilogue(activation="relu", scale=0.5, shift=3.0, row_scales=rows, column_scales=cols),
                          c_in=_strided(c_in, pad + 1, offset))
        torch.cuda.synchronize()
        assert torch.equal(c, want), (pad, offset)
