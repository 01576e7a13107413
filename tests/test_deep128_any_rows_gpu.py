"""The four-stage 128x128 kernel with a partial last K tile, rows at any alignment, and B as [K,N] with any N: extents that its
rule gives it (asserted from the launched kernel's name).  Operands are small integers: sums are exact and compared bit for bit;
what lies around the operands' rows is NaN and must reach no element of C."""
import pytest

from conftest import launched_kernels

pytestmark = pytest.mark.gpu

SRC = {"bf16": 0, "f16": 5, "i8": 2}


def _inside_nan(values, pad, offset):
    import torch
    rows, cols = values.shape
    nan = float("nan") if values.dtype.is_floating_point else 77
    store = torch.full((offset + rows * (cols + pad) + 64,), nan, dtype=values.dtype, device=values.device)
    view = store[offset:offset + rows * (cols + pad)].view(rows, cols + pad)[:, :cols]
    view.copy_(values)
    return view


def _check(device, kind, layout, pad, offset, m, n, k, split):
    import torch
    from vecops_amd import capi
    dtype = {"bf16": torch.bfloat16, "f16": torch.float16, "i8": torch.int8}[kind]
    gen = torch.Generator().manual_seed(m + n + k)
    x = torch.randint(-3, 4, (m, k), generator=gen).to(dtype).to(device)
    y = torch.randint(-3, 4, (n, k), generator=gen).to(dtype).to(device)
    sums = x.double() @ y.double().t()
    a = _inside_nan(x, pad, offset)
    b = _inside_nan(y, pad, offset) if layout == "nk" else _inside_nan(y.t().contiguous(), pad, offset).t()
    c = torch.full((m, n), 77, dtype=torch.int32 if kind == "i8" else torch.float32, device=device)
    request = capi.family_request("tile_128", capi.SELECT_REQUIRE, split_k=split)
    kernels = launched_kernels(lambda: capi.matmul_family(a, b, c, request))
    partial = k % (128 if kind == "i8" else 64) != 0 or (layout == "kn" and n % 8 != 0)
    assert kernels[0] == f"tile_gemm_deep128_kernel<{SRC[kind]},{int(layout == 'kn')},0,{int(partial)}>" and len(kernels) == (2 if split > 1 else 1)
    c.fill_(77)
    capi.matmul_family(a, b, c, request)
    torch.cuda.synchronize()
    assert torch.equal(c, sums.to(c.dtype))
    capi.matmul(a, b, c.fill_(77))           # the library's own plan
    torch.cuda.synchronize()
    assert torch.equal(c, sums.to(c.dtype))


# 16-byte aligned rows: more than 128 tiles (132, 156, 180, 256); K one chunk past a K tile, one short of it, and between
@pytest.mark.parametrize("kind,m,n,k", [("bf16", 1400, 1500, 968), ("f16", 1400, 1500, 1016), ("bf16", 1531, 1663, 2600),
                                        ("f16", 1793, 1500, 520), ("bf16", 1999, 2048, 1000), ("f16", 2048, 1930, 2104),
                                        ("i8", 1400, 1500, 3472), ("i8", 1531, 1663, 3568), ("i8", 1793, 1500, 2704), ("i8", 2048, 1930, 2160)])
def test_partial_k_tile(device, kind, m, n, k):
    _check(device, kind, "nk", 0, 0, m, n, k, 1)


# rows at any alignment: 52 to 192 tiles, 48 K tiles or more; K in whole tiles, one element past one, one short of one
@pytest.mark.parametrize("kind,k,split", [("bf16", 3073, 1), ("bf16", 3135, 1), ("f16", 4001, 1), ("f16", 3136, 1), ("bf16", 4001, 2), ("f16", 3201, 4),
                                          ("i8", 6145, 1), ("i8", 6271, 1), ("i8", 6272, 1), ("i8", 7001, 2), ("i8", 8001, 4)])
@pytest.mark.parametrize("pad,offset", [(0, 0), (1, 1), (3, 5)])
def test_rows_at_any_alignment(device, kind, k, split, pad, offset):
    m, n = {1: (1200, 2200), 2: (1000, 1793), 4: (600, 1300)}[split]
    if k % 64 == 0 and pad == 0:
        pad = 1                                # (aligned rows without it)
    _check(device, kind, "nk", pad, offset, m, n, k, split)


# B as [K,N]: any count of tiles; N of every kind
@pytest.mark.parametrize("m,n", [(1400, 1300), (1000, 1793), (257, 513), (100, 129)])
@pytest.mark.parametrize("k,split", [(513, 1), (575, 1), (1025, 2), (520, 1), (3072, 1)])
@pytest.mark.parametrize("kind,pad,offset", [("bf16", 0, 0), ("f16", 3, 1)])
def test_b_as_kn(device, kind, pad, offset, m, n, k, split):
    _check(device, kind, "kn", pad, offset, m, n + (3 if n % 8 == 4 else 0), k, split)


@pytest.mark.parametrize("kind,batch,m,n,k", [("bf16", 3, 768, 896, 3201), ("f16", 2, 900, 1000, 3075), ("i8", 3, 768, 1000, 6150), ("bf16", 5, 777, 801, 968)])
def test_batches(device, kind, batch, m, n, k):
    import torch
    from vecops_amd import capi
    dtype = {"bf16": torch.bfloat16, "f16": torch.float16, "i8": torch.int8}[kind]
    gen = torch.Generator().manual_seed(4)
    a = torch.randint(-3, 4, (batch, m, k), generator=gen).to(dtype).to(device)
    b = torch.randint(-3, 4, (batch, n, k), generator=gen).to(dtype).to(device)
    c = torch.full((batch, m, n), 77, dtype=torch.int32 if kind == "i8" else torch.float32, device=device)
    request = capi.family_request("tile_128", capi.SELECT_REQUIRE, split_k=1)
    assert launched_kernels(lambda: capi.matmul_family(a, b, c, request)) == [f"tile_gemm_deep128_kernel<{SRC[kind]},0,0,1>"]
    c.fill_(77)
    capi.matmul_family(a, b, c, request)
    torch.cuda.synchronize()
    assert torch.equal(c, torch.matmul(a.double(), b.double().transpose(1, 2).contiguous()).to(c.dtype))


def test_whole_k_tiles_run_without_the_partial_ones_code(device):
    for kind, k in (("bf16", 1024), ("f16", 1024), ("i8", 2048)):
        _check(device, kind, "nk", 0, 0, 1400, 1500, k, 1)
    for kind in ("bf16", "f16"):
        _check(device, kind, "kn", 0, 0, 1000, 1496, 1024, 1)


# past the rule: the two-stage kernel (more than 192 tiles) and 64x64 tiles, in the library's own plans
@pytest.mark.parametrize("m,n,k,kernel", [(2000, 2000, 1040, "tile_gemm_kernel<2,2,2,2,2,4,4,1>"), (1256, 1752, 3088, "tile_gemm_kernel<2,2,2,1,1,0,0,1>")])
def test_bytes_with_a_short_partial_k(device, m, n, k, kernel):
    import torch
    from vecops_amd import capi
    gen = torch.Generator().manual_seed(k)
    a, b = (torch.randint(-127, 128, (rows, k), generator=gen).to(torch.int8).to(device) for rows in (m, n))
    c = torch.full((m, n), 77, dtype=torch.int32, device=device)
    assert launched_kernels(lambda: capi.matmul(a, b, c)) == [kernel]
    c.fill_(77)
    capi.matmul(a, b, c)
    torch.cuda.synchronize()
    assert torch.equal(c, (a.double() @ b.double().t()).to(torch.int32))
