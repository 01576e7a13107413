"""The four-stage 128x128 kernel with a partial last K tile, rows at any alignment, and B as [K,N] with any N.  Operands are small
integers: sums are exact and compared bit for bit; what lies around the operands' rows is NaN and must reach no element of C."""
import pytest

pytestmark = pytest.mark.gpu


def _inside_nan(values, pad, offset):
    import torch
    rows, cols = values.shape
    nan = float("nan") if values.dtype.is_floating_point else 77
    store = torch.full((offset + rows * (cols + pad) + 64,), nan, dtype=values.dtype, device=values.device)
    view = store[offset:offset + rows * (cols + pad)].view(rows, cols + pad)[:, :cols]
    view.copy_(values)
    return view


# (m, n): more than half the units, few tiles; K: one element past a K tile, one short of it, a single whole one among few
@pytest.mark.parametrize("m,n", [(1400, 1300), (1000, 1793), (257, 513), (100, 129)])
@pytest.mark.parametrize("k,split", [(513, 1), (575, 1), (1025, 2), (2600, 3), (520, 1), (4001, 4), (3072, 1)])
@pytest.mark.parametrize("kind,layout,pad,offset", [("bf16", "nk", 0, 0), ("f16", "nk", 1, 1), ("i8", "nk", 3, 5), ("bf16", "kn", 0, 0), ("f16", "kn", 3, 1)])
def test_against_exact_sums(device, m, n, k, split, kind, layout, pad, offset):
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
    capi.matmul_family(a, b, c, capi.family_request("tile_128", capi.SELECT_REQUIRE, split_k=split))
    torch.cuda.synchronize()
    assert torch.equal(c, sums.to(c.dtype))
    capi.matmul(a, b, c.fill_(77))           # the library's own plan
    torch.cuda.synchronize()
    assert torch.equal(c, sums.to(c.dtype))


def test_batches(device):
    import torch
    from vecops_amd import capi
    gen = torch.Generator().manual_seed(4)
    a = torch.randint(-3, 4, (5, 777, 3001), generator=gen).bfloat16().to(device)
    b = torch.randint(-3, 4, (5, 801, 3001), generator=gen).bfloat16().to(device)
    c = torch.empty((5, 777, 801), dtype=torch.float32, device=device)
    capi.matmul_family(a, b, c, capi.family_request("tile_128", capi.SELECT_REQUIRE, split_k=1))
    torch.cuda.synchronize()
    assert torch.equal(c, torch.matmul(a.double(), b.double().transpose(1, 2).contiguous()).float())
