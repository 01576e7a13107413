"""B handed over as [K,N] row-major with an N that is no multiple of eight, or rows that line up with nothing: the loads run along
N at any alignment, a row's last chunk reads into what lies behind it (columns of C that are never stored), and the last K tile of
a tile that does so goes through checked loads.

Operands are small integers, so that sums are exact and compared bit for bit; what lies between B's rows, in front of and behind
it is NaN and must reach no element of C."""
import pytest

pytestmark = pytest.mark.gpu

FAMILIES = ["tile_256", "tile_256x128", "tile_128x256", "tile_128", "tile_64"]


def _b_as_kn(values, pad, offset):
    """values [K,N] inside NaN: rows `pad` elements longer, `offset` elements into the storage."""
    import torch
    k, n = values.shape
    store = torch.full((offset + k * (n + pad) + 64,), float("nan"), dtype=values.dtype, device=values.device)
    b = store[offset:offset + k * (n + pad)].view(k, n + pad)[:, :n]
    b.copy_(values)
    return b.t()


def _check(device, capi, src, compute, m, n, k, pad, offset, request=None, batch=None):
    import torch
    gen = torch.Generator().manual_seed(m + 7 * n + k)
    lead = () if batch is None else (batch,)
    a = torch.randint(-3, 4, (*lead, m, k), generator=gen).to(src).to(device)
    values = torch.randint(-3, 4, (*lead, k, n), generator=gen).to(src).to(device)
    want = torch.matmul(a.double(), values.double().contiguous()).float()
    b = _b_as_kn(values, pad, offset) if batch is None else values.transpose(1, 2)
    c = torch.full((*lead, m, n), 77.0, dtype=torch.float32, device=device)
    if request is None:
        capi.matmul(a, b, c, compute=compute)
    else:
        plan = capi.plan_matmul_family(a, b, c, request, compute=compute)
        assert capi.FAMILY_NAMES[plan.family] == capi.FAMILY_NAMES[request.family] and plan.b_layout == 1 and plan.vector_b == 1
        capi.matmul_family(a, b, c, request, compute=compute)
    torch.cuda.synchronize()
    assert torch.equal(c, want)


# K: whole K tiles (the last one is then checked only where the chunks reach past N), ragged, shorter than one; N: every
# remainder of eight, one chunk and less than a chunk in the last tile, one tile exactly but for a column
@pytest.mark.parametrize("family", FAMILIES)
@pytest.mark.parametrize("src", ["bf16", "f16", "f32", "f32c"])
@pytest.mark.parametrize("m,n,k", [(300, 391, 128), (257, 255, 320), (130, 513, 77), (64, 9, 64), (70, 63, 1), (200, 260, 200)])
@pytest.mark.parametrize("pad,offset", [(0, 0), (3, 1)])
def test_families(device, family, src, m, n, k, pad, offset):
    import torch
    from vecops_amd import capi
    dtype = {"bf16": torch.bfloat16, "f16": torch.float16}.get(src, torch.float32)
    compute = capi.COMPUTE_F32 if src == "f32c" else capi.COMPUTE_BF16
    _check(device, capi, dtype, compute, m, n, k, pad, offset, capi.family_request(family, capi.SELECT_REQUIRE, split_k=1))


# (N odd, the rows of B padded to a multiple of eight elements: loads that write LDS, as aligned rows take)
@pytest.mark.parametrize("family", FAMILIES + ["tile_192"])
@pytest.mark.parametrize("src", ["bf16", "f16", "f32", "f32c"])
@pytest.mark.parametrize("m,n,k", [(300, 391, 128), (257, 255, 320), (130, 513, 77), (64, 9, 64), (520, 777, 648), (70, 63, 1)])
def test_odd_n_in_rows_that_line_up(device, family, src, m, n, k):
    import torch
    from conftest import launched_kernels
    from vecops_amd import capi
    dtype = {"bf16": torch.bfloat16, "f16": torch.float16}.get(src, torch.float32)
    if family == "tile_192" and dtype == torch.float32:
        pytest.skip("the 192 x 192 tile takes 16-bit and 8-bit operands")
    compute = capi.COMPUTE_F32 if src == "f32c" else capi.COMPUTE_BF16
    gen = torch.Generator().manual_seed(m + 7 * n + k)
    store = torch.randint(-3, 4, (m, (k + 7) // 8 * 8), generator=gen).to(dtype).to(device)
    a, values = store[:, :k], torch.randint(-3, 4, (k, n), generator=gen).to(dtype).to(device)
    b = _b_as_kn(values, -n % 8, 0)
    c = torch.full((m, n), 77.0, dtype=torch.float32, device=device)
    request = capi.family_request(family, capi.SELECT_REQUIRE, split_k=1)
    plan = capi.plan_matmul_family(a, b, c, request, compute=compute)
    assert capi.FAMILY_NAMES[plan.family] == family and plan.b_layout == 1 and plan.vector_b == 1
    kernels = launched_kernels(lambda: capi.matmul_family(a, b, c, request, compute=compute))
    if dtype != torch.float32 and family != "tile_64" and kernels[0].startswith("tile_gemm_kernel"):
        assert kernels[0].split(",")[5:7] == ["4", "5"]      # LOAD_KDMA and LOAD_NTR_DMA
    if (family, k) in (("tile_256", 648), ("tile_192", 648), ("tile_128x256", 648)) and dtype != torch.float32:
        assert kernels[0].startswith("tile_gemm_kernel")
    c.fill_(77)
    capi.matmul_family(a, b, c, request, compute=compute)
    torch.cuda.synchronize()
    assert torch.equal(c, torch.matmul(a.double(), values.double()).float())


@pytest.mark.parametrize("n", [1001, 1002, 1004, 1007, 4097])
@pytest.mark.parametrize("m,k", [(1000, 1024), (333, 4001), (17, 640)])
def test_the_librarys_own_plans(device, m, n, k):
    import torch
    from vecops_amd import capi
    for dtype, compute in ((torch.bfloat16, capi.COMPUTE_BF16), (torch.float32, capi.COMPUTE_BF16), (torch.float32, capi.COMPUTE_F32)):
        _check(device, capi, dtype, compute, m, n, k, 0, 0)


@pytest.mark.parametrize("split", [2, 5])
def test_k_splits_and_batches(device, split):
    import torch
    from vecops_amd import capi
    _check(device, capi, torch.bfloat16, capi.COMPUTE_BF16, 200, 387, 640, 1, 3, capi.family_request("tile_128", capi.SELECT_REQUIRE, split_k=split))
    _check(device, capi, torch.float16, capi.COMPUTE_BF16, 100, 131, 320, 0, 0, batch=3)


def test_grouped(device):
    import torch
    from vecops_amd import capi
    gen = torch.Generator().manual_seed(1)
    a = [torch.randint(-3, 4, (r, 320), generator=gen).bfloat16().to(device) for r in (300, 77, 200)]
    values = [torch.randint(-3, 4, (320, n), generator=gen).bfloat16().to(device) for n in (1001, 999, 1003)]
    c = [torch.empty((x.shape[0], v.shape[1]), dtype=torch.float32, device=device) for x, v in zip(a, values)]
    capi.matmul_grouped(a, [_b_as_kn(v, 1, 1) for v in values], c)
    torch.cuda.synchronize()
    for x, v, out in zip(a, values, c):
        assert torch.equal(out, x.float() @ v.float())


def test_rows_that_overlap_keep_the_general_loads(device):
    """A k stride smaller than N leaves no row behind the last one: such a view is loaded element by element."""
    import torch
    from vecops_amd import capi
    gen = torch.Generator().manual_seed(2)
    store = torch.randint(-3, 4, (64 * 10 + 33,), generator=gen).bfloat16().to(device)
    values = store.as_strided((64, 33), (10, 1))
    a = torch.randint(-3, 4, (50, 64), generator=gen).bfloat16().to(device)
    c = torch.empty((50, 33), dtype=torch.float32, device=device)
    assert capi.plan_matmul(a, values.t(), c).vector_b == 0
    capi.matmul(a, values.t(), c)
    torch.cuda.synchronize()
    assert torch.equal(c, a.float() @ values.float())
