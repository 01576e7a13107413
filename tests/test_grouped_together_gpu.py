"""Grouped calls in one launch: groups in the product's own kernel arguments (up to twenty-four; more through the table), groups
that split K on their own together on slim tiles, or with all others on one tile.  Operands are small integers: sums are exact,
whatever their order, and compared bit for bit."""
import pytest

pytestmark = pytest.mark.gpu


def _run(device, shapes, kind="bf16", out="f32", cin=False, offset=0):
    import torch
    from vecops_amd import capi
    dtype = {"bf16": torch.bfloat16, "f16": torch.float16, "i8": torch.int8}[kind]
    result = torch.int32 if kind == "i8" else {"f32": torch.float32}.get(out, dtype)
    gen = torch.Generator().manual_seed(len(shapes))
    a, b, c, ci, want = [], [], [], [], []
    for i, shape in enumerate(shapes):
        *lead, m, n, k = shape
        x = torch.randint(-3, 4, (*lead, m, k), generator=gen).to(dtype)
        y = torch.randint(-3, 4, (*lead, n, k), generator=gen).to(dtype)
        sums = x.double() @ y.double().transpose(-1, -2)
        z = torch.randint(-9, 10, (*lead, m, n), generator=gen).to(result) if cin and i % 2 else None
        want.append((sums + (z.double() if z is not None else 0)).float().to(result))
        store = torch.zeros(x.numel() + offset, dtype=dtype, device=device)   # (rows at any alignment)
        a.append(store[offset:].view(x.shape))
        a[-1].copy_(x)
        b.append(y.to(device))
        c.append(torch.full((*lead, m, n), 77, dtype=result, device=device))
        ci.append(z.to(device) if z is not None else None)
    capi.matmul_grouped(a, b, c, c_in_list=ci)
    torch.cuda.synchronize()
    for i, shape in enumerate(shapes):
        assert torch.equal(c[i].cpu(), want[i]), (i, shape)
    Operands = capi.Operand * len(shapes)
    return capi.lib().vecops_hip_matmul_grouped_workspace(len(shapes), *(Operands(*map(capi.operand, t)) for t in (a, b)), None,
                                                          Operands(*map(capi.operand, c)), 0)


@pytest.mark.parametrize("count,table", [(2, False), (3, False), (12, False), (13, False), (23, False), (24, False), (25, True), (49, True)])
@pytest.mark.parametrize("kind,out", [("bf16", "f32"), ("f16", "f16"), ("i8", "i32")])
def test_groups_in_the_launchs_arguments(device, count, table, kind, out):
    """K of up to seven K tiles: no group splits it; the first and the last group end where the argument's room does."""
    need = _run(device, [(1 + 17 * i % 300, 20 + 13 * i % 400, 64 + 8 * (i % 40)) for i in range(count)], kind, out, cin=True)
    assert (need > 256) == table


# rows per group, N, K: a row alone and sixteen (the skinny family's) among others, rows at any alignment, K ragged
@pytest.mark.parametrize("rows,n,k", [([42, 7, 100, 33, 16, 1, 64, 30], 409, 1985), ([33, 40, 20, 5, 1, 16, 60, 17, 33, 30, 29, 31], 896, 2048),
                                      ([22, 30, 19, 3], 768, 8183), ([183, 150, 200, 170, 129], 640, 3080), ([300, 1], 70, 8192)])
@pytest.mark.parametrize("kind,out,cin,offset", [("bf16", "bf16", False, 0), ("bf16", "f32", True, 0), ("f16", "f16", True, 1), ("i8", "i32", True, 3)])
def test_groups_that_split_k_on_their_own(device, rows, n, k, kind, out, cin, offset):
    _run(device, [(m, n, k) for m in rows], kind, out, cin, offset)


def test_more_of_them_than_one_launch_carries(device):
    assert _run(device, [(20 + i % 9, 250 + i, 6000) for i in range(53)]) == 256


def test_all_groups_on_one_tile(device):
    """Few and long: one launch on 128x128 tiles takes less than two launches for each."""
    assert _run(device, [(150 + 10 * i, 1890, 6144) for i in range(12)], "f16", "f16") == 256


def test_among_others(device):
    """Beside groups in whole tiles, one with no rows, one with K = 0 and one of two batches."""
    _run(device, [(42, 409, 1985)] * 9 + [(700, 900, 264), (0, 64, 32), (64, 100, 0), (2, 37, 300, 1200), (1000, 1300, 264), (42, 409, 1985)])
    _run(device, [(42, 409, 1985)] * 9 + [(700, 900, 264)])


def test_repeated_and_captured(device):
    import torch
    from vecops_amd import capi
    gen = torch.Generator().manual_seed(1)
    a = [torch.randint(-3, 4, (m, 1984), generator=gen).bfloat16().to(device) for m in (42, 7, 100, 33, 16, 1, 64, 30)]
    b = [torch.randint(-3, 4, (409, 1984), generator=gen).bfloat16().to(device) for _ in a]
    c = [torch.empty((x.shape[0], 409), device=device) for x in a]
    want = [x.float() @ y.float().t() for x, y in zip(a, b)]
    workspace = torch.empty(1 << 20, dtype=torch.uint8, device=device)
    run = lambda: capi.matmul_grouped(a, b, c, workspace=workspace)
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run()
    for _ in range(4):
        for t in c:
            t.fill_(77.0)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(c, want))


SRC = {"bf16": 0, "f16": 5, "i8": 2}


def _kernels_and_values(device, shapes, kind):
    """(m, n, k, layout of b) of each group: the kernels of the call; its values checked."""
    import torch
    from conftest import launched_kernels
    from vecops_amd import capi
    dtype = {"bf16": torch.bfloat16, "f16": torch.float16, "i8": torch.int8}[kind]
    gen = torch.Generator().manual_seed(len(shapes))
    a, b, c = [], [], []
    for m, n, k, layout in shapes:
        a.append(torch.randint(-3, 4, (m, k), generator=gen).to(dtype).to(device))
        y = torch.randint(-3, 4, (n, k), generator=gen).to(dtype).to(device)
        b.append(y if layout == "nk" else y.t().contiguous().t())
        c.append(torch.empty((m, n), dtype=torch.int32 if kind == "i8" else torch.float32, device=device))
    names = launched_kernels(lambda: capi.matmul_grouped(a, b, c))
    for t in c:
        t.fill_(77)
    capi.matmul_grouped(a, b, c)
    torch.cuda.synchronize()
    for x, y, out in zip(a, b, c):
        assert torch.equal(out, (x.double() @ y.t().contiguous().double()).to(out.dtype))
    return names


@pytest.mark.parametrize("tile,rows,n,k", [((32, 32), [22, 30, 19, 3], 768, 8183), ((32, 64), [60, 59, 60, 57, 60, 60, 58, 60], 700, 4096),
                                           ((64, 64), [128, 127, 126, 128, 120, 128, 128, 125, 128], 700, 4090), ((64, 64), [120, 119] * 6, 600, 4096),
                                           ((128, 64), [128, 127] * 6, 1000, 4096)])
@pytest.mark.parametrize("kind", ["bf16", "f16", "i8"])
def test_each_slim_tile(device, kind, tile, rows, n, k):
    names = _kernels_and_values(device, [(m, n, k, "nk") for m in rows], kind)
    assert names == [f"tile_gemm_slim_grouped_kernel<{SRC[kind]},{tile[0]},{tile[1]}>"]


# groups with B as [K,N] beside long K-contiguous ones: they would turn the loads of a launch together into element loads
# (tile_gemm_grouped_kernel<..., 1, 1, ...>)
LONG = [(150 + 10 * i, 1890, 6144, "nk") for i in range(12)]


@pytest.mark.parametrize("shapes,together,others", [
    ([(256, 2048, 8192, "nk")] * 8 + [(64, 256, 256, "kn")], "tile_gemm_grouped_kernel<5,2,2,2,2,4,4,", "tile_gemm_kernel<5,2,2,1,1,0,3,"),
    (LONG + [(300, 700, 264, "kn")], "tile_gemm_grouped_kernel<5,2,2,2,2,4,4,", "tile_gemm_kernel<5,2,2,1,1,0,3,"),
    ([(42, 409, 1985, "nk")] * 18 + [(64, 256, 256, "kn")] * 2, "tile_gemm_slim_grouped_kernel<5,32,64>", "tile_gemm_grouped_kernel<5,2,2,1,1,0,3,"),
    (LONG + [(700, 900, 264, "kn")] * 14, "tile_gemm_slim_grouped_kernel<5,128,64>", "tile_gemm_grouped_kernel<5,2,2,4,4,0,3,")])
def test_other_layouts_stay_apart(device, shapes, together, others):
    names = _kernels_and_values(device, shapes, "f16")
    assert len(names) == 2 and sorted(name.startswith(together) for name in names) == [False, True]
    assert sorted(name.startswith(others) for name in names) == [False, True]


def test_an_unaligned_group_among_aligned_ones(device):
    names = _kernels_and_values(device, LONG + [(700, 904, 264, "nk")] * 6 + [(300, 640, 333, "nk")], "f16")
    assert len(names) == 1 and names[0].startswith("tile_gemm_grouped_kernel<5,2,2,2,2,0,0,")
