"""Extents that line up with nothing: K-contiguous rows at any alignment on the 128x256 tile."""
import numpy as np
import pytest

from conftest import rel_err
from test_matmul_gpu import fp32_tol

pytestmark = pytest.mark.gpu
ROWS_I8 = (515, 6766, 1027)      # int8 products that the library itself puts on the 128x256 tile with rows at any alignment


def _operands(device, dtype, m, n, k, seed=1, batch=()):
    import torch
    g = torch.Generator(device=device).manual_seed(seed)
    make = lambda *shape: torch.randn(shape, generator=g, device=device).to(dtype)  # noqa: E731
    return make(*batch, m, k), make(*batch, n, k)


def _exact(a, b):
    return np.matmul(a.double().cpu().numpy(), b.double().cpu().numpy().swapaxes(-1, -2))


@pytest.mark.parametrize("batch,m,n,k,split", [(1, 128, 256, 65, 1), (2, 130, 300, 129, 1), (1, 5, 9, 1001, 1), (3, 257, 513, 301, 1),
                                               (1, 300, 520, 63, 1), (1, 64, 64, 7, 1), (1, 129, 257, 4099, 5), (8, 777, 1000, 3001, 1)])
@pytest.mark.parametrize("kind", ["bf16", "f16", "i8"])
def test_rows_kernel(device, kind, batch, m, n, k, split):
    """Bit for bit what the 256x128 tile's kernel gives: the same instructions in the same order along K."""
    import torch
    from vecops_amd import capi
    shape = (batch,) if batch > 1 else ()
    if kind == "i8":
        g = torch.Generator(device=device).manual_seed(5)
        a, b = (torch.randint(-128, 128, (*shape, r, k), generator=g, device=device, dtype=torch.int8) for r in (m, n))
    else:
        a, b = _operands(device, torch.bfloat16 if kind == "bf16" else torch.float16, m, n, k, batch=shape)
    out = torch.int32 if kind == "i8" else torch.float32
    c, other = (torch.full((*shape, m, n), 7, dtype=out, device=device) for _ in range(2))
    capi.matmul_family(a, b, c, capi.family_request("tile_128x256", split_k=split))
    capi.matmul_family(a, b, other, capi.family_request("tile_256x128", split_k=split))
    torch.cuda.synchronize()
    assert torch.equal(c, other)
    if kind != "i8":
        assert rel_err(c.cpu().numpy(), _exact(a, b)) <= fp32_tol(max(k, 32))


@pytest.mark.parametrize("batch,m,n,k", [(1, 130, 300, 129), (2, 257, 513, 301), (1, 128, 256, 65)])
@pytest.mark.parametrize("kind", ["bf16", "f16", "i8"])
def test_rows_kernel_c_inputs_and_16_bit_results(device, kind, batch, m, n, k):
    """C inputs, 16-bit results and strided C on the 128x256 tile: what its plain sums give."""
    import torch
    from vecops_amd import capi
    dtype = {"bf16": torch.bfloat16, "f16": torch.float16, "i8": torch.int8}[kind]
    shape = (batch,) if batch > 1 else ()
    g = torch.Generator(device=device).manual_seed(9)
    if kind == "i8":
        a, b = (torch.randint(-128, 128, (*shape, r, k), generator=g, device=device, dtype=torch.int8) for r in (m, n))
        out, cin = torch.int32, torch.randint(-2 ** 31, 2 ** 31 - 1, (*shape, m, n), generator=g, device=device, dtype=torch.int32)
    else:
        a, b = _operands(device, dtype, m, n, k, batch=shape)
        out, cin = dtype, torch.randn((*shape, m, n), generator=g, device=device).to(dtype)
    request = capi.family_request("tile_128x256", split_k=1)
    sums = capi.matmul_family(a, b, torch.empty((*shape, m, n), dtype=torch.int32 if kind == "i8" else torch.float32, device=device), request)
    plus = sums + (cin if kind == "i8" else cin.float())
    empty = lambda *s: torch.full(s, 7, dtype=out, device=device)  # noqa: E731
    assert torch.equal(capi.matmul_family(a, b, empty(*shape, m, n), request), sums.to(out))
    assert torch.equal(capi.matmul_family(a, b, empty(*shape, m, n), request, c_in=cin), plus.to(out))
    bias = cin[..., :1, :].expand(*shape, m, n)
    assert torch.equal(capi.matmul_family(a, b, empty(*shape, m, n), request, c_in=bias),
                       (sums + (bias if kind == "i8" else bias.float())).to(out))
    for c in (empty(*shape, n, m).transpose(-1, -2), empty(*shape, m, n + 5)[..., :n], empty(*shape, m, 2 * n)[..., ::2]):
        assert torch.equal(capi.matmul_family(a, b, c, request, c_in=cin), plus.to(out))


@pytest.mark.parametrize("activation", ["none", "relu"])
def test_rows_kernel_transforms(device, activation):
    import torch
    from vecops_amd import capi
    m, n, k = 772, 4815, 257
    a, b = _operands(device, torch.bfloat16, m, n, k)
    sums = torch.empty((m, n), device=device)
    columns = torch.rand(n, device=device) + 0.5
    ep = capi.epilogue(activation=activation, column_scales=columns, scale=0.5, shift=0.25)
    assert capi.FAMILY_NAMES[capi.plan_matmul(a, b, sums).family] == "tile_128x256"
    capi.matmul(a, b, sums)
    bias = torch.randn((1, n), device=device).expand(m, n)
    for ci in (None, bias):
        c = torch.full((m, n), float("nan"), device=device)
        assert capi.FAMILY_NAMES[capi.plan_matmul_fused(a, b, c, ep, c_in=ci).family] == "tile_128x256"
        v = ((sums if ci is None else sums + ci) * columns) * 0.5 + 0.25
        assert torch.equal(capi.matmul_fused(a, b, c, ep, c_in=ci), torch.relu(v) if activation == "relu" else v)


def test_rows_kernel_dequantised(device):
    import torch
    from vecops_amd import capi
    m, n, k = ROWS_I8
    g = torch.Generator(device=device).manual_seed(5)
    a, b = (torch.randint(-128, 128, (r, k), generator=g, device=device, dtype=torch.int8) for r in (m, n))
    sums = torch.empty((m, n), dtype=torch.int32, device=device)
    assert capi.FAMILY_NAMES[capi.plan_matmul(a, b, sums).family] == "tile_128x256"
    capi.matmul_family(a, b, sums, capi.family_request("tile_256x128", split_k=1))
    rows, columns = torch.rand(m, device=device) + 0.5, torch.rand(n, device=device) + 0.5
    correction = torch.randint(-1000, 1000, (n,), device=device, dtype=torch.int32)
    c = torch.empty((m, n), device=device)
    assert torch.equal(capi.matmul_i8_dequant(a, b, rows, columns, c), (sums.float() * rows[:, None]) * columns)
    assert torch.equal(capi.matmul_i8_dequant(a, b, rows, columns, c, correction=correction),
                       ((sums + correction).float() * rows[:, None]) * columns)
