"""Extents that line up with nothing: K-contiguous rows at any alignment on the 128x256 tile."""
import numpy as np
import pytest

from conftest import rel_err
from test_matmul_gpu import fp32_tol

pytestmark = pytest.mark.gpu


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
