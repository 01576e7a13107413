"""The weight-only ring kernel (w8a16_ring.hip): every count of weight rows a workgroup takes, single rows past it, K of one
stage, of part of one, of rings that wrap and of an odd multiple of 64, every group size, padded rows - and products beside the
rule's lines (K below a stage, three or four rows), which the other kernels of the family run."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,group,pad", [
    (5, 17, 64, 64, 0), (16, 16, 512, 128, 0), (7, 257, 576, 64, 16), (16, 1000, 1216, 64, 0), (9, 4096, 1024, 256, 0),     # 16 rows
    (3, 2048, 4096, 128, 0), (4, 333, 6400, 256, 32), (16, 1089, 12672, 128, 0), (15, 4097, 640, 128, 0),                     # 16 and 32
    (5, 8191, 1152, 128, 0), (12, 9408, 1088, 64, 0), (16, 12288, 2048, 128, 16), (8, 12289, 2176, 128, 0),                   # 32, 48, 64
    (14, 16384, 1024, 64, 0), (6, 16385, 1024, 128, 0), (10, 9378, 14208, 64, 0), (5, 700, 128, 128, 0),
    (9, 8193, 320, 64, 0), (6, 16383, 256, 128, 16), (7, 16385, 1152, 128, 0), (5, 8192, 448, 64, 0), (7, 20000, 64, 64, 0),   # the lines of K
    (3, 4097, 2112, 64, 0), (4, 1025, 8448, 256, 32), (3, 16385, 5120, 128, 0), (4, 1024, 8448, 64, 0)])
def test_against_float64(device, m, n, k, group, pad):
    import torch
    from vecops_amd import capi
    g = torch.Generator(device=device).manual_seed(m * n)
    x = torch.randn((m, k + pad), generator=g, device=device).bfloat16()[:, :k]
    w = torch.randint(-128, 128, (n, k + pad), generator=g, device=device, dtype=torch.int8)[:, :k]
    scales = torch.rand((n, k // group), generator=g, device=device) + 0.5
    y = torch.full((m, n + 1), float("nan"), device=device, dtype=torch.bfloat16)
    capi.matmul_w8a16_group(x, w, scales, y[:, :n], group)
    torch.cuda.synchronize()
    weights = (w.double().reshape(n, k // group, group) * scales.double()[:, :, None]).reshape(n, k)
    want = x.double() @ weights.T.contiguous()
    # one rounding to bf16 (8 significant bits, the first of them 1: at most 2^-8 of the value), and the fp32 sums': each of the K products' roundings, and those of the terms
    # +128 and -128 of a weight, at most 2^-24 of the sum of their sizes
    size = x.double().abs() @ (weights.abs() + 128.0 * scales.double().repeat_interleave(group, dim=1)).T.contiguous()
    bound = want.abs() * 2.0 ** -8 + size * (2.0 ** -24 * (k / 64 + 16)) + 1e-30
    assert bool(((y[:, :n].double() - want).abs() <= bound * 1.01).all())
    assert bool(y[:, n].isnan().all())       # nothing behind a row


def test_zeros_and_infinities_stay_in_their_rows(device):
    """A group's scale of infinity, and an activation that is not finite, reach the sums they belong to and no other."""
    import torch
    from vecops_amd import capi
    m, n, k, group = 6, 100, 640, 64
    x = torch.ones((m, k), device=device, dtype=torch.bfloat16)
    w = torch.ones((n, k), device=device, dtype=torch.int8)
    scales = torch.ones((n, k // group), device=device)
    scales[7, 3] = float("inf")
    x[2, 500] = float("nan")
    y = torch.empty((m, n), device=device, dtype=torch.bfloat16)
    capi.matmul_w8a16_group(x, w, scales, y, group)
    torch.cuda.synchronize()
    want = torch.full((m, n), float(k), device=device)
    want[:, 7] = float("inf")
    want[2] = float("nan")
    assert torch.equal(torch.nan_to_num(y.float(), nan=-1.0), torch.nan_to_num(want.bfloat16().float(), nan=-1.0))
