"""fp32 activations quantised on the way in (vecops' RuntimePerRowAsymmetricQuantizeTransform,
matmul/Quantization.h:91-146) through the C ABI: vecops_hip_quantize_rows and the one-call pipeline
vecops_hip_matmul_runtime_quant (tests/ops/MatmulConversionTestCommon.h:1437-1540), bit for bit against the
golden vectors of the real vecops build and against the oracle."""
import os

import numpy as np
import pytest

from golden_cases import (QUANT_BATCHED_CASES, QUANT_CASES, QUANT_EDGE_ZERO_POINTS, make_quant_batched_inputs,
                          make_quant_inputs, quant_batched_by_oracle, quant_edge_inputs)
from oracle import oracle as O
from vecops_amd import synth

pytestmark = pytest.mark.gpu
GOLD = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "vecops_quant_golden.npz"))


def dev(x, device):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x)).to(device)


def test_quantize_rows_edge_values_and_double_rounding(device):
    import torch
    from vecops_amd import capi
    a, _, mult = quant_edge_inputs()
    for zp in QUANT_EDGE_ZERO_POINTS:
        q = torch.full(a.shape, 99, dtype=torch.uint8, device=device)
        capi.quantize_rows(dev(a, device), dev(mult, device), zp, q)
        assert np.array_equal(q.cpu().numpy().astype(np.int32), GOLD[f"edge_zp{zp}"]), zp
    fa, fm = GOLD["fma_a"], GOLD["fma_multipliers"]
    q = torch.zeros(fa.shape, dtype=torch.uint8, device=device)
    capi.quantize_rows(dev(fa, device), dev(fm, device), -15, q)
    assert np.array_equal(q.cpu().numpy().astype(np.int32), GOLD["fma_bytes"])       # 1 everywhere; a fused rounding gives 0


@pytest.mark.parametrize("batch,m,k", [(1, 19, 69), (1, 1, 1), (3, 37, 130), (1, 300, 4096), (2, 5, 3), (3, 20, 2049)])
def test_quantize_rows_strided_and_batched(device, oracle, batch, m, k):
    """Rank 2 and 3, row strides wider than K on both sides, K not a multiple of four, a transposed source."""
    import torch
    from vecops_amd import capi
    mult = (np.float32(3.0) + synth.uniform_pm1(1, (batch * m,))).astype(np.float32)
    x = (synth.uniform_pm1(2, (batch * m, k)) * np.float32(60.0)).astype(np.float32)
    want = oracle.quantize_rows(x, mult, 100).reshape(batch, m, k)
    store = torch.full((batch, m, k + 5), float("nan"), device=device)
    store[:, :, :k] = dev(x.reshape(batch, m, k), device)
    qstore = torch.full((batch, m, k + 3), 77, dtype=torch.uint8, device=device)
    xv, qv = store[:, :, :k], qstore[:, :, :k]
    if batch == 1:
        xv, qv = xv[0], qv[0]
    capi.quantize_rows(xv, dev(mult, device), 100, qv)
    assert np.array_equal(qstore[:, :, :k].cpu().numpy(), want)
    assert (qstore[:, :, k:] == 77).all()
    if batch == 1:                                                   # source stored [K,M]
        xt = dev(np.ascontiguousarray(x.T), device).t()
        q2 = torch.zeros((m, k), dtype=torch.uint8, device=device)
        capi.quantize_rows(xt, dev(mult, device), 100, q2)
        assert np.array_equal(q2.cpu().numpy(), want[0])


@pytest.mark.parametrize("case", QUANT_CASES, ids=lambda c: c["name"])
def test_runtime_quant_pipeline_golden(device, case):
    import torch
    from vecops_amd import capi
    inp = make_quant_inputs(case)
    c = torch.full((case["m"], case["n"]), float("nan"), device=device)
    capi.matmul_runtime_quant(dev(inp["a"], device), dev(inp["multipliers"], device), case["zp"], dev(inp["b"], device),
                              dev(inp["row_scales"], device), dev(inp["column_scales"], device), c,
                              correction=dev(inp["correction"], device))
    torch.cuda.synchronize()
    assert np.array_equal(c.cpu().numpy().view(np.uint32), GOLD[case["name"] + "_f32"].view(np.uint32))


@pytest.mark.parametrize("m,n,k", [(2048, 1100, 4096), (1, 300, 512), (16, 4096, 4096), (255, 63, 8191)])
def test_runtime_quant_pipeline_against_the_oracle(device, oracle, m, n, k):
    """Tile, split-K and narrow shapes; B given [K,N]; no correction row."""
    import torch
    from vecops_amd import capi
    mult = (np.float32(2.0) + synth.uniform_pm1(1, (m,))).astype(np.float32)
    a = ((synth.uniform_pm1(2, (m, k)) * np.float32(140.0) + np.float32(120.0)) / mult[:, None]).astype(np.float32)
    b = synth.int8_sym(3, (n, k))
    rs, cs = (np.float32(1.0) / mult).astype(np.float32), synth.scales(4, n)
    q = oracle.quantize_rows(a, mult, 8)
    acc = np.zeros((m, n), np.int32)
    oracle.matmul(q, b, acc, atom=O.ATOM_I8I32, acc_f64=True, c_bf16=False)
    want = oracle.fused_outputs(acc, np.float32, row_scales=rs, column_scales=cs)
    bt = dev(np.ascontiguousarray(b.T), device).t()                  # [N,K] view of a [K,N] array
    c = torch.full((m, n), float("nan"), device=device)
    capi.matmul_runtime_quant(dev(a, device), dev(mult, device), 8, bt, dev(rs, device), dev(cs, device), c)
    torch.cuda.synchronize()
    assert np.array_equal(c.cpu().numpy().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("case", QUANT_CASES, ids=lambda c: c["name"])
def test_runtime_quant_pipeline_packed_weights_golden(device, case):
    """The reference test's own operands: B packed first, the compensated pack's sidecar as the correction row
    (tests/ops/MatmulConversionTestCommon.h:1484-1510, ops/MatmulPack.h:52-58)."""
    import torch
    from vecops_amd import capi
    inp = make_quant_inputs(case)
    packed, comp = capi.pack_b(dev(inp["b"], device), a_zero_point=case["zp"])
    assert np.array_equal(comp.cpu().numpy(), inp["correction"])
    c = torch.full((case["m"], case["n"]), float("nan"), device=device)
    capi.matmul_runtime_quant_packed_b(dev(inp["a"], device), dev(inp["multipliers"], device), case["zp"], packed,
                                       dev(inp["row_scales"], device), dev(inp["column_scales"], device), c, correction=comp)
    torch.cuda.synchronize()
    assert np.array_equal(c.cpu().numpy().view(np.uint32), GOLD[case["name"] + "_f32"].view(np.uint32))


def test_runtime_quant_batched_activations_shared_weights(device, oracle):
    """Rank-3 a and c against one b (vecops' BroadcastB case, row scales indexed batch * M + row,
    tests/ops/MatmulConversionTestCommon.h:1277-1434): the batches fold into rows."""
    import torch
    from vecops_amd import capi
    batch, m, n, k = 3, 37, 150, 300
    mult = (np.float32(2.0) + synth.uniform_pm1(1, (batch * m,))).astype(np.float32)
    a = ((synth.uniform_pm1(2, (batch * m, k)) * np.float32(140.0) + np.float32(120.0)) / mult[:, None]).astype(np.float32)
    b = synth.int8_sym(3, (n, k))
    rs, cs = (np.float32(1.0) / mult).astype(np.float32), synth.scales(4, n)
    corr = (-8 * b.astype(np.int64).sum(axis=1)).astype(np.int32)
    acc = (oracle.quantize_rows(a, mult, 8).astype(np.int64) @ b.astype(np.int64).T + corr).astype(np.int32)
    want = oracle.fused_outputs(acc, np.float32, row_scales=rs, column_scales=cs).reshape(batch, m, n)
    c = torch.full((batch, m, n), float("nan"), device=device)
    capi.matmul_runtime_quant(dev(a.reshape(batch, m, k), device), dev(mult, device), 8, dev(b, device), dev(rs, device),
                              dev(cs, device), c, correction=dev(corr, device))
    torch.cuda.synchronize()
    assert np.array_equal(c.cpu().numpy().view(np.uint32), want.view(np.uint32))
    # rows that do not run on from batch to batch in a: quantised from where they are, the product still folds
    gapped = torch.zeros((batch, m + 1, k), device=device)
    gapped[:, :m] = dev(a.reshape(batch, m, k), device)
    c.fill_(float("nan"))
    capi.matmul_runtime_quant(gapped[:, :m], dev(mult, device), 8, dev(b, device), dev(rs, device), dev(cs, device), c,
                              correction=dev(corr, device))
    # ... and in c: batch by batch
    cg = torch.full((batch, m + 2, n), float("nan"), device=device)
    capi.matmul_runtime_quant(gapped[:, :m], dev(mult, device), 8, dev(b, device), dev(rs, device), dev(cs, device), cg[:, :m],
                              correction=dev(corr, device))
    torch.cuda.synchronize()
    assert np.array_equal(c.cpu().numpy().view(np.uint32), want.view(np.uint32))
    assert np.array_equal(cg[:, :m].cpu().numpy().view(np.uint32), want.view(np.uint32))
    assert torch.isnan(cg[:, m:]).all()


@pytest.mark.parametrize("case", QUANT_BATCHED_CASES, ids=[c["name"] for c in QUANT_BATCHED_CASES])
def test_runtime_quant_batched_golden(device, case):
    """Shared or per-batch activations and weights (tests/ops/MatmulConversionTestCommon.h:1277-1434; a batch stride of
    0 shares an operand): bit for bit against the outputs of the real vecops build."""
    import torch
    from vecops_amd import capi
    inp = make_quant_batched_inputs(case)
    batch, m, n, k = case["batch"], case["m"], case["n"], case["k"]
    a = dev(inp["a"], device).expand(batch, m, k)                   # a leading extent of 1 becomes batch stride 0
    b = dev(inp["b"], device).expand(batch, n, k)
    c = torch.full((batch, m, n), float("nan"), device=device)
    capi.matmul_runtime_quant(a, dev(inp["multipliers"], device), inp["zero_point"], b, dev(inp["row_scales"], device),
                              dev(inp["column_scales"], device), c, correction=dev(inp["correction"], device))
    torch.cuda.synchronize()
    assert np.array_equal(c.cpu().numpy().view(np.uint32), GOLD[case["name"] + "_f32"].view(np.uint32))


@pytest.mark.parametrize("batch,m,n,k,shared_a,shared_b", [(4, 300, 520, 1030, False, False), (5, 64, 1000, 4096, True, False),
                                                           (3, 7, 2048, 512, False, False), (6, 130, 130, 129, False, True)])
def test_runtime_quant_batched_against_the_oracle(device, oracle, batch, m, n, k, shared_a, shared_b):
    """Bigger batched shapes (several tiles per batch, a skinny M, K with a tail), operands with gaps between rows and
    batches, and the explicit batch strides of vecops_hip_matmul_runtime_quant_batched - among them one set of scales
    for per-batch activations (stride 0), which the conventional entry cannot say."""
    import torch
    from vecops_amd import capi
    case = {"kind": "seeded", "batch": batch, "m": m, "n": n, "k": k, "shared_a": shared_a, "shared_b": shared_b}
    inp = make_quant_batched_inputs(case)
    want = quant_batched_by_oracle(oracle, inp, batch)
    ab, bb = inp["a"].shape[0], inp["b"].shape[0]
    a_store = torch.full((ab, m + 1, k + 4), float("nan"), device=device)
    a_store[:, :m, :k] = dev(inp["a"], device)
    b_store = torch.full((bb, n + 2, k + 16), 99, dtype=torch.int8, device=device)
    b_store[:, :n, :k] = dev(inp["b"], device)
    a, b = a_store[:, :m, :k].expand(batch, m, k), b_store[:, :n, :k].expand(batch, n, k)
    c_store = torch.full((batch, m + 3, n + 4), float("nan"), device=device)
    c = c_store[:, :m, :n]
    mult, rs, cs = dev(inp["multipliers"], device), dev(inp["row_scales"], device), dev(inp["column_scales"], device)
    corr = dev(inp["correction"], device)
    capi.matmul_runtime_quant(a, mult, inp["zero_point"], b, rs, cs, c, correction=corr)
    torch.cuda.synchronize()
    assert np.array_equal(c.cpu().numpy().view(np.uint32), want.view(np.uint32))
    assert torch.isnan(c_store[:, m:]).all() and torch.isnan(c_store[:, :, n:]).all()
    # the same through the explicit strides
    c_store.fill_(float("nan"))
    capi.matmul_runtime_quant_batched(a, mult, inp["zero_point"], 0 if shared_a else m, b, rs, cs, c, correction=corr,
                                      correction_batch_stride=0 if shared_b else n)
    torch.cuda.synchronize()
    assert np.array_equal(c.cpu().numpy().view(np.uint32), want.view(np.uint32))
    if not shared_a:
        # per-batch activations under ONE set of multipliers / scales (those of batch 0) and one correction row
        inp0 = dict(inp, multipliers=np.tile(inp["multipliers"][:m], batch), row_scales=np.tile(inp["row_scales"][:m], batch),
                    correction=np.tile(inp["correction"][:n], bb))
        want0 = quant_batched_by_oracle(oracle, inp0, batch)
        c_store.fill_(float("nan"))
        capi.matmul_runtime_quant_batched(a, mult, inp["zero_point"], 0, b, rs, cs, c, correction=corr, correction_batch_stride=0)
        torch.cuda.synchronize()
        assert np.array_equal(c.cpu().numpy().view(np.uint32), want0.view(np.uint32))


def test_runtime_quant_zero_extents_and_rejections(device):
    import torch
    from vecops_amd import capi
    one = torch.ones(4, device=device)
    c = torch.full((4, 6), float("nan"), device=device)
    corr = torch.arange(6, dtype=torch.int32, device=device)
    capi.matmul_runtime_quant(torch.empty((4, 0), device=device), one, 3, torch.empty((6, 0), dtype=torch.int8, device=device),
                              one, torch.ones(6, device=device), c, correction=corr)
    torch.cuda.synchronize()
    assert torch.equal(c, corr.float().expand(4, 6))                  # K == 0: the correction row, dequantised
    capi.matmul_runtime_quant(torch.empty((0, 8), device=device), one, 3, torch.zeros((6, 8), dtype=torch.int8, device=device),
                              one, torch.ones(6, device=device), torch.empty((0, 6), device=device))
    with pytest.raises(capi.VecopsHipError) as e:                     # bf16 activations are not this entry's business
        capi.matmul_runtime_quant(torch.zeros((4, 8), dtype=torch.bfloat16, device=device), one, 3,
                                  torch.zeros((6, 8), dtype=torch.int8, device=device), one, torch.ones(6, device=device), c)
    assert e.value.code == 2
    with pytest.raises(capi.VecopsHipError) as e:
        capi.quantize_rows(torch.zeros((4, 8), device=device), one, 3, torch.zeros((4, 9), dtype=torch.uint8, device=device))
    assert e.value.code == 1


@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (3, 7, 15), (17, 33, 127), (24, 250, 129), (5, 40, 2047), (300, 257, 2049),
                                   (130, 64, 4100), (70, 128, 1024), (70, 128, 1025), (70, 129, 1000), (65, 9, 72)])
def test_runtime_quant_packed_edges_equal_the_unpacked_call(device, m, n, k):
    """Packed weights at the edges of the quantisation's 2048-element pieces, of the K padding of the quantised rows (none where N is narrow and K short) and
    of the row sums' eight-row workgroups, in a workspace full of garbage: the unpacked call's bits (integer sums)."""
    import torch
    from vecops_amd import capi
    a = dev((synth.uniform_pm1(1, (m, k)) * np.float32(60.0)).astype(np.float32), device)
    b = dev(synth.int8_sym(2, (n, k)), device)
    mult = dev((np.float32(3.0) + synth.uniform_pm1(3, (m,))).astype(np.float32), device)
    rs, cs = dev(synth.scales(4, m), device), dev(synth.scales(5, n), device)
    packed, corr = capi.pack_b(b, a_zero_point=128)
    sums = b.cpu().numpy().astype(np.int64).sum(axis=1)
    assert np.array_equal(corr.cpu().numpy(), (-128 * sums).astype(np.int32))
    q = torch.empty((m, k), dtype=torch.uint8, device=device)
    capi.quantize_rows(a, mult, 128, q)
    acc = q.cpu().numpy().astype(np.int64) @ b.cpu().numpy().astype(np.int64).T - 128 * sums
    want = (acc.astype(np.int32).astype(np.float32) * rs.cpu().numpy()[:, None]) * cs.cpu().numpy()[None, :]
    ws = torch.full((1 << 24,), 0xA5, dtype=torch.uint8, device=device)
    for packed_call in (True, False):
        c = torch.full((m, n), float("nan"), device=device)
        call, weights = (capi.matmul_runtime_quant_packed_b, packed) if packed_call else (capi.matmul_runtime_quant, b)
        call(a, mult, 128, weights, rs, cs, c, correction=corr, workspace=ws)
        torch.cuda.synchronize()
        assert np.array_equal(c.cpu().numpy().view(np.uint32), want.view(np.uint32)), packed_call


def _quantized(a, mult, zero_point):
    """The same multiply, add and truncation element by element (values far from the ends of int32)."""
    import torch
    return (a * mult[:, None] + float(zero_point)).to(torch.int32).clamp(0, 255).to(torch.uint8)


@pytest.mark.parametrize("m,k", [((1 << 24) + 3, 5), (70001, 1030), (33001, 2049)])
def test_quantize_more_rows_than_workgroups(device, m, k):
    """Contiguous rows by the million: a workgroup each would be more than a launch takes, so the workgroups stride over
    them; and several ten thousand pieces, a workgroup each."""
    import torch
    from vecops_amd import capi
    a = torch.randn((m, k), generator=torch.Generator(device).manual_seed(1), device=device)
    mult = torch.linspace(20.0, 60.0, m, device=device)
    q = torch.full((m, k), 99, dtype=torch.uint8, device=device)
    capi.quantize_rows(a, mult, 100, q)
    assert torch.equal(q, _quantized(a, mult, 100))


@pytest.mark.parametrize("packed", [False, True])
def test_runtime_quant_more_rows_than_a_launch_has_workgroups(device, packed):
    import torch
    from vecops_amd import capi
    m, n, k = (1 << 24) + 3, 9, 16
    gen = torch.Generator(device).manual_seed(2)
    a = torch.randn((m, k), generator=gen, device=device)
    b = torch.randint(-127, 128, (n, k), generator=gen, device=device, dtype=torch.int8)
    mult, rs, cs = torch.linspace(20.0, 60.0, m, device=device), torch.linspace(0.5, 2.0, m, device=device), torch.rand(n, device=device)
    c = torch.full((m, n), float("nan"), device=device)
    if packed:
        capi.matmul_runtime_quant_packed_b(a, mult, 100, capi.pack_b(b), rs, cs, c)
    else:
        capi.matmul_runtime_quant(a, mult, 100, b, rs, cs, c)
    # sixteen products of at most 255 * 127: every partial sum is a whole number that fp32 holds
    want = (_quantized(a, mult, 100).float() @ b.float().t()) * rs[:, None] * cs[None, :]
    assert torch.equal(c, want)


@pytest.mark.parametrize("m,k", [(1, 1), (3, 5), (65, 130), (300, 2049), (64, 1024)])
@pytest.mark.parametrize("x_contiguous,q_contiguous", [(True, False), (False, True), (False, False)])
def test_quantize_rows_contiguous_on_one_side(device, x_contiguous, q_contiguous, m, k):
    """One side stored [M,K] with rows at odd addresses, the other [K,M]: a quad is taken whole where its side allows it,
    and nothing outside the rows is written."""
    import torch
    from vecops_amd import capi
    x = torch.randn((m, k), generator=torch.Generator(device).manual_seed(3), device=device)
    mult = torch.linspace(20.0, 60.0, m, device=device)

    def stored(contiguous, fill, dtype):
        store = torch.full((m, k + 3) if contiguous else (k, m + 3), fill, dtype=dtype, device=device)
        return store, store[:, 1:k + 1] if contiguous else store[:, 1:m + 1].t()

    _, xv = stored(x_contiguous, float("nan"), torch.float32)
    xv.copy_(x)
    qstore, qv = stored(q_contiguous, 77, torch.uint8)
    capi.quantize_rows(xv, mult, 100, qv)
    assert torch.equal(qv, _quantized(x, mult, 100))
    assert (qstore[:, 0] == 77).all() and (qstore[:, -2:] == 77).all()


@pytest.mark.parametrize("n,k", [(65504, 33), (65505, 1), (65505, 200), (65536, 128), (65545, 512), (65545, 513), (100000, 500)])
def test_packed_row_sums_of_many_panels(device, n, k):
    """Weights of about 2048 panels of 32 rows, where the sums of short rows change from a workgroup for eight rows to a wavefront a
    panel: as the correction of unsigned activations and of runtime-quantised ones.  (Up to 513 products of at most
    255 * 127: every partial sum is a whole number that fp32 holds.)"""
    import torch
    from vecops_amd import capi
    gen = torch.Generator(device).manual_seed(4)
    m = 17
    b = torch.randint(-127, 128, (n, k), generator=gen, device=device, dtype=torch.int8)
    packed, corr = capi.pack_b(b, a_zero_point=100)
    a8 = torch.randint(0, 256, (m, k), generator=gen, device=device, dtype=torch.uint8)
    c = torch.full((m, n), -7, dtype=torch.int32, device=device)
    capi.matmul_packed_b(a8, packed, c)
    assert torch.equal(c, (a8.float() @ b.float().t()).to(torch.int32))
    a = torch.randn((m, k), generator=gen, device=device)
    mult, rs, cs = torch.linspace(20.0, 60.0, m, device=device), torch.linspace(0.5, 2.0, m, device=device), torch.rand(n, device=device)
    out = torch.full((m, n), float("nan"), device=device)
    capi.matmul_runtime_quant_packed_b(a, mult, 100, packed, rs, cs, out, correction=corr)
    want = ((_quantized(a, mult, 100).float() - 100.0) @ b.float().t()) * rs[:, None] * cs[None, :]
    assert torch.equal(out, want)
