"""The slim tiles (tile_gemm_slim.hip): what the library runs in place of the rule table's own 64x64 or 128x128 tiles where
few of them, or many K tiles for each, leave the chip waiting.  Each tile at the edges of its rows, columns and K - single
elements past a tile, K shorter than a chunk, one K tile, a partial tile behind any number of whole ones, rings that wrap -
with rows at any alignment, C inputs, output types, scales and transforms.  Results alone do not tell which kernel ran:
test_slim_plan_cpu.py pins the tile of every entry of SHAPES, the tests below that need one ask the plan for it, and those
that set `slim_tile` themselves run what they name."""
import numpy as np
import pytest

from conftest import rel_err
from test_matmul_gpu import fp32_tol

pytestmark = pytest.mark.gpu

# (m, n, k): by the estimates of take_slim_tile (capi.hip), with the tile each takes
SHAPES = {
    "32x16": [(17, 350, 960), (1, 21, 205), (33, 257, 1913), (1, 49, 447), (2, 20, 319), (20, 16, 520), (1, 37, 384)],
    "32x32": [(64, 4096, 1024), (2, 6689, 454), (1, 5035, 385), (33, 2672, 448), (97, 1999, 2048)],
    "32x48": [(33, 4285, 640), (32, 9231, 1216), (17, 11007, 1501), (1, 11713, 705)],
    "32x64": [(31, 14336, 640), (17, 12743, 512), (2, 14529, 769)],
    "64x48": [(33, 8209, 2560), (65, 5678, 1536), (129, 3338, 1344), (33, 8880, 2049), (100, 4224, 4672)],
    "64x64": [(127, 8001, 1023), (64, 14336, 768), (65, 7553, 1472), (65, 7754, 1217)],
    "128x48": [(128, 11008, 4096), (149, 6050, 640), (68, 12193, 512)],
    "128x64": [(128, 14336, 2048), (196, 7813, 904), (195, 8117, 961), (65, 16255, 1023)],
    # beside them, where the table's own tiles are ahead
    "none": [(129, 6083, 512), (65, 11787, 641), (513, 2401, 960), (129, 8170, 239), (257, 5377, 190), (65, 13433, 512)],
}
ALL = [s for shapes in SHAPES.values() for s in shapes]
TILES = [(32, 16), (32, 32), (32, 48), (32, 64), (64, 48), (64, 64), (128, 48), (128, 64)]


def _operands(device, dtype, m, n, k, seed=1, batch=(), pad=0):
    import torch
    g = torch.Generator(device=device).manual_seed(seed)
    if dtype == torch.int8:
        make = lambda shape: torch.randint(-128, 128, shape, generator=g, device=device, dtype=torch.int8)  # noqa: E731
    else:
        make = lambda shape: torch.randn(shape, generator=g, device=device).to(dtype)  # noqa: E731
    return make((*batch, m, k + pad))[..., :k], make((*batch, n, k + pad))[..., :k]


def _exact(a, b):
    """The products of the operands as they are, in float64 (int8: exact below 2^53)."""
    return np.matmul(a.double().cpu().numpy(), b.double().cpu().numpy().swapaxes(-1, -2))


@pytest.mark.parametrize("m,n,k", ALL)
@pytest.mark.parametrize("kind", ["bf16", "f16"])
def test_against_float64(device, kind, m, n, k):
    import torch
    from vecops_amd import capi
    dtype = torch.bfloat16 if kind == "bf16" else torch.float16
    a, b = _operands(device, dtype, m, n, k)
    c = torch.full((m, n), float("nan"), device=device)
    capi.matmul(a, b, c)
    prepared = torch.full((m, n), float("nan"), device=device)
    capi.PreparedMatmul(a, b, prepared)()
    rounded = torch.full((m, n), float("nan"), device=device, dtype=dtype)
    capi.matmul(a, b, rounded)
    torch.cuda.synchronize()
    assert rel_err(c.cpu().numpy(), _exact(a, b)) <= fp32_tol(k)
    assert torch.equal(c, prepared)
    assert torch.equal(c.to(dtype), rounded)     # one rounding of the same sums


@pytest.mark.parametrize("m,n,k,pad", [(17, 350, 960, 0), (33, 257, 1913, 0), (31, 300, 513, 2), (64, 2072, 1912, 8), (129, 999, 1000, 1),
                                       (100, 700, 4099, 0), (128, 11008, 1024, 0), (40, 640, 447, 0)])
def test_int8_exact(device, m, n, k, pad):
    """Exact sums, rows at every byte alignment; and dequantised, two roundings a value, with a correction row."""
    import torch
    from vecops_amd import capi
    a, b = _operands(device, torch.int8, m, n, k, pad=pad)
    c = torch.full((m, n), -1, dtype=torch.int32, device=device)
    capi.matmul(a, b, c)
    rows, columns = torch.rand(m, device=device) + 0.5, torch.rand(n, device=device) + 0.5
    correction = torch.randint(-1000, 1000, (n,), device=device, dtype=torch.int32)
    f = torch.full((m, n), float("nan"), device=device)
    capi.matmul_i8_dequant(a, b, rows, columns, f, correction=correction)
    torch.cuda.synchronize()
    want = torch.from_numpy(_exact(a, b).astype(np.int64)).to(torch.int32).to(device)
    assert torch.equal(c, want)
    assert torch.equal(f, ((want + correction).float() * rows[:, None]) * columns)


@pytest.mark.parametrize("m,n,k", [(17, 350, 960), (129, 4225, 1025), (127, 801, 1023), (128, 4800, 1920)])
@pytest.mark.parametrize("form", ["full", "bias", "strided", "transform", "transposed", "padded"])
def test_epilogues(device, m, n, k, form):
    """A C input's forms, the fused transform, C with strides that take the general store: all add to, or are made from, the
    same sums, so the plain product's fp32 result gives the expected bits."""
    import torch
    from vecops_amd import capi
    a, b = _operands(device, torch.bfloat16, m, n, k)
    sums = torch.empty((m, n), device=device)
    capi.matmul(a, b, sums)
    g = torch.Generator(device=device).manual_seed(7)
    cin = torch.randn((m, n), generator=g, device=device).bfloat16()
    c = torch.full((m, n), float("nan"), device=device, dtype=torch.bfloat16)
    if form == "bias":
        cin = cin[:1].expand(m, n)
    elif form == "strided":
        wide = torch.randn((m, 2 * n), generator=g, device=device).bfloat16()
        cin = wide[:, ::2]
    elif form == "transposed":
        c = torch.full((n, m), float("nan"), device=device, dtype=torch.bfloat16).t()
    elif form == "padded":
        c = torch.full((m, n + 3), float("nan"), device=device, dtype=torch.bfloat16)[:, :n]
    if form == "transform":
        scales = torch.rand(n, generator=g, device=device) + 0.5
        capi.matmul_fused(a, b, c, capi.epilogue(activation="relu", column_scales=scales, scale=0.5, shift=0.25), c_in=cin)
        want = torch.relu(((sums + cin.float()) * scales) * 0.5 + 0.25)
    else:
        capi.matmul(a, b, c, c_in=cin)
        want = sums + cin.float()
    torch.cuda.synchronize()
    assert torch.equal(c, want.bfloat16())


def test_batches(device):
    import torch
    from vecops_amd import capi
    a, b = _operands(device, torch.float16, 33, 260, 1000, batch=(5,))
    c = torch.full((5, 33, 260), float("nan"), device=device)
    capi.matmul(a, b, c)
    torch.cuda.synchronize()
    assert rel_err(c.cpu().numpy(), _exact(a, b)) <= fp32_tol(1000)


def test_whose_plan_it_is(device):
    """The table's own plan runs on a slim tile wherever it comes from; a required family and split run as named."""
    import torch
    from vecops_amd import capi
    a, b = _operands(device, torch.bfloat16, 64, 2048, 1408)
    own, planned, automatic, required = (torch.empty((64, 2048), device=device) for _ in range(4))
    plan = capi.plan_matmul(a, b, own)
    assert capi.FAMILY_NAMES[plan.family] == "tile_64" and plan.split_k == 1
    capi.matmul(a, b, own)
    capi.matmul_planned(a, b, planned, plan)
    capi.matmul_family(a, b, automatic, capi.family_request("tile_64", capi.SELECT_AUTOMATIC))
    capi.matmul_family(a, b, required, capi.family_request("tile_64", capi.SELECT_REQUIRE, split_k=1))
    torch.cuda.synchronize()
    assert torch.equal(own, planned) and torch.equal(own, automatic)
    assert not torch.equal(own, required)        # K in four parts here, front to back there
    assert rel_err(own.cpu().numpy(), required.cpu().numpy()) <= fp32_tol(1408)


def test_captured(device):
    """Replayed several times with work of its own between the replays."""
    import torch
    from vecops_amd import capi
    a, b = _operands(device, torch.bfloat16, 33, 1027, 1913)
    want = torch.empty((33, 1027), device=device)
    capi.matmul(a, b, want)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        c = torch.empty_like(want)
        call = capi.PreparedMatmul(a, b, c)
        call()
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            capi.PreparedMatmul(a, b, c)()
    for _ in range(3):
        c.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, want)


def test_planned_calls_run_what_the_plan_names(device):
    """A plan made for a required or preferred family gives that family's bits in the planned call too, where the table's own
    plan has the same family and split; a slim tile in a plan is checked like the rest of it."""
    import torch
    from vecops_amd import capi
    a, b = _operands(device, torch.bfloat16, 64, 2048, 1408)
    make = lambda: torch.full((64, 2048), 7.0, device=device)  # noqa: E731
    own = capi.matmul(a, b, make())
    for selection in (capi.SELECT_REQUIRE, capi.SELECT_PREFER):
        for split in (0, 1):
            request = capi.family_request("tile_64", selection, split_k=split)
            plan = capi.plan_matmul_family(a, b, make(), request)
            table = capi.plan_matmul(a, b, make())
            assert (plan.family, plan.split_k, plan.slim_tile) == (table.family, table.split_k, 0) and table.slim_tile != 0
            named, planned = capi.matmul_family(a, b, make(), request), capi.matmul_planned(a, b, make(), plan)
            assert torch.equal(named, planned) and not torch.equal(named, own)
    plan = capi.plan_matmul(a, b, make())
    for bm, bn in ((32, 16), (32, 32), (32, 48), (32, 64), (64, 48), (64, 64), (128, 48), (128, 64)):   # any of them may be asked for
        plan.slim_tile = 256 * bm + bn
        assert torch.equal(capi.matmul_planned(a, b, make(), plan), own)   # K in the same four parts
    c = make()
    for code in (1, 256 * 48 + 48, 256 * 64 + 32, 0xffff):
        plan.slim_tile = code
        with pytest.raises(capi.VecopsHipError) as e:
            capi.matmul_planned(a, b, c, plan)
        assert e.value.code == 1
    plan.slim_tile = 256 * 32 + 16
    with pytest.raises(capi.VecopsHipError):      # operands that slim tiles do not serve
        capi.matmul_planned(a, torch.empty((1408, 2048), device=device, dtype=torch.bfloat16).t(), c, plan)
    plan.family = capi.FAMILY_CODES["tile_256"]   # and tiles that they do not stand in for
    with pytest.raises(capi.VecopsHipError):
        capi.matmul_planned(a, b, c, plan)
    torch.cuda.synchronize()
    assert float(c.min()) == 7.0 and float(c.max()) == 7.0


def test_no_workspace(device):
    """128 x 11008 x 4096: the table's tiles would split K, the slim tile takes nothing - no workspace has to be handed in, and
    the entry points allocate and hold none."""
    import ctypes as C
    import torch
    from vecops_amd import capi
    a, b = _operands(device, torch.bfloat16, 128, 11008, 4096)
    c = torch.empty((128, 11008), device=device)
    plan = capi.plan_matmul(a, b, c)
    assert plan.split_k > 1 and plan.workspace_bytes == plan.split_k * 128 * 11008 * 4 and plan.slim_tile and plan.scratch_bytes == 0
    want = capi.matmul(a, b, c).clone()
    operands = [C.byref(o) if o is not None else None for o in (capi.operand(a), capi.operand(b), None, capi.operand(c))]
    lib = capi.lib()
    for call in (lambda: lib.vecops_hip_matmul(*operands, 0, None, 0, capi._stream_handle(None)),
                 lambda: lib.vecops_hip_matmul_planned(*operands, 0, C.byref(plan), None, 0, capi._stream_handle(None)),
                 lambda: lib.vecops_hip_matmul_static_workspace(*operands, 0, capi._stream_handle(None))):
        c.fill_(float("nan"))
        capi._check(call())
        assert torch.equal(c, want)
    plan.slim_tile = 0                   # the table's own tiles need theirs
    assert lib.vecops_hip_matmul_planned(*operands, 0, C.byref(plan), None, 0, None) == 1
    stream = torch.cuda.current_stream()
    prepared = capi.PreparedMatmul(a, b, c)
    ep = capi.epilogue(activation="relu")
    for call in (lambda: capi.matmul(a, b, c), lambda: capi.matmul(a, b, c, stream=stream), prepared,
                 lambda: capi.matmul_fused(a, b, c, ep), lambda: capi.matmul_fused(a, b, c, ep, stream=stream),
                 lambda: capi.matmul_planned(a, b, c, capi.plan_matmul(a, b, c))):
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        call()
        torch.cuda.synchronize()
        assert torch.cuda.max_memory_allocated() == before
    assert prepared._keep[4] is None


def _run_on(tile, a, b, c, c_in=None):
    """The product on the named slim tile, whatever the library would choose."""
    from vecops_amd import capi
    plan = capi.plan_matmul_family(a, b, c, capi.family_request("tile_64", split_k=1), c_in=c_in)
    plan.slim_tile = 256 * tile[0] + tile[1]
    return capi.matmul_planned(a, b, c, plan, c_in=c_in)


# (row tiles and rows past them, column tiles and columns past them, K): a K inside one chunk, inside one K tile, one element past
# it, whole stages, and rings that wrap with a partial tile and without
EDGES = [(1, -1, 1, 1, 9), (1, 1, 2, -1, 63), (0, 1, 3, 3, 65), (2, 0, 1, 0, 256), (1, 0, 2, 5, 1291), (1, 17, 1, 2, 2048)]


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("kind", ["bf16", "f16", "i8"])
def test_every_instance(device, kind, tile):
    """Against float64 (int8: exactly), and with C inputs, 16-bit results and strided C: added to or made from the same sums."""
    import torch
    dtype = {"bf16": torch.bfloat16, "f16": torch.float16, "i8": torch.int8}[kind]
    for i, (mt, mr, nt, nr, k) in enumerate(EDGES):
        m, n, pad = mt * tile[0] + mr, nt * tile[1] + nr, i % 3
        a, b = _operands(device, dtype, m, n, k, seed=i, pad=pad)
        g = torch.Generator(device=device).manual_seed(i)
        if kind == "i8":
            sums = _run_on(tile, a, b, torch.full((m, n), -1, dtype=torch.int32, device=device))
            want = torch.from_numpy(_exact(a, b).astype(np.int64)).to(torch.int32).to(device)
            assert torch.equal(sums, want), (i, "sums")
            cin = torch.randint(-2 ** 31, 2 ** 31 - 1, (m, n), generator=g, device=device, dtype=torch.int32)
            out, convert = torch.int32, lambda x: x
        else:
            sums = _run_on(tile, a, b, torch.full((m, n), float("nan"), device=device))
            # (fp32_tol grows with K in tiles of 32 terms: at least one)
            assert rel_err(sums.cpu().numpy(), _exact(a, b)) <= fp32_tol(max(k, 32)), (i, "sums")
            cin = torch.randn((m, n), generator=g, device=device).to(dtype)
            out, convert = dtype, lambda x: x.to(dtype)  # noqa: B023
            assert torch.equal(_run_on(tile, a, b, torch.empty((m, n), device=device, dtype=dtype)), sums.to(dtype)), (i, "16 bits")
        plus = lambda x: sums + (x if kind == "i8" else x.float())  # noqa: B023,E731
        wide = torch.empty((m, 2 * n), device=device, dtype=out).copy_(torch.cat([cin, cin], 1))
        for name, c, ci in (("full", torch.empty((m, n), device=device, dtype=out), cin),
                            ("bias", torch.empty((m, n), device=device, dtype=out), cin[:1].expand(m, n)),
                            ("column bias", torch.empty((m, n), device=device, dtype=out), cin[:, :1].expand(m, n)),
                            ("strided input", torch.empty((m, n), device=device, dtype=out), wide[:, ::2]),
                            ("transposed C", torch.empty((n, m), device=device, dtype=out).t(), cin),
                            ("padded C", torch.empty((m, n + 3), device=device, dtype=out)[:, :n], cin),
                            ("strided C", torch.empty((m, 2 * n), device=device, dtype=out)[:, ::2], cin)):
            c.fill_(7)
            assert torch.equal(_run_on(tile, a, b, c, c_in=ci), convert(plus(ci))), (i, name)
        c = cin.clone()                                    # the C input in place
        assert torch.equal(_run_on(tile, a, b, c, c_in=c), convert(plus(cin))), (i, "in place")


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("kind", ["bf16", "i8"])
def test_batches_with_c_inputs_and_padded_rows(device, kind, tile):
    import torch
    dtype = torch.bfloat16 if kind == "bf16" else torch.int8
    batch, m, n, k = 3, tile[0] + 1, 2 * tile[1] + 1, 197
    a, b = _operands(device, dtype, m, n, k, batch=(batch,), pad=3)
    out = torch.float32 if kind == "bf16" else torch.int32
    cin = torch.arange(batch * m * n, device=device, dtype=torch.int32).view(batch, m, n).to(out)
    one = torch.stack([_run_on(tile, a[i], b[i], torch.empty((m, n), dtype=out, device=device)) for i in range(batch)])
    empty = lambda: torch.full((batch, m, n), 7, dtype=out, device=device)  # noqa: E731
    assert torch.equal(_run_on(tile, a, b, empty()), one)
    assert torch.equal(_run_on(tile, a, b, empty(), c_in=cin), one + cin)
    bias = cin[:1, :1].expand(batch, m, n)
    assert torch.equal(_run_on(tile, a, b, empty(), c_in=bias), one + bias)
    shared = b[:1].expand(batch, n, k)                     # one B for every batch
    want = torch.stack([_run_on(tile, a[i], b[0], torch.empty((m, n), dtype=out, device=device)) for i in range(batch)])
    assert torch.equal(_run_on(tile, a, shared, empty()), want)


# (m, n, k) on which the library's own plan takes each tile, for int8
INT8 = {(32, 16): (45, 16, 511), (32, 32): (35, 2081, 648), (32, 48): (33, 4418, 1025), (32, 64): (33, 6146, 1800),
        (64, 48): (65, 5442, 2624), (64, 64): (65, 8002, 1937), (128, 48): (132, 6095, 1408), (128, 64): (68, 16319, 1921)}
BF16 = {(32, 16): (47, 15, 193), (32, 32): (38, 2162, 321), (32, 48): (34, 4162, 513), (32, 64): (34, 6239, 897),
        (64, 48): (67, 5441, 1248), (64, 64): (65, 8159, 913), (128, 48): (149, 6050, 640), (128, 64): (195, 8117, 961)}


@pytest.mark.parametrize("tile", TILES)
def test_int8_dequantised_on_every_tile(device, tile):
    import torch
    from vecops_amd import capi
    m, n, k = INT8[tile]
    a, b = _operands(device, torch.int8, m, n, k, seed=3)
    c = torch.full((m, n), -1, dtype=torch.int32, device=device)
    assert capi.plan_matmul(a, b, c).slim_tile == 256 * tile[0] + tile[1]
    capi.matmul(a, b, c)
    rows, columns = torch.rand(m, device=device) + 0.5, torch.rand(n, device=device) + 0.5
    correction = torch.randint(-100000, 100000, (n,), device=device, dtype=torch.int32)
    plain, corrected = (torch.full((m, n), float("nan"), device=device) for _ in range(2))
    capi.matmul_i8_dequant(a, b, rows, columns, plain)
    capi.matmul_i8_dequant(a, b, rows, columns, corrected, correction=correction)
    want = torch.from_numpy(_exact(a, b).astype(np.int64)).to(torch.int32).to(device)
    assert torch.equal(c, want)
    assert torch.equal(plain, (want.float() * rows[:, None]) * columns)
    assert torch.equal(corrected, ((want + correction).float() * rows[:, None]) * columns)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("activation", ["none", "relu", "sigmoid", "silu"])
def test_transforms_on_every_tile(device, tile, activation):
    """The transform of the same sums: bit for bit, but for the two activations on the hardware's exponential."""
    import torch
    from vecops_amd import capi
    m, n, k = BF16[tile]
    a, b = _operands(device, torch.bfloat16, m, n, k, seed=4)
    a = (a.float() * 0.05).bfloat16()
    sums = torch.empty((m, n), device=device)
    assert capi.plan_matmul(a, b, sums).slim_tile == 256 * tile[0] + tile[1]
    capi.matmul(a, b, sums)
    g = torch.Generator(device=device).manual_seed(7)
    rows, columns = torch.rand(m, generator=g, device=device) + 0.5, torch.rand(n, generator=g, device=device) + 0.5
    cin = torch.randn((m, n), generator=g, device=device)
    for ci in (None, cin, cin[:1].expand(m, n)):
        ep = capi.epilogue(activation=activation, row_scales=rows, column_scales=columns, scale=0.5, shift=0.25)
        c = torch.full((m, n), float("nan"), device=device)
        assert capi.plan_matmul_fused(a, b, c, ep, c_in=ci).slim_tile == 256 * tile[0] + tile[1]
        capi.matmul_fused(a, b, c, ep, c_in=ci)
        v = (((sums if ci is None else sums + ci) * rows[:, None]) * columns) * 0.5 + 0.25
        if activation in ("none", "relu"):
            assert torch.equal(c, torch.relu(v) if activation == "relu" else v)
        else:
            want = torch.sigmoid(v.double()) * (v.double() if activation == "silu" else 1.0)
            # (the library states 1e-6 relative for the exponential; the sums and quotients around it are fp32)
            assert bool(((c.double() - want).abs() <= 2e-6 * want.abs() + 1e-30).all())
            half = torch.empty((m, n), device=device, dtype=torch.bfloat16)
            assert torch.equal(capi.matmul_fused(a, b, half, ep, c_in=None if ci is None else ci.bfloat16()),
                               capi.matmul_fused(a, b, torch.empty_like(c), ep, c_in=None if ci is None else ci.bfloat16().float()).bfloat16())
