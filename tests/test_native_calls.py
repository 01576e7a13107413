"""The entry points' per-call work in native code (host/torch/calls.cpp): calls on plain device tensors on the current stream
give what the Python form gives (which a stream named by the caller still takes), and every other call is left to it."""
import pytest
import torch

from vecops_amd import capi
from vecops_amd import host_api as H
from vecops_amd import torch_bridge as tb


def test_calls_that_are_left_to_the_python_form():
    calls = capi.native_calls()
    a, b, c = torch.zeros(4, 8), torch.zeros(5, 8), torch.zeros(4, 5)
    assert calls.matmul(a, b, c, None, 0, None) == -1                       # host tensors
    assert calls.matmul(a.to("meta"), b.to("meta"), c.to("meta"), None, 0, None) == -1
    assert calls.matmul(a, None, c, None, 0, None) == -1
    assert calls.matmul(a, b, "c", None, 0, None) == -1
    assert calls.matmul_fused(a, b, c, None, 0, None, 1 << 80) == -1
    assert calls.matmul_w8a16_group(a, b, a, c, 2.0) == -1
    assert calls.matmul_i8_dequant(a, b, a, a, c, None, None, -1) == -1
    assert calls.matmul_runtime_quant(a, a, 1 << 40, b, a, a, c, None, None, -1) == -1
    assert calls.matmul_packed_b(a, b, c, None, 0, None, 5) == -1
    with pytest.raises(TypeError, match="expected 6 arguments"):
        calls.matmul(a, b, c)


def _bf16(device, *shape):
    return torch.randn(*shape, device=device).bfloat16()


@pytest.mark.gpu
def test_products_equal_the_python_form(device):
    stream = torch.cuda.current_stream()
    i8 = lambda *shape: torch.randint(-128, 128, shape, device=device, dtype=torch.int8)  # noqa: E731
    both = lambda call, like: (call(torch.full_like(like, 3), None), call(torch.full_like(like, 5), stream))  # noqa: E731
    out = []
    for m, n, k in ((33, 260, 1000), (255, 63, 8191), (1, 512, 4096)):
        a, b, cin = _bf16(device, m, k), _bf16(device, n, k), torch.randn(m, n, device=device)
        f = torch.empty(m, n, device=device)
        out += [both(lambda c, s: capi.matmul(a, b, c, stream=s), f),  # noqa: B023
                both(lambda c, s: capi.matmul(a, b, c, c_in=cin, stream=s), f.bfloat16()),  # noqa: B023
                both(lambda c, s: capi.matmul(a.float(), b.float(), c, compute=capi.COMPUTE_F32, stream=s), f)]  # noqa: B023
        ep = capi.epilogue(activation="relu", scale=0.5)
        out.append(both(lambda c, s: capi.matmul_fused(a, b, c, ep, c_in=cin[:1].expand(m, n), stream=s), f.bfloat16()))  # noqa: B023
        packed = capi.pack_b(b)
        out.append(both(lambda c, s: capi.matmul_packed_b(a, packed, c, stream=s), f))  # noqa: B023
        ia, ib = i8(m, k), i8(n, k)
        rows, columns = torch.rand(m, device=device) + 0.5, torch.rand(n, device=device) + 0.5
        corr = torch.arange(n, device=device, dtype=torch.int32)
        ipacked = capi.pack_b(ib)
        out.append(both(lambda c, s: capi.matmul_i8_dequant(ia, ib, rows, columns, c, correction=corr, stream=s), f))  # noqa: B023
        if m > 16:
            out.append(both(lambda c, s: capi.matmul_i8_dequant_packed_b(ia, ipacked, rows, columns, c, stream=s), f))  # noqa: B023
        x = torch.randn(m, k, device=device)
        out += [both(lambda c, s: capi.matmul_runtime_quant(x, rows, 128, ib, rows, columns, c, stream=s), f),  # noqa: B023
                both(lambda c, s: capi.matmul_runtime_quant_packed_b(x, rows, 128, ipacked, rows, columns, c, correction=corr, stream=s), f)]  # noqa: B023
    x, w = _bf16(device, 4, 512), i8(256, 512)
    scales = torch.rand(256, 4, device=device)
    out.append(both(lambda c, s: capi.matmul_w8a16_group(x, w, scales, c, 128, stream=s), _bf16(device, 4, 256)))
    torch.cuda.synchronize()
    for native, python in out:
        assert torch.equal(native, python)


@pytest.mark.gpu
def test_workspaces_streams_and_refusals(device):
    a, b = _bf16(device, 255, 8191), _bf16(device, 63, 8191)
    want = capi.matmul(a, b, torch.empty(255, 63, device=device))
    need = int(capi.plan_matmul(a, b, want).workspace_bytes)
    for size in (need, 16):      # the caller's own, and one that is too small: another is allocated
        workspace = torch.empty(size, dtype=torch.uint8, device=device)
        assert torch.equal(capi.matmul(a, b, torch.empty_like(want), workspace=workspace), want)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        assert torch.equal(capi.matmul(a, b, torch.empty_like(want)), want)
    with pytest.raises(capi.VecopsHipError, match="K of a") as e:
        capi.matmul(a, b[:, :-1], want)
    assert e.value.code == 1
    with pytest.raises(KeyError):
        capi.matmul(a.long(), b.long(), want)
    with pytest.raises(IndexError):
        capi.matmul(a[None, None], b[None, None], want[None, None])
    with pytest.raises(AssertionError):
        capi.matmul_w8a16_group(a[:4].t(), torch.zeros(8, 4, dtype=torch.int8, device=device), torch.ones(8, 1, device=device),
                                torch.empty(8191, 8, device=device, dtype=torch.bfloat16), 4)


@pytest.mark.gpu
def test_wrapped_tensors_are_refused_as_before(device):
    a, b, c = _bf16(device, 3, 4, 64), _bf16(device, 8, 64), torch.empty(3, 4, 8, device=device)
    with pytest.raises(RuntimeError, match="storage|data_ptr|data pointer"):
        torch.vmap(lambda x, y: capi.matmul(x, b, y))(a, c)


@pytest.mark.gpu
def test_registered_operator_forms(device):
    """Outputs returned or not, scalars, optional tensors, specialization values, mixed host and device tensors, errors."""
    plain = tb.register("vecops_hip_n::matmul")
    returning = tb.register("vecops_hip_nr::matmul", return_outputs=True)
    a, b = _bf16(device, 5, 4096), _bf16(device, 520, 4096)
    want = capi.matmul(a, b, torch.empty(5, 520, device=device))
    c = torch.empty(5, 520, device=device)
    assert plain(a, b, None, c) is c and torch.equal(c, want)
    c = torch.empty(5, 520, device=device)
    assert returning(a, b, None, c) is c and torch.equal(c, want)
    c = torch.empty(5, 520, device=device)
    got = torch.ops.vecops_hip_nr.matmul(a, b, None, c)
    assert torch.equal(got if isinstance(got, torch.Tensor) else got[0], want)
    for _ in range(12):          # more signatures than a thread keeps
        for m in (1, 2, 3, 4, 5, 17, 33, 40, 255):
            c = torch.empty(m, 520, device=device)
            plain(a[:1].expand(m, 4096).contiguous(), b, None, c)
            assert torch.allclose(c, want[:1].expand(m, 520), rtol=1e-5, atol=1e-4)
    with pytest.raises(H.HostError) as e:
        plain(a, b[:, :-1], None, c)
    assert e.value.code == 1 and "K" in e.value.message
    with pytest.raises(KeyError):
        plain(a.double(), b.double(), None, c.double())
    fused = tb.register("vecops_hip_n::matmul_fused")
    c = torch.empty(5, 520, device=device)
    fused(a, b, None, None, None, 1, 0.5, 0.25, 0.0, 0.0, c)
    # (the same entry of the library: a product without a transform takes another kernel at these extents)
    assert torch.equal(c, capi.matmul_fused(a, b, torch.empty_like(c), capi.epilogue(activation="relu", scale=0.5, shift=0.25)))


@pytest.mark.gpu
def test_the_interpreter_lock_is_given_up_during_a_call(device):
    """With threads switched only where one gives up the lock, another thread gets to run while this one does nothing but
    calls."""
    import sys
    import threading
    a, b, c = _bf16(device, 33, 512), _bf16(device, 260, 512), torch.empty(33, 260, device=device)
    scales = torch.rand(33, device=device), torch.rand(260, device=device)
    ia, ib = (torch.randint(-9, 9, (r, 512), device=device, dtype=torch.int8) for r in (33, 260))
    ep, packed, x = capi.epilogue(activation="relu"), capi.pack_b(b), torch.randn(33, 512, device=device)
    ipacked, w_scales, y = capi.pack_b(ib), torch.rand(260, 4, device=device), _bf16(device, 5, 260)
    calls = [lambda: capi.matmul(a, b, c), lambda: capi.matmul_fused(a, b, c, ep), lambda: capi.matmul_packed_b(a, packed, c),
             lambda: capi.matmul_i8_dequant(ia, ib, *scales, c), lambda: capi.matmul_w8a16_group(a[:5], ib, w_scales, y, 128),
             lambda: capi.matmul_runtime_quant(x, scales[0], 128, ib, *scales, c),
             lambda: capi.matmul_runtime_quant_packed_b(x, scales[0], 128, ipacked, *scales, c)]
    interval = sys.getswitchinterval()
    for call in calls:
        call()
        torch.cuda.synchronize()
        go, ran = threading.Lock(), []
        go.acquire()
        thread = threading.Thread(target=lambda: (go.acquire(), ran.append(1)))  # noqa: B023
        thread.start()
        sys.setswitchinterval(1000.0)
        try:
            go.release()         # the thread may run from here on, once this one gives up the interpreter lock
            for _ in range(5000):
                if ran:
                    break
                call()
            done = bool(ran)
        finally:
            sys.setswitchinterval(interval)
        thread.join(60)
        torch.cuda.synchronize()
        assert done


@pytest.mark.gpu
def test_calls_from_several_threads(device):
    """Each thread on a stream of its own, products that allocate a workspace among them."""
    import threading
    shapes = [(255, 63, 8191), (128, 11008, 512), (33, 260, 1000), (700, 900, 264)]
    operands = [(_bf16(device, m, k), _bf16(device, n, k)) for m, n, k in shapes]
    want = [capi.matmul(a, b, torch.empty(a.shape[0], b.shape[0], device=device)) for a, b in operands]
    torch.cuda.synchronize()
    results, errors = {}, []

    def work(index):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                for turn in range(20):
                    i = (index + turn) % len(shapes)
                    a, b = operands[i]
                    results[index, turn] = i, capi.matmul(a, b, torch.full_like(want[i], float("nan")))
            stream.synchronize()
        except Exception as e:  # noqa: BLE001
            errors.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    torch.cuda.synchronize()
    assert not errors and len(results) == 80
    assert all(torch.equal(got, want[i]) for i, got in results.values())


def test_without_the_extension(monkeypatch):
    """Not built (no torch headers where the library was made): a warning, and every call takes the Python form; operators are
    registered as before."""
    monkeypatch.setattr(capi, "CALLS_PATH", capi.CALLS_PATH + ".missing")
    monkeypatch.setattr(capi, "_calls", None)
    with pytest.warns(RuntimeWarning, match="missing"):
        calls = capi.native_calls()
    a, b, c = torch.zeros(4, 8), torch.zeros(5, 8), torch.zeros(4, 5)
    assert calls.matmul(a, b, c, None, 0, None) == -1 and calls.matmul_w8a16_group(a, b, a, c, 8) == -1
    assert capi.native_calls() is calls           # (one warning)
    tb.register("vecops_hip_no_extension::matmul")
    for key in ("CUDA", "CPU", "Meta"):
        assert torch._C._dispatch_has_kernel_for_dispatch_key("vecops_hip_no_extension::matmul", key)


@pytest.mark.gpu
def test_products_without_the_extension(device, monkeypatch):
    a, b = _bf16(device, 5, 4096), _bf16(device, 520, 4096)
    want = capi.matmul(a, b, torch.empty(5, 520, device=device))
    monkeypatch.setattr(capi, "CALLS_PATH", capi.CALLS_PATH + ".missing")
    monkeypatch.setattr(capi, "_calls", None)
    with pytest.warns(RuntimeWarning, match="missing"):
        assert torch.equal(capi.matmul(a, b, torch.empty_like(want)), want)
    plain = tb.register("vecops_hip_no_extension_g::matmul")
    c = torch.empty_like(want)
    assert plain(a, b, None, c) is c and torch.equal(c, want)
