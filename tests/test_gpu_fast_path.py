"""The operators' native call path (mlxq._fast) against their general path, which a caller-given
workspace or output forces: the same bits for operands that need no preparation, and the general
path's handling (copies, errors) for those that do."""
import ctypes
import os
import subprocess
import sys

import pytest
import torch

from gpu_util import banner


@pytest.fixture(scope="module")
def mlxq():
    import mlxq as m
    m.load()
    return m


def test_host_tensors_take_the_general_path(mlxq):
    """No GPU needed: every function declines, and the operator reports the error."""
    f = mlxq._lib.fast()
    x, wq = torch.zeros(2, 64), torch.zeros(4, 8, dtype=torch.int32)
    s = torch.zeros(4, 1)
    assert f.quantized_matmul(x, wq, s, s, 64, 4) is None
    assert f.linear(x, wq, s, s, 64, 4, None, None, None, 1.0, 0) is None
    assert f.swiglu(x, (wq, s, s), [wq, s, s], 64, 4) is None
    assert f.embedding(torch.zeros(3, dtype=torch.int32), wq, s, s, 64, 4, 1) is None
    assert f.dequantize(wq, s, s, 64, 4) is None and f.quantize_batched([x, x], 64, 4) is None
    assert f.quantize_batched((x,), 64, 4) is None and f.quantize_batched([], 64, 4) is None
    assert f.linear(None, 3, "a", s, 64, 4, None, None, None, 1.0, 0) is None
    assert f.quantized_matmul(x) is None
    with pytest.raises(ValueError):
        mlxq.quantized_matmul(x, wq, s, s)


def _pack(N, K, gs, bits, sb, dev="cuda"):
    g = torch.Generator(device=dev).manual_seed(N + K)
    wq = torch.randint(-2 ** 31, 2 ** 31, (N, K * bits // 32), generator=g, device=dev, dtype=torch.int32)
    mk = lambda: (torch.randn((N, K // gs), generator=g, device=dev) * 0.02).to(sb)  # noqa: E731
    return wq, mk(), mk()


@pytest.mark.gpu
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("sb", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(128,), (1, 128), (5, 128), (2, 9, 128)])
def test_fast_matches_general(mlxq, xdt, sb, shape):
    banner("fast path", xdt, sb, shape)
    N = 40
    p = _pack(N, 128, 64, 4, sb)
    x = torch.randn(shape, device="cuda").to(xdt)
    bias = torch.randn(N, device="cuda").to(torch.bfloat16)
    a, b = (torch.randn(128, 8, device="cuda") * 0.1).to(sb), (torch.randn(8, N, device="cuda") * 0.1).to(sb)
    ws = torch.empty(1 << 20, dtype=torch.uint8, device="cuda")
    for kw in ({}, {"bias": bias}, {"bias": bias, "lora_a": a, "lora_b": b, "lora_scale": 0.5}, {"activation": 1}):
        got, want = mlxq.linear(x, *p, 64, 4, **kw), mlxq.linear(x, *p, 64, 4, workspace=ws, **kw)
        assert got.dtype == want.dtype and got.shape == want.shape == shape[:-1] + (N,) and torch.equal(got, want)
    got = mlxq.quantized_matmul(x, *p, True, 64, 4)
    out = torch.empty_like(got)
    assert torch.equal(got, mlxq.quantized_matmul(x, *p, True, 64, 4, out=out)) and got.shape == shape[:-1] + (N,)


@pytest.mark.gpu
def test_fast_swiglu_embedding_and_prepared_operands(mlxq):
    gate, up = _pack(48, 128, 64, 4, torch.bfloat16), _pack(48, 128, 64, 4, torch.bfloat16)
    x = torch.randn((3, 128), device="cuda").to(torch.bfloat16)
    h = mlxq.swiglu(x, gate, up)
    out = torch.empty_like(h)
    assert torch.equal(h, mlxq.swiglu(x, list(gate), up, out=out))
    ids = torch.tensor([[3, 0], [47, 99]], device="cuda", dtype=torch.int32)
    for dt in (torch.bfloat16, torch.float32):
        e = mlxq.embedding(ids, *gate, out_dtype=dt)
        want = mlxq.embedding(ids.long(), *gate, out_dtype=dt)  # int64 ids: the general path
        assert e.shape == (2, 2, 128) and e.dtype == dt and torch.equal(e.isnan(), want.isnan())
        assert torch.equal(e.nan_to_num(), want.nan_to_num()) and e[1, 1].isnan().all()
    # operands that need preparation: strided and unaligned views, as before
    want = mlxq.linear(x, *gate)
    wide = torch.zeros((3, 256), device="cuda", dtype=torch.bfloat16)
    wide[:, 1:129] = x
    assert torch.equal(mlxq.linear(wide[:, 1:129], *gate), want)
    assert torch.equal(mlxq.linear(x, gate[0], gate[1].t().contiguous().t(), gate[2]), want)
    shifted = torch.zeros(48 * 2 + 1, device="cuda", dtype=torch.bfloat16)
    shifted[1:] = gate[1].flatten()
    assert torch.equal(mlxq.linear(x, gate[0], shifted[1:].view(48, 2), gate[2]), want)
    assert mlxq.linear(x[:0], *gate).shape == (0, 48)
    # refusals keep their kind
    with pytest.raises(mlxq.MlxqError) as e:
        mlxq.linear(x[:, :64], *gate)
    assert e.value.status == 1
    with pytest.raises(mlxq.MlxqError) as e:
        mlxq.swiglu(torch.zeros((9, 128), device="cuda", dtype=torch.bfloat16), gate, up)
    assert e.value.status == 2
    with pytest.raises(mlxq.MlxqError):
        mlxq.linear(x, *gate, 64, 4, activation=9)
    with pytest.raises(mlxq.MlxqError):
        mlxq.quantized_matmul(x, *gate, False, 64, 4)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,K,gs,bits,count", [(5, 192, 64, 4, 1), (33, 128, 128, 8, 3), (7, 96, 32, 4, 17)])
def test_fast_quantize_dequantize(mlxq, dt, N, K, gs, bits, count):
    ws = [(torch.randn((N, K), device="cuda") * 0.02).to(dt) for _ in range(count)]
    got = mlxq.quantize_batched(ws, gs, bits)
    want = mlxq.quantize_batched(tuple(ws), gs, bits)  # a tuple: the general path
    assert type(got) is list and all(type(t) is tuple for t in got)
    for g, w in zip(got, want):
        for a, b in zip(g, w):
            assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b)
        assert g[2].data_ptr() - g[1].data_ptr() == w[2].data_ptr() - w[1].data_ptr()
    d = mlxq.dequantize(*got[0], gs, bits)
    strided = got[0][1].t().contiguous().t()  # needs preparation: the general path
    assert d.dtype == dt and torch.equal(d, mlxq.dequantize(got[0][0], strided, got[0][2], gs, bits))
    with pytest.raises(mlxq.MlxqError):
        mlxq.dequantize(got[0][0], got[0][1][:, :0], got[0][2], gs, bits)
    with pytest.raises(mlxq.MlxqError):
        mlxq.quantize_batched(ws, 48, bits)


def test_stream_query_is_looked_up_at_import():
    """No GPU needed: the module takes torch's stream query when it is loaded (a first call of several
    threads at once must not import), so it does not load without one."""
    code = ("import torch, sys; sys.path.insert(0, {!r}); import mlxq; q = torch._C._cuda_getCurrentRawStream\n"
            "del torch._C._cuda_getCurrentRawStream\n"
            "try:\n    import mlxq._fast; print('loaded')\n"
            "except (ImportError, AttributeError):\n    torch._C._cuda_getCurrentRawStream = q; import mlxq._fast; print('ok')\n")
    pkg = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mlx-gen_amd")
    r = subprocess.run([sys.executable, "-c", code.format(pkg)], capture_output=True, text=True, timeout=110)
    assert r.stdout.strip() == "ok", r.stdout + r.stderr


@pytest.mark.gpu
def test_device_error_is_raised_once(mlxq):
    """A launch check that finds an error (here one that a refused hipSetDevice left recorded on this
    thread) raises MLXQ_EDEVICE with the library's message, as the general path does, and is not tried again."""
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    hip = ctypes.CDLL(path)
    p = _pack(40, 128, 64, 4, torch.bfloat16)
    x = torch.ones((2, 128), device="cuda", dtype=torch.bfloat16)
    ids = torch.zeros(3, device="cuda", dtype=torch.int32)
    w = [torch.ones((8, 128), device="cuda")]
    out = torch.empty((2, 40), device="cuda", dtype=torch.bfloat16)
    calls = [lambda: mlxq.quantized_matmul(x, *p, out=out),  # the general path
             lambda: mlxq.quantized_matmul(x, *p), lambda: mlxq.linear(x, *p), lambda: mlxq.swiglu(x, p, p),
             lambda: mlxq.embedding(ids, *p), lambda: mlxq.dequantize(*p), lambda: mlxq.quantize_batched(w)]
    for call in calls:
        call()
        torch.cuda.synchronize()
        assert hip.hipSetDevice(9999) != 0
        try:
            with pytest.raises(mlxq.MlxqError, match="launch failed") as e:
                call()
        finally:
            hip.hipGetLastError()
        assert e.value.status == 3
        call()
    torch.cuda.synchronize()


@pytest.mark.gpu
def test_nested_tensors_stay_refused(mlxq):
    p = _pack(32, 64, 64, 4, torch.bfloat16)
    row = torch.ones(64, device="cuda", dtype=torch.bfloat16)
    x = torch.nested.nested_tensor([row, row, row])
    for call in (lambda: mlxq.linear(x, *p), lambda: mlxq.quantized_matmul(x, *p), lambda: mlxq.swiglu(x, p, p)):
        with pytest.raises(RuntimeError, match="Nested"):
            call()
