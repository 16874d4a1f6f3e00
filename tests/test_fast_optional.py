"""The operators without the native call path (another Python or torch than it was built for, or none
built): the general path takes every call, with one warning.  The HIP library itself stays required."""
import os
import subprocess
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "mlx-gen_amd")

CALLS = """
import sys, warnings
sys.path.insert(0, {pkg!r})
import torch, mlxq
{before}
x, wq, s = torch.zeros(2, 64), torch.zeros(4, 8, dtype=torch.int32), torch.zeros(4, 1)
with warnings.catch_warnings(record=True) as w:
    warnings.simplefilter("always")
    for call in (lambda: mlxq.quantized_matmul(x, wq, s, s), lambda: mlxq.linear(x, wq, s, s), lambda: mlxq.dequantize(wq, s, s),
                 lambda: mlxq.swiglu(x, (wq, s, s), (wq, s, s)), lambda: mlxq.quantize_batched([x]),
                 lambda: mlxq.embedding(torch.zeros(3, dtype=torch.int32), wq, s, s)):
        try:
            call()
            print("no error")
        except ValueError as e:
            assert "GPU tensors only" in str(e), e
print(len([m for m in w if issubclass(m.category, RuntimeWarning) and "mlxq._fast" in str(m.message)]))
"""


@pytest.mark.parametrize("before,warned", [
    ("", "0"), ("sys.modules['mlxq._fast'] = None", "1"), ("torch.__version__ = '1.0'", "1"),
])
def test_operators_without_the_native_path(before, warned):
    r = subprocess.run([sys.executable, "-c", CALLS.format(pkg=PKG, before=before)], capture_output=True, text=True, timeout=110)
    assert r.returncode == 0 and r.stdout.strip() == warned, r.stdout + r.stderr


def test_makefile_without_torch():
    """The libraries build where the Python has no torch; the native path is left out."""
    r = subprocess.run(["make", "-n", "-B", "-C", os.path.join(PKG, "csrc"), "PYTHON=/bin/false", "all"], capture_output=True,
                       text=True, timeout=110)
    assert r.returncode == 0 and "libmlxq_hip.so" in r.stdout and "fast.cpp" not in r.stdout, r.stdout + r.stderr


@pytest.mark.gpu
def test_same_results_without_the_native_path(monkeypatch):
    import mlxq
    g = torch.Generator(device="cuda").manual_seed(1)
    w = [(torch.randn((48, 128), generator=g, device="cuda") * 0.02).to(torch.bfloat16) for _ in range(2)]
    x = torch.randn((3, 128), generator=g, device="cuda").to(torch.bfloat16)
    ids = torch.tensor([3, 47], device="cuda", dtype=torch.int32)

    def every():
        p, q = mlxq.quantize_batched(w, 64, 4)
        return [*p, mlxq.quantized_matmul(x, *p), mlxq.linear(x, *p, activation=2), mlxq.swiglu(x, p, q), mlxq.dequantize(*q),
                mlxq.embedding(ids, *p)]

    want = every()
    monkeypatch.setattr(mlxq._lib, "_fast", mlxq._lib._NoFast())
    for a, b in zip(every(), want):
        assert a.dtype == b.dtype and torch.equal(a, b)
