"""f32 activations at group size 32 (M > 8): the error is relative to the weights, not to the codes.

The three-pass form holds both operands to 16 significant bits (x = x_hi + x_lo, w = w_hi + w_lo with
each part rounded to bf16, so |lo| <= 2^-9 |v| and |v - hi - lo| <= 2^-18 |v|) and drops x_lo . w_lo: a
product is off by at most 3 * 2^-18 |x w| < 2^-16 |x w|, whatever scale and bias cancel in w = s c + b.
The three sums of K products add (3 K + 4) 2^-24 of their magnitudes.  A product formed from the codes
instead (s . (x . c) + b . X) is off by 2^-18 |x| s c and overflows with |x| 15 K, far before w does.
"""
import numpy as np
import pytest
import torch

from gpu_util import banner

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mlxq():
    import mlxq as m
    m.load()
    return m


def _pack(rng, N, K, bits, near):
    """Weights small against s c: b = -s c for one of the top four codes (s a power of two, so both are
    exact in bf16) and, with `near`, fifteen codes in sixteen among those four."""
    top = 2 ** bits - 4
    codes = rng.integers(0, 2 ** bits, (N, K), dtype=np.uint32)
    if near:
        codes = np.where(rng.random((N, K)) < 15 / 16, codes % 4 + top, codes).astype(np.uint32)
    per = 32 // bits
    words = np.zeros((N, K // per), np.uint32)
    for i in range(per):
        words |= codes[:, i::per] << np.uint32(i * bits)
    s = np.ldexp(1.0, rng.integers(-9, -5, (N, K // 32)))
    b = -s * (top + rng.integers(0, 4, (N, K // 32)))
    w = codes * np.repeat(s, 32, 1) + np.repeat(b, 32, 1)
    return w, torch.from_numpy(words.view(np.int32)).to("cuda"), *(torch.from_numpy(t).to("cuda") for t in (s, b))


@pytest.mark.parametrize("lora", [False, True])
@pytest.mark.parametrize("sb", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K,bits", [(9, 130, 640, 4), (33, 257, 1280, 8), (200, 96, 64, 4), (129, 300, 3072, 4),
                                        (700, 520, 1088, 8), (40, 70, 96, 4)])
def test_f32_group32_error_is_relative_to_the_weights(mlxq, lora, sb, M, N, K, bits):
    banner("f32 g32", lora, sb, M, N, K, bits)
    rng = np.random.default_rng(M + N + K)
    w, wq, s, b = _pack(rng, N, K, bits, True)
    x = rng.standard_normal((M, K)).astype(np.float32)
    ab = {"lora_a": torch.zeros(K, 8, device="cuda"), "lora_b": torch.zeros(8, N, device="cuda")} if lora else {}
    y = mlxq.linear(torch.from_numpy(x).to("cuda"), wq, s.to(sb), b.to(sb), 32, bits, **ab)
    want = x.astype(np.float64) @ w.T
    bound = (2.0 ** -16 + (3 * K + 4) * 2.0 ** -24) * (np.abs(x).astype(np.float64) @ np.abs(w).T)
    err = np.abs(y.double().cpu().numpy() - want)
    rel = np.linalg.norm(err) / np.linalg.norm(want)
    print(f"    worst error / bound {np.max(err / bound):.3f} rel {rel:.2e}", flush=True)
    assert np.all(err <= bound)
    # independent roundings add as squares: three of at most 2^-18 of a product, and the sums'
    assert rel < 3 ** 0.5 * 2.0 ** -18 + (3 * K) ** 0.5 * 2.0 ** -24


@pytest.mark.parametrize("scale", [2.0 ** 115, 2.0 ** 120])
def test_f32_group32_large_activations(mlxq, scale):
    """|x| about 2^115 and 2^120 against weights of about 2^-10: the results are finite, sums of x with the
    codes themselves would not be."""
    rng = np.random.default_rng(5)
    M, N, K, bits = 20, 64, 640, 8
    w, wq, s, b = _pack(rng, N, K, bits, True)
    x = (rng.standard_normal((M, K)) * scale).astype(np.float32)
    want = x.astype(np.float64) @ (w * 2.0 ** -6).T
    s, b = ((t * 2.0 ** -6).to(torch.bfloat16) for t in (s, b))
    y = mlxq.linear(torch.from_numpy(x).to("cuda"), wq, s, b, 32, bits).double().cpu().numpy()
    assert np.abs(want).max() < 2.0 ** 127 and np.isfinite(y).all()
    assert np.linalg.norm((y - want) / scale) < 1e-5 * np.linalg.norm(want / scale)
