"""The small-grid GEMM with four waves per tile (more 64x64 tiles than CUs) at the edges of its tiles
and of each wave's share of K.

Reference: float64 over the weights dequantized to bf16, round_bf16(fma(code, scale, bias)).  Products
of two bf16 values are exact in f32, so the result is within the f32 accumulation, (K + 4) * 2^-24 of
the sum of magnitudes, and one rounding to bf16, at most 2^-8 of the product;
a bias adds one more rounding, of the sum.
"""
import pytest
import torch

from gpu_util import banner

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mlxq():
    import mlxq as m
    m.load()
    return m


# Tiles just past 256 and up to the kernel's 1152; rows and columns one past and one short of a tile;
# K steps that split unevenly over four waves (9, 11, 13), the shortest K (8 steps), group counts that
# the staged scales take (multiples of 8) and that they do not.
@pytest.mark.parametrize("M,N,K,gs,bits", [
    (65, 8192 + 1, 512, 64, 4), (257, 3265, 576, 64, 4), (333, 3072, 704, 32, 4), (300, 3300, 832, 64, 8),
    (200, 4127, 1024, 128, 4), (130, 5567, 640, 128, 8), (9, 16500, 512, 32, 8), (449, 4097, 1536, 64, 4),
])
@pytest.mark.parametrize("bias", [False, True])
def test_small_four_waves(mlxq, M, N, K, gs, bits, bias):
    banner("small four waves", M, N, K, gs, bits, bias)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    wq = torch.randint(-2 ** 31, 2 ** 31, (N, K * bits // 32), generator=g, device="cuda", dtype=torch.int32)
    s, z = ((torch.randn((N, K // gs), generator=g, device="cuda") * std).to(torch.bfloat16) for std in (0.01, 0.05))
    x = torch.randn((M, K), generator=g, device="cuda").to(torch.bfloat16)
    b = torch.randn(N, generator=g, device="cuda").to(torch.bfloat16) if bias else None
    y = mlxq.linear(x, wq, s, z, gs, bits, bias=b)
    w = mlxq.dequantize(wq, s, z, gs, bits).double()
    assert w.shape == (N, K)
    want = x.double() @ w.t().contiguous()
    bound = (K + 4) * 2.0 ** -24 * (x.double().abs() @ w.abs().t().contiguous()) + 2.0 ** -8 * want.abs()
    if bias:
        want = want + b.double()
        bound += 2.0 ** -8 * want.abs()
    err = (y.double() - want).abs()
    print(f"    worst error / bound {(err / bound).max().item():.3f}", flush=True)
    assert bool((err <= bound).all())
