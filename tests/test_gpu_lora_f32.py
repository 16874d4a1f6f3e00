"""The f32 LoRA residual (promote(x, factors) is f32): x.A and (x.A).B on the f32 matrix cores.

Every case is the residual alone (y = 0 in f32) against float64.  The bound: an f32 sum of K terms
in any order is within K * 2^-24 of the sum of their magnitudes, so with |x|.|A| = S the staged
x.A is within K * 2^-24 * S and the result within (K + R + 2) * 2^-24 * (|x|.|A|).|B| * scale,
element by element.
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


DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


# Ranks: one column block, a padded one, two adjacent columns per lane (even), an odd rank past 16
# (single columns over several blocks), four per lane, the maximum.  K: fewer steps than waves, a
# remainder past whole chunks, not a multiple of 16 (the one-thread-per-output form).  M, N: one
# row, tiles cut at 16, 32, 64 and 256, odd N (no paired stores).
@pytest.mark.parametrize("xdt,fdt", [("f32", "bf16"), ("f32", "f32"), ("f16", "bf16"), ("f16", "f32"), ("bf16", "f32")])
@pytest.mark.parametrize("M,K,N,rank", [
    (1, 64, 1, 1), (5, 48, 65, 8), (17, 1040, 258, 16), (33, 2048, 255, 18), (16, 3072, 64, 32),
    (31, 160, 96, 33), (65, 992, 514, 64), (32, 512, 300, 100), (9, 256, 40, 256), (40, 72, 130, 32),
])
def test_lora_residual_f32(mlxq, xdt, fdt, M, K, N, rank):
    banner("lora f32", xdt, fdt, M, K, N, rank)
    rng = np.random.default_rng(M * 1000 + rank)
    mk = lambda shape, dt: torch.from_numpy(rng.standard_normal(shape).astype(np.float32)).to("cuda").to(DT[dt])  # noqa: E731
    x, a, b = mk((M, K), xdt), mk((K, rank), fdt), mk((rank, N), fdt)
    y = torch.zeros((M, N), dtype=torch.float32, device="cuda")
    out = mlxq.lora_residual(x, y, a, b, 0.75)
    torch.cuda.synchronize()
    xd, ad, bd = (t.double().cpu().numpy() for t in (x, a, b))
    want = 0.75 * ((xd @ ad) @ bd)
    bound = 0.75 * (K + rank + 2) * 2.0 ** -24 * ((np.abs(xd) @ np.abs(ad)) @ np.abs(bd))
    err = np.abs(out.double().cpu().numpy() - want)
    print(f"    worst error / bound {np.max(err / np.maximum(bound, 1e-300)):.3f}", flush=True)
    assert np.all(err <= bound)


def test_lora_residual_f32_infinity(mlxq):
    """An infinite activation reaches its own row only, and padding ranks (17 of 32) stay zero."""
    x = torch.ones((33, 64), device="cuda")
    x[4, 63] = float("inf")
    a = torch.ones((64, 17), device="cuda")
    b = torch.ones((17, 70), device="cuda")
    out = mlxq.lora_residual(x, torch.zeros((33, 70), device="cuda"), a, b, 1.0)
    torch.cuda.synchronize()
    assert torch.isinf(out[4]).all()
    keep = [i for i in range(33) if i != 4]
    assert (out[keep] == 64 * 17).all()


@pytest.mark.parametrize("xdt,fdt,ydt", [("bf16", "bf16", "bf16"), ("bf16", "bf16", "f32"), ("f32", "bf16", "f32"), ("f16", "f32", "bf16"),
                                         ("bf16", "f32", "bf16")])
@pytest.mark.parametrize("N,rank", [(640, 8), (333, 17), (64, 32), (1, 1), (2050, 64)])
def test_lora_epilogue_grid_forms(mlxq, xdt, fdt, ydt, N, rank):
    """One, four or sixteen waves per 32 x 64 block (over 512 blocks, up to 512, up to 64): the same bits,
    with paired columns and (odd N, a y that starts at an odd element) single ones."""
    banner("lora epilogue forms", xdt, fdt, ydt, N, rank)
    g = torch.Generator(device="cuda").manual_seed(N + rank)
    mk = lambda shape, dt: torch.randn(shape, generator=g, device="cuda").to(DT[dt])  # noqa: E731
    blocks_n = (N + 63) // 64
    M = 32 * (512 // blocks_n + 1) - 5
    x, a, b, y = mk((M, 96), xdt), mk((96, rank), fdt), mk((rank, N), fdt), mk((M, N), ydt)
    big = mlxq.lora_residual(x, y.clone(), a, b, 0.75)
    xs, fs = x.double(), mlxq.promote(DT[xdt], DT[fdt])
    r = (xs @ a.double()).to(fs).double() @ b.double()
    want = y.double() + (r.to(fs).double() * 0.75).to(fs).double()
    tol = 2.0 ** -6 if "bf16" in (str(fs)[-4:], ydt) or fs == torch.bfloat16 else 1e-5
    assert ((big.double() - want).norm() / want.norm()).item() < tol
    for m0, rows in ((0, 32 * max(1, 512 // blocks_n)), (32, 32 * max(1, 64 // blocks_n) - 3), (M - 5, 5)):
        shifted = torch.empty(rows * N + 1, device="cuda", dtype=DT[ydt])
        for ys in (y[m0:m0 + rows].clone(), shifted[1:].view(rows, N).copy_(y[m0:m0 + rows])):
            got = mlxq.lora_residual(x[m0:m0 + rows], ys, a, b, 0.75)
            assert torch.equal(got, big[m0:m0 + rows]), (m0, rows)
