"""The factored f32 GEMM (fp16, f32 and bf16 activations whose product is f32) at the edges of its
tiles, groups and pipeline, against float64.

fp16 and bf16 activations: every product of an activation and a code is exact, so the result is
within the f32 accumulation: (K + groups + 4) * 2^-24 of sum_g |s_g| |x|.c + |b_g| |x|, where every
order of summation stays.  f32 activations are held to 16 significant bits: 2^-16 of the code term
besides (two roundings of at most 2^-9 each leave 2^-18 of a value; 2^-16 is the stated limit).
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


def _pack(rng, N, K, gs, bits, sb):
    codes = rng.integers(0, 2 ** bits, (N, K), dtype=np.uint32)
    per = 32 // bits
    words = np.zeros((N, K // per), np.uint32)
    for i in range(per):
        words |= codes[:, i::per] << np.uint32(i * bits)
    mk = lambda std: torch.from_numpy((rng.standard_normal((N, K // gs)) * std).astype(np.float32)).to("cuda").to(DT[sb])  # noqa: E731
    return codes, torch.from_numpy(words.view(np.int32)).to("cuda"), mk(0.01), mk(0.1)


def _check(mlxq, x, pack, gs, bits, what, **kw):
    codes, wq, s, b = pack
    y = mlxq.linear(x, wq, s, b, gs, bits, **kw)
    torch.cuda.synchronize()
    assert y.dtype == torch.float32
    K = codes.shape[1]
    xd = x.double().cpu().numpy()
    sd, bd = (np.repeat(t.double().cpu().numpy(), gs, 1) for t in (s, b))
    want = xd @ (codes * sd + bd).T
    ax = np.abs(xd)
    bound = (K + K // gs + 4) * 2.0 ** -24 * (ax @ (codes * np.abs(sd) + np.abs(bd)).T)
    if x.dtype == torch.float32:
        bound += 2.0 ** -16 * (ax @ (codes * np.abs(sd)).T)
    err = np.abs(y.double().cpu().numpy() - want)
    rel = np.linalg.norm(err) / np.linalg.norm(want)
    print(f"    {what} rel {rel:.2e} worst error / bound {np.max(err / bound):.3f}", flush=True)
    assert np.all(err <= bound)
    assert rel < (3e-5 if x.dtype == torch.float32 else 2e-6)


# Steps of K: one, two, three, odd counts, exactly one bias batch of 16 groups, one more and one
# less, several; odd group counts (scale rows that start mid-word).  M and N: one past and one short
# of the 32-row blocks, the 64- and 128-row tiles and the 256 columns.
@pytest.mark.parametrize("xdt,sb", [("f16", "bf16"), ("f32", "bf16"), ("f16", "f32"), ("f32", "f32"), ("bf16", "f32")])
@pytest.mark.parametrize("M,N,K,gs,bits", [
    (9, 1, 64, 64, 4), (33, 31, 128, 128, 8), (64, 257, 192, 64, 8), (65, 256, 64, 32, 4),
    (31, 255, 1024, 64, 4), (127, 33, 1088, 64, 8), (129, 300, 960, 64, 4), (20, 513, 2048, 128, 4),
    (40, 64, 2176, 128, 8), (63, 97, 512, 32, 8), (17, 130, 576, 32, 4), (12, 40, 448, 32, 8),
    (30, 70, 2304, 64, 4),
    # K-groups: as many steps as groups, one more, uneven shares, an odd first group (scale rows that
    # start mid-word), 64-row tiles in two groups, and grids that fill the CUs
    (33, 63, 256, 64, 4), (32, 65, 320, 64, 8), (40, 200, 448, 64, 4), (9, 4096, 1152, 128, 4), (77, 5120, 1280, 64, 8),
    (256, 3000, 704, 64, 4), (250, 2100, 832, 32, 8), (512, 2048, 1536, 128, 8),
    (4224, 2100, 320, 64, 4), (5000, 2600, 576, 64, 4), (6100, 2050, 2176, 128, 4), (4100, 3100, 192, 32, 4), (6200, 1030, 384, 128, 8), (3000, 2600, 128, 32, 4),
])
def test_strip_edges(mlxq, xdt, sb, M, N, K, gs, bits):
    banner("strip", xdt, sb, M, N, K, gs, bits)
    rng = np.random.default_rng(M + 7 * N + K)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to("cuda").to(DT[xdt])
    _check(mlxq, x, _pack(rng, N, K, gs, bits, sb), gs, bits, f"{xdt}/{sb}")


@pytest.mark.parametrize("M", [40, 5000])
def test_strip_fp16_subnormals_and_large(mlxq, M):
    """fp16 activations over their whole range: subnormals (2^-24 up) and values near 65504."""
    rng = np.random.default_rng(M)
    K, N = 256, 1100
    x = torch.from_numpy(np.ldexp(rng.standard_normal((M, K)), rng.integers(-24, 14, (M, 1))).astype(np.float16)).to("cuda")
    _check(mlxq, x, _pack(rng, N, K, 64, 8, "bf16"), 64, 8, "fp16 range")


def test_strip_nonfinite_rows_stay_apart(mlxq):
    """A row with an infinity or a NaN leaves every other row as it was."""
    rng = np.random.default_rng(3)
    for dt in ("f16", "f32"):
        x = torch.from_numpy(rng.standard_normal((70, 640)).astype(np.float32)).to("cuda").to(DT[dt])
        codes, wq, s, b = _pack(rng, 90, 640, 64, 4, "bf16")
        clean = mlxq.linear(x, wq, s, b, 64, 4)
        x2 = x.clone()
        x2[3, 5] = float("inf")
        x2[66, 639] = float("nan")
        y = mlxq.linear(x2, wq, s, b, 64, 4)
        torch.cuda.synchronize()
        keep = [i for i in range(70) if i not in (3, 66)]
        assert torch.equal(y[keep], clean[keep])
        assert not torch.isfinite(y[3]).any() and torch.isnan(y[66]).all()


@pytest.mark.parametrize("xdt,fdt,act,rank", [("f32", "bf16", 1, 32), ("f16", "f32", 0, 17), ("f32", "f32", 2, 8), ("f16", "bf16", 3, 64)])
@pytest.mark.parametrize("M,N", [(33, 100), (4200, 1536)])
def test_strip_bias_lora_act(mlxq, xdt, fdt, act, rank, M, N):
    """The fused epilogue against the product, the bias, lora_residual and the activation apart."""
    rng = np.random.default_rng(rank + M)
    mk = lambda shape, dt, std=1.0: torch.from_numpy((rng.standard_normal(shape) * std).astype(np.float32)).to("cuda").to(DT[dt])  # noqa: E731
    K = 320
    x, bias, a, b = mk((M, K), xdt), mk((N,), "bf16"), mk((K, rank), fdt, 0.05), mk((rank, N), fdt, 0.05)
    _, wq, s, z = _pack(rng, N, K, 64, 4, "bf16")
    got = mlxq.linear(x, wq, s, z, 64, 4, bias=bias, lora_a=a, lora_b=b, lora_scale=0.5, activation=act)
    p = mlxq.linear(x, wq, s, z, 64, 4, bias=bias)
    p = mlxq.lora_residual(x, p, a, b, 0.5).double()
    torch.cuda.synchronize()
    if act in (1, 3):
        p = 0.5 * p * (1 + torch.erf(p / 2 ** 0.5))
    elif act == 2:
        p = 0.5 * p * (1 + torch.tanh((2 / np.pi) ** 0.5 * (p + 0.044715 * p ** 3)))
    # f32 sums and the activations' stated few-1e-7 errors
    rel = ((got.double() - p).norm() / p.norm()).item()
    print(f"    rel {rel:.2e}", flush=True)
    assert rel < 2e-6


@pytest.mark.parametrize("xdt", ["bf16", "f16"])
@pytest.mark.parametrize("M,N,K,gs,bits", [(33, 65, 320, 64, 4), (40, 200, 448, 64, 8), (20, 64, 704, 64, 4), (40, 70, 832, 32, 4),
                                           (9, 4096, 1152, 128, 4), (250, 2100, 832, 32, 8)])
def test_strip_infinity_in_uneven_k_groups(mlxq, xdt, M, N, K, gs, bits):
    """K shared unevenly among a workgroup's K-groups: an infinity anywhere in a row of positive activations
    against positive codes, scales and biases gives infinities, not the NaN of a step that a shorter share
    runs besides."""
    banner("strip infinity", xdt, M, N, K, gs, bits)
    rng = np.random.default_rng(K)
    _, wq, s, b = _pack(rng, N, K, gs, bits, "f32")
    wq, s, b = wq | (0x11111111 if bits == 4 else 0x01010101), s.abs() + 0.5, b.abs() + 0.25
    x = torch.from_numpy(rng.uniform(0.5, 1.5, (M, K)).astype(np.float32)).to("cuda").to(DT[xdt])
    clean = mlxq.linear(x, wq, s, b, gs, bits)
    for i, k in enumerate(range(0, K, 16)):
        row = i % M
        x2 = x.clone()
        x2[row, k] = float("inf")
        y = mlxq.linear(x2, wq, s, b, gs, bits)
        assert bool((y[row] == float("inf")).all()), k
        y[row] = clean[row]
        assert torch.equal(y, clean), k


@pytest.mark.parametrize("xdt,M,N,K", [("f16", 70, (1 << 22) + 40, 64), ("bf16", 9, (1 << 23) - 64, 64), ("f16", 66, 33, (1 << 22) + 64)])
def test_strip_widest(mlxq, xdt, M, N, K):
    """Widths past 2^22: products with the codes stay exact (2e-7 of the result, where weights split into
    bf16 parts give 2e-6).  Some columns of the wide ones, from both ends and the middle.  A long K is summed
    in f32 over K / 64 groups, whose two terms cancel (b = -7.5 s): 2^-24 times the root of their number and
    the terms' size, about 8 times the sum's."""
    banner("strip widest", xdt, M, N, K)
    g = torch.Generator(device="cuda").manual_seed(K)
    wq = torch.randint(-2 ** 31, 2 ** 31, (N, K // 8), generator=g, device="cuda", dtype=torch.int32)
    s = torch.randn((N, K // 64), generator=g, device="cuda") * 0.01
    b = s * -7.5
    x = torch.randn((M, K), generator=g, device="cuda").to(DT[xdt])
    y = mlxq.linear(x, wq, s, b, 64, 4)
    pick = torch.arange(N, device="cuda") if N < 1000 else torch.cat([torch.arange(n, n + 300, device="cuda") for n in (0, N // 2, N - 300)])
    want = torch.zeros((M, len(pick)), dtype=torch.float64, device="cuda")
    shift = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
    for k in range(0, K, 1 << 20):
        k1 = min(K, k + (1 << 20))
        codes = ((wq[pick, k // 8:k1 // 8][..., None] >> shift) & 15).view(len(pick), -1).double()
        w = codes * s[pick, k // 64:k1 // 64].double().repeat_interleave(64, 1) + b[pick, k // 64:k1 // 64].double().repeat_interleave(64, 1)
        want += x[:, k:k1].double() @ w.t().contiguous()
    rel = ((y[:, pick].double() - want).norm() / want.norm()).item()
    print(f"    rel {rel:.2e}", flush=True)
    assert rel < (5e-7 if K < 1000 else 8 * 2.0 ** -24 * (K / 64) ** 0.5)
