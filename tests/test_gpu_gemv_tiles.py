"""The decode GEMV's several-tiles form, its long-K plans with up to eight rows in one launch, and its
own bias and activation, at the edges of tiles and of the rows a workgroup walks.

Reference: float64 over the exact dequantized weights (the GEMV's definition), rounded to bf16 as the
call rounds: within one bf16 ulp of the product (2^-8 of its magnitude) plus the f32 accumulation,
(K + 64) * 2^-24 of the sum of magnitudes; a bias adds one more bf16 rounding, of the sum.
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


def _pack(seed, N, K, gs, bits):
    g = torch.Generator(device="cuda").manual_seed(seed)
    wq = torch.randint(-2 ** 31, 2 ** 31, (N, K * bits // 32), generator=g, device="cuda", dtype=torch.int32)
    mk = lambda std: (torch.randn((N, K // gs), generator=g, device="cuda") * std).to(torch.bfloat16)  # noqa: E731
    return wq, mk(0.01), mk(0.05)


def _dense(p, gs, bits):
    shift = torch.arange(0, 32, bits, device="cuda", dtype=torch.int32)
    codes = ((p[0][..., None] >> shift) & (2 ** bits - 1)).view(p[0].shape[0], -1).double()
    s, b = (t.double().repeat_interleave(gs, 1) for t in p[1:])
    return codes * s + b, codes * s.abs() + b.abs()


# N against 256 CUs: just past and short of 16 rows each, two tiles and a row, a last workgroup with one
# row, odd N; K through single rounds, rings of two and ragged last waves; every (bits, group size).
@pytest.mark.parametrize("M,K,N,gs,bits", [
    (3, 1024, 4097, 64, 4), (8, 2560, 8193, 128, 4), (4, 4096, 8447, 64, 4), (5, 11008, 4100, 64, 4),
    (8, 4096, 12290, 64, 4), (1, 4096, 14336, 64, 8), (6, 1280, 12289, 32, 4), (8, 3072, 9216, 32, 8),
    (1, 2880, 5760, 64, 4), (4, 2880, 130, 64, 4), (8, 1088, 9000, 64, 4), (5, 96, 33, 32, 4), (2, 1184, 77, 32, 4),
    (6, 736, 711, 32, 8), (1, 32, 5, 32, 8), (3, 64, 300, 64, 4), (8, 11072, 200, 64, 4),
    (7, 2048, 8960, 128, 8), (3, 6144, 8703, 64, 8), (8, 14336, 300, 64, 4), (6, 18944, 130, 128, 4),
])
@pytest.mark.parametrize("bias,act", [(False, 0), (True, 0), (True, 3)])
def test_gemv_tiles(mlxq, M, K, N, gs, bits, bias, act):
    banner("gemv tiles", M, K, N, gs, bits, bias, act)
    p = _pack(N + K, N, K, gs, bits)
    x = torch.randn((M, K), device="cuda").to(torch.bfloat16)
    b = torch.randn(N, device="cuda").to(torch.bfloat16) if bias else None
    y = mlxq.linear(x, *p, gs, bits, bias=b)
    w, mag = _dense(p, gs, bits)
    want = x.double() @ w.t().contiguous()
    bound = (K + 64) * 2.0 ** -24 * (x.double().abs() @ mag.t().contiguous()) + 2.0 ** -8 * want.abs()
    if bias:
        want = want + b.double()
        bound += 2.0 ** -8 * want.abs()
    err = (y.double() - want).abs()
    print(f"    worst error / bound {(err / bound).max().item():.3f}", flush=True)
    assert bool((err <= bound).all())
    if act:  # the activation of the rounded sum, bit for bit the elementwise epilogue's table
        z = mlxq.linear(x, *p, gs, bits, bias=b, activation=act)
        eye = torch.zeros((M, 64), device="cuda", dtype=torch.bfloat16)
        r = mlxq.lora_residual(eye, y.clone(), torch.zeros((64, 1), device="cuda", dtype=torch.bfloat16),
                               torch.zeros((1, N), device="cuda", dtype=torch.bfloat16), 1.0)
        assert torch.equal(r, y)
        sel = (torch.zeros((N, 8), dtype=torch.int32, device="cuda"), torch.zeros((N, 1), dtype=torch.bfloat16, device="cuda"),
               torch.zeros((N, 1), dtype=torch.bfloat16, device="cuda"))
        for m in range(M):  # a product of zero plus y as the bias, through the GEMM's table
            t = mlxq.linear(torch.zeros((9, 64), device="cuda", dtype=torch.bfloat16), *sel, 64, 4, bias=y[m].contiguous(),
                            activation=act)
            assert torch.equal(t[0], z[m])


@pytest.mark.parametrize("M,K,F,gs,bits", [(3, 4096, 8200, 64, 4), (5, 4096, 11008, 64, 4), (8, 2048, 8193, 128, 8), (8, 3072, 8300, 64, 8)])
def test_swiglu_tiles(mlxq, M, K, F, gs, bits):
    """Several tiles per workgroup against the same rows asked for in pieces of one tile each."""
    if K == 4096:  # a K that is no multiple of the load step stays outside the fused form
        with pytest.raises(mlxq.MlxqError) as e:
            mlxq.swiglu(torch.zeros((M, 2880), device="cuda", dtype=torch.bfloat16), _pack(1, 64, 2880, 64, 4), _pack(2, 64, 2880, 64, 4))
        assert e.value.status == 2
    g, u = _pack(1, F, K, gs, bits), _pack(2, F, K, gs, bits)
    x = torch.randn((M, K), device="cuda").to(torch.bfloat16)
    h = mlxq.swiglu(x, g, u, gs, bits)
    for f0 in range(0, F, 4096):
        f1 = min(F, f0 + 4096)
        part = mlxq.swiglu(x, tuple(t[f0:f1].contiguous() for t in g), tuple(t[f0:f1].contiguous() for t in u), gs, bits)
        assert torch.equal(h[:, f0:f1], part)


@pytest.mark.parametrize("K,N,valu", [(800, 14530, True), (1248, 12288, True), (32, 12300, True), (1248, 12287, False), (1280, 14530, False)])
def test_one_row_q8_ragged_k(mlxq, K, N, valu):
    """One Q8 row whose K ends inside a load step runs on the VALU kernel from 48 weight rows per CU on
    (256 CUs); either kernel is within half a bf16 ulp and the f32 sums of the exact product."""
    banner("one row q8 ragged", K, N)
    p = _pack(K, N, K, 32, 8)
    x = torch.randn((1, K), device="cuda").to(torch.bfloat16)
    y = mlxq.quantized_matmul(x, *p, True, 32, 8)
    w, mag = _dense(p, 32, 8)
    want = x.double() @ w.t().contiguous()
    bound = (K + 64) * 2.0 ** -24 * (x.double().abs() @ mag.t().contiguous()) + 2.0 ** -8 * want.abs()
    assert bool(((y.double() - want).abs() <= bound).all())
    if valu:
        assert torch.equal(y, mlxq.qmv_valu(x, *p, 32, 8))
