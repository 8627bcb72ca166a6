"""The weight-streaming GEMMs for a few activation rows (up to 64), bf16 and fp8, through the operators."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def randn(shape, seed, std=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(shape, generator=g, device="cuda") * std).bfloat16()


# rows at the edges of the 16 / 32 / 64-row forms; columns that leave a block of 16 or a 64-column tile ragged; K of 16,
# 17, 33 and 37 slabs of 64 (an uneven share per wave) and lengths that are cut into 2, 4 and 8 parts; the first K below
# the kernel's range
@pytest.mark.parametrize("M,N,K", [(1, 8, 1024), (2, 24, 1088), (15, 1032, 1024), (16, 136, 2112), (17, 4096, 4096),
                                   (20, 4088, 2368), (32, 6144, 4096), (33, 264, 2048), (48, 14336, 2048),
                                   (64, 4096, 8192), (7, 4096, 14336), (64, 8, 8192), (64, 10248, 2112), (3, 16, 960)])
def test_few_row_bf16_launches(M, N, K):
    """`linear` against the fp32 product (2^-7 of the largest output: the output's bf16 rounding and the order of the fp32
    sums), the residual epilogue and the fused gate/up/SiLU launch with the bits of the separate ones, and the same bits
    in a second run (the parts of K meet in any order and are added in one)."""
    from dynaflow_amd import _cabi, ops

    v, s = ctypes.c_int(), ctypes.c_int()
    assert _cabi.load().dfhip_gemm_bf16_plan(M, N, K, ctypes.byref(v), ctypes.byref(s)) == 0
    assert (v.value == 8) == (K >= 1024 and M <= 32)
    x, w, r = randn((M, K), 1), randn((N, K), 2, 0.05), randn((M, N), 3)
    y = ops.linear(x, w)
    want = x.float() @ w.float().t()
    limit = 2.0 ** -7 * want.abs().max().item()
    assert (y.float() - want).abs().max().item() <= limit
    assert (ops.linear_variant(x, w, -2).float() - want).abs().max().item() <= limit
    assert torch.equal(ops.linear(x, w), y)
    if K >= 1024:        # the kernel itself, planned or not
        assert (ops.linear_variant(x, w, 8).float() - want).abs().max().item() <= limit
    assert torch.equal(ops.linear_add(x, w, r), r + y)
    up = randn((N, K), 4, 0.05)
    fused = ops.gate_up_silu(x, w, up)
    assert torch.equal(fused, ops.silu_mul(ops.linear_variant(x, w, -2), ops.linear_variant(x, up, -2), True))


@pytest.mark.parametrize("M,N,K", [(1, 8, 2048), (15, 1032, 2176), (16, 136, 4096), (17, 4096, 4224), (33, 264, 8192),
                                   (64, 10248, 4736), (12, 8192, 28672)])
def test_few_row_fp8_launches(M, N, K):
    """fp8 `linear` against the fp32 product of the dequantised operands (2^-6 of the largest output, as for the other
    fp8 kernels), and the fused launch with the codes and scale of the separate operators."""
    from dynaflow_amd import ops
    from dynaflow_amd.fp8_mlp import quantize_weight_per_channel

    xq, xs = ops.quant_fp8(randn((M, K), 5))
    (wq, ws), (uq, us) = (quantize_weight_per_channel(randn((N, K), seed, 0.05)) for seed in (6, 7))
    y = ops.linear_fp8(xq, wq, xs, ws)
    want = (xq.float() * xs) @ (wq.float() * ws[:, None]).t()
    assert (y.float() - want).abs().max().item() <= 2.0 ** -6 * want.abs().max().item()
    q, scale = ops.gate_up_silu_quant_fp8(xq, wq, uq, xs, ws, us)
    want_q, want_scale = ops.silu_mul_quant_fp8(y, ops.linear_fp8(xq, uq, xs, us))
    assert torch.equal(scale, want_scale) and torch.equal(q.view(torch.uint8), want_q.view(torch.uint8))


# 64-row tiles (33 .. 64 rows; 16 .. 32 with a short K) and the first row that has the 128-row ones; ragged columns, K in
# up to 10 parts
@pytest.mark.parametrize("M,N,K", [(16, 1032, 1088), (33, 1024, 1024), (48, 4096, 14336), (64, 6152, 4096),
                                   (64, 1032, 8192), (57, 14344, 1152), (65, 1032, 8192)])
def test_tiles_of_64_rows(M, N, K):
    """Against the fp32 product (bound as above); the fused launch in both of its forms (lone and beside another one)
    with the bits of the separate launches whose K is whole; rows of a launch of more than 64, whose K is whole, with the
    bits of a launch of few."""
    from dynaflow_amd import ops

    x, w, up, r = randn((M, K), 11), randn((N, K), 12, 0.05), randn((N, K), 13, 0.05), randn((M, N), 14)
    want = x.float() @ w.float().t()
    limit = 2.0 ** -7 * want.abs().max().item()
    for side_by_side in (1, 2):
        with ops.launch_options(side_by_side):
            y = ops.linear(x, w)
            assert (y.float() - want).abs().max().item() <= limit
            assert torch.equal(ops.linear(x, w), y)
            assert torch.equal(ops.linear_add(x, w, r), r + y)
            fused = ops.gate_up_silu(x, w, up)
        whole = [ops.linear_variant(x, t, 6) for t in (w, up)]
        assert (whole[0].float() - want).abs().max().item() <= limit
        assert torch.equal(fused, ops.silu_mul(*whole, True))
    few = x[:40].contiguous()
    assert torch.equal(ops.linear_variant(few, w, 6), whole[0][:40])


# columns of which 256 compute units get uneven shares, the last tile ragged or not, whole and in two parts
@pytest.mark.parametrize("M,N,K", [(1, 12280, 1024), (16, 12288, 1088), (32, 12264, 2048), (17, 6136, 4096), (24, 7720, 2112)])
def test_columns_dealt_unevenly(M, N, K):
    """Within the bound of the other few-row launches of the fp32 product, bf16 and fp8."""
    from dynaflow_amd import ops
    from dynaflow_amd.fp8_mlp import quantize_weight_per_channel

    x, w, r = randn((M, K), 1), randn((N, K), 2, 0.05), randn((M, N), 3)
    want = x.float() @ w.float().t()
    limit = 2.0 ** -7 * want.abs().max().item()
    y = ops.linear(x, w)
    assert (y.float() - want).abs().max().item() <= limit
    assert (ops.linear_variant(x, w, 8).float() - want).abs().max().item() <= limit
    assert torch.equal(ops.linear_add(x, w, r), r + y)
    if K % 128 == 0:
        xq, xs = ops.quant_fp8(x)
        wq, ws = quantize_weight_per_channel(w)
        y = ops.linear_fp8(xq, wq, xs, ws)
        want = (xq.float() * xs) @ (wq.float() * ws[:, None]).t()
        assert (y.float() - want).abs().max().item() <= 2.0 ** -6 * want.abs().max().item()


# 18496 .. 20480 columns are between one and a half and two rounds of the compute units; 16 and 17 rows are one and two blocks
@pytest.mark.parametrize("N,K", [(18944, 3584), (18496, 4096), (20480, 4096)])
def test_the_order_of_sums_is_that_of_the_columns(N, K):
    """Whatever the rows are and whether gate and up come in one launch: the fused launch has the bits of the separate ones,
    and rows of a launch of 17 those of a launch of 16 and of one (bf16 throughout, fp8 where both are streamed).  Operands over
    many binades, so that the order of the fp32 sums shows."""
    from dynaflow_amd import ops
    from dynaflow_amd.fp8_mlp import quantize_weight_per_channel

    spread = lambda shape, seed: randn(shape, seed) * torch.exp2(randn(shape, seed + 50, 4.0))
    x, gate, up = spread((17, K), 1), spread((N, K), 2), spread((N, K), 3)
    fused = {M: ops.gate_up_silu(x[:M], gate, up) for M in (1, 16, 17)}
    for M, got in fused.items():
        assert torch.equal(got, ops.silu_mul(ops.linear(x[:M], gate), ops.linear(x[:M], up), True)), M
        assert torch.equal(got, fused[17][:M]), M
    xq, xs = ops.quant_fp8(x)
    (wq, ws), (uq, us) = quantize_weight_per_channel(gate), quantize_weight_per_channel(up)
    y = {M: ops.linear_fp8(xq[:M], wq, xs, ws) for M in (1, 16, 17)}
    for M in (1, 16, 17):
        q, scale = ops.gate_up_silu_quant_fp8(xq[:M], wq, uq, xs, ws, us)
        want_q, want_scale = ops.silu_mul_quant_fp8(y[M], ops.linear_fp8(xq[:M], uq, xs, us))
        assert torch.equal(scale, want_scale) and torch.equal(q.view(torch.uint8), want_q.view(torch.uint8)), M
        if K >= 4096:
            assert torch.equal(y[M], y[17][:M]), M
