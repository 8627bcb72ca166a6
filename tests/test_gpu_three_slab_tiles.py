"""The tiles of which LDS holds three slabs and more (variants 10 .. 15 of the bf16 GEMM, three of them of the fp8 one): the bits of the 256-row
tiles at the edges of tiles, slabs and of their ring, K in parts, epilogues, and the plan that chooses them."""
import ctypes

import pytest
import torch

from dynaflow_amd import _cabi

gpu = pytest.mark.gpu
TILES = [(224, 192), (160, 256), (128, 256), (192, 192), (128, 192), (128, 128)]
VARIANTS, FP8_VARIANTS = list(range(10, 16)), (11, 12, 15)


def randn(shape, seed, std=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(shape, generator=g, device="cuda") * std).bfloat16()


def spread(shape, seed):
    """Values over many binades: the order of fp32 sums shows in some of the results."""
    return randn(shape, seed) * torch.exp2(randn(shape, seed + 50, 4.0))


def bf16_tiles(x, w, variant, split_k=1, residual=None, workspace=None):
    lib, (M, K), N = _cabi.load(), x.shape, w.shape[0]
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    if split_k > 1 and workspace is None:
        workspace = torch.zeros(lib.dfhip_gemm_bf16_tiles_workspace_bytes(M, N, variant, split_k), dtype=torch.uint8,
                                device="cuda")
    assert lib.dfhip_gemm_bf16_nt_tiles(
        x.data_ptr(), K, w.data_ptr(), K, residual.data_ptr() if residual is not None else None, out.data_ptr(), N, M, N, K,
        variant, split_k, workspace.data_ptr() if split_k > 1 else None, workspace.numel() if split_k > 1 else 0,
        torch.cuda.current_stream().cuda_stream) == 0
    return out


def test_plans_and_arguments():
    """Every planned variant can be launched as planned; what is not such a tile, or has no room for its parts, is refused."""
    lib, v, s = _cabi.load(), ctypes.c_int(), ctypes.c_int()
    seen = set()
    for M in (1, 17, 33, 64, 128, 129, 200, 300, 420, 560, 670, 777, 1100, 1337, 1554, 2048, 2880, 4096):
        for N, K in ((14336, 4096), (4096, 14336), (6144, 4096), (28672, 8192), (8192, 28672), (2048, 5632), (264, 512)):
            for share in (1, 2, 4):
                for may_split in (0, 1):
                    assert lib.dfhip_gemm_bf16_plan_tiles(M, N, K, share, may_split, ctypes.byref(v), ctypes.byref(s)) == 0
                    assert (s.value == 1 or may_split) and 1 <= s.value <= 16
                    if v.value >= 10:
                        assert M > 128 and K // 64 >= 8 * (s.value - 1)
                        assert (lib.dfhip_gemm_bf16_tiles_workspace_bytes(M, N, v.value, s.value) > 0) == (s.value > 1)
                    seen.add(v.value)
                    if K % 128 == 0:
                        assert lib.dfhip_gemm_fp8_plan_tiles(M, N, K, share, may_split, ctypes.byref(v), ctypes.byref(s)) == 0
                        assert s.value == 1 or (may_split and K > N)
                        if s.value > 1:
                            assert lib.dfhip_gemm_fp8_splitk_workspace_bytes(M, N, v.value, s.value) > 0
    assert set(VARIANTS) & seen and 0 in seen and 8 in seen
    ok = (16, 64, 16, 64, None, 16, 8, 1, 8, 64)
    assert lib.dfhip_gemm_bf16_nt_tiles(*ok, 9, 1, None, 0, None) == -7
    assert lib.dfhip_gemm_bf16_nt_tiles(*ok, 16, 1, None, 0, None) == -7
    assert lib.dfhip_gemm_bf16_nt_tiles(*ok, 10, 2, None, 0, None) == -7             # one slab in two parts
    two = (16, 128, 16, 128, None, 16, 8, 1, 8, 128)
    assert lib.dfhip_gemm_bf16_nt_tiles(*two, 10, 2, None, 0, None) == -1
    assert lib.dfhip_gemm_bf16_nt_tiles(*two, 10, 2, 16, 64, None) == -7
    assert lib.dfhip_gemm_bf16_nt_tiles(None, *ok[1:], 10, 1, None, 0, None) == -1
    assert lib.dfhip_gemm_bf16_plan_tiles(64, 64, 64, 0, 1, ctypes.byref(v), ctypes.byref(s)) == -7
    assert lib.dfhip_gemm_fp8_plan_tiles(64, 64, 0, 1, 1, ctypes.byref(v), ctypes.byref(s)) == -2


@gpu
@pytest.mark.parametrize("slabs", [1, 2, 3, 4, 7, 12])
@pytest.mark.parametrize("variant", VARIANTS)
def test_tiles_have_the_bits_of_256_rows(variant, slabs):
    """One row, a row less and more than a tile and columns past one; fewer slabs than the ring holds, as many and more."""
    from dynaflow_amd import ops

    rows, cols = TILES[variant - 10]
    for M, N in ((1, 8), (rows - 1, cols + 8), (2 * rows + 1, cols - 8)):
        x, w = spread((M, 64 * slabs), 1), spread((N, 64 * slabs), 2)
        want = ops.linear_variant(x, w, 0)
        assert torch.equal(ops.linear_variant(x, w, variant), want)
        r = randn((M, N), 3)
        assert torch.equal(bf16_tiles(x, w, variant, residual=r), want + r)
        if variant not in FP8_VARIANTS:
            continue
        xq, wq = ((t.float() / t.float().abs().max() * 448).to(torch.float8_e4m3fn)
                  for t in (spread((M, 128 * slabs), 4), spread((N, 128 * slabs), 5)))
        xs, ws = torch.full((1,), 0.01, device="cuda"), torch.rand((N,), device="cuda")
        assert torch.equal(ops.linear_fp8_variant(xq, wq, xs, ws, variant), ops.linear_fp8_variant(xq, wq, xs, ws, 0))


@gpu
@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("split_k", [2, 3, 5, 16])
def test_parts_of_k(variant, split_k):
    """Against the fp32 product: the bf16 rounding of the result (2^-8 of it) and the fp32 sums; the same bits in every run on
    the same workspace, whose counters are left at zero."""
    lib, (rows, cols) = _cabi.load(), TILES[variant - 10]
    M, N, K = rows + 3, 2 * cols + 8, 128 * (2 * split_k + 1)
    x, w = randn((M, K), 1), randn((N, K), 2, 0.05)
    want = x.float() @ w.float().t()
    ws = torch.zeros(lib.dfhip_gemm_bf16_tiles_workspace_bytes(M, N, variant, split_k), dtype=torch.uint8, device="cuda")
    runs = [bf16_tiles(x, w, variant, split_k, workspace=ws) for _ in range(3)]
    assert (runs[0].float() - want).abs().max().item() <= 2.0 ** -7 * want.abs().max().item()
    assert torch.equal(runs[0], runs[1]) and torch.equal(runs[0], runs[2]) and not ws[:4096].any()
    r = randn((M, N), 3)
    assert torch.equal(bf16_tiles(x, w, variant, split_k, residual=r, workspace=ws), runs[0] + r)
    if variant not in FP8_VARIANTS:
        return
    xq, wq = (x.float() * 16).to(torch.float8_e4m3fn), (w.float() * 256).to(torch.float8_e4m3fn)
    xs, wsc = torch.full((1,), 0.1, device="cuda"), torch.full((N,), 0.01, device="cuda")
    want = xq.float() @ wq.float().t() * 1e-3
    nbytes = lib.dfhip_gemm_fp8_splitk_workspace_bytes(M, N, variant, split_k)
    assert nbytes <= ws.numel()
    for _ in range(2):
        out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert lib.dfhip_gemm_fp8_nt_splitk(
            xq.data_ptr(), K, wq.data_ptr(), K, out.data_ptr(), N, xs.data_ptr(), wsc.data_ptr(), M, N, K, variant, split_k,
            ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream) == 0
        assert (out.float() - want).abs().max().item() <= 2.0 ** -7 * want.abs().max().item()


@gpu
@pytest.mark.parametrize("M,I,K", [(300, 5632, 1024), (400, 5632, 1024), (670, 5640, 1024), (1337, 5632, 512), (777, 14336, 512),
                                   (96, 14336, 1024), (200, 14336, 512), (48, 14336, 4096)])
def test_gate_up_silu_epilogues(M, I, K):
    """bf16 and fp8 gate + up + SiLU*mul at sizes where such tiles are planned: the bits of the separate launches."""
    from dynaflow_amd import ops

    x, w, up = randn((M, K), 3), randn((I, K), 4, 0.05), randn((I, K), 5, 0.05)
    xq, xs = ops.quant_fp8(spread((M, K), 6))
    (wq, ws), (uq, us) = (((t.float() / t.float().abs().max() * 448).to(torch.float8_e4m3fn), torch.rand((I,), device="cuda"))
                          for t in (spread((I, K), 7), spread((I, K), 8)))
    for share in (1, 2):
        with ops.launch_options(share):
            separate = ops.silu_mul(ops.linear_variant(x, w, -2), ops.linear_variant(x, up, -2), True)
            assert torch.equal(ops.gate_up_silu(x, w, up), separate)
            q, scale = ops.gate_up_silu_quant_fp8(xq, wq, uq, xs, ws, us)
            want_q, want_scale = ops.silu_mul_quant_fp8(ops.linear_fp8(xq, wq, xs, ws), ops.linear_fp8(xq, uq, xs, us))
            assert torch.equal(scale, want_scale) and torch.equal(q.view(torch.uint8), want_q.view(torch.uint8))
