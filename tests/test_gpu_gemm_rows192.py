"""The 192 x 256 tiles of the bf16 GEMM (variant 9): same bits as the 256 x 256 ones, at the edges of tiles and slabs."""
import ctypes

import pytest
import torch

from dynaflow_amd import _cabi

gpu = pytest.mark.gpu


def randn(shape, seed, std=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(shape, generator=g, device="cuda") * std).bfloat16()


def plan(M, N, K, share=1):
    v, s = ctypes.c_int(), ctypes.c_int()
    assert _cabi.load().dfhip_gemm_bf16_plan_shared(M, N, K, share, ctypes.byref(v), ctypes.byref(s)) == 0
    return v.value, s.value


def test_where_the_192_row_tiles_are_planned():
    """Fewer of the shorter rounds; never where K is split; a shape that 256 rows cut evenly keeps its tiles."""
    assert plan(670, 14336, 4096) == (9, 1) and plan(2331, 4096, 14336) == (9, 1)
    assert plan(777, 14336, 4096) == (5, 1) and plan(1554, 4096, 14336) == (0, 2)
    for M, N, K in ((2048, 14336, 4096), (4096, 14336, 4096), (8192, 6144, 4096), (8192, 4096, 14336)):
        for share in (1, 2):
            assert plan(M, N, K, share)[0] != 9


@gpu
@pytest.mark.parametrize("M,N,K", [(1, 8, 64), (95, 136, 128), (97, 264, 192), (192, 256, 64), (193, 520, 256),
                                   (385, 1032, 320), (670, 14336, 1024)])
def test_192_row_tiles_have_the_bits_of_256(M, N, K):
    """One row, half a tile and one row more, whole tiles, one row past them; columns ragged in the first and the second
    half of a tile; K of one slab, two, and more than the ring holds.  The order of K is the same, so are the bits."""
    from dynaflow_amd import ops

    x, w = randn((M, K), 1), randn((N, K), 2, 0.05)
    y = ops.linear_variant(x, w, 9)
    want = x.float() @ w.float().t()
    assert (y.float() - want).abs().max().item() <= 2.0 ** -7 * want.abs().max().item()
    assert torch.equal(y, ops.linear_variant(x, w, 0))


@gpu
@pytest.mark.parametrize("M,N,K", [(670, 12288, 1024), (300, 14336, 1024), (7, 264, 320)])
def test_planned_192_row_tiles_with_epilogues(M, N, K):
    """Residual (670 rows: planned) and SiLU*mul epilogues against the separate 256-row launches, bit for bit."""
    from dynaflow_amd import ops

    x, w, up = randn((M, K), 3), randn((N, K), 4, 0.05), randn((N, K), 5, 0.05)
    if M == 670:
        assert plan(M, N, K) == (9, 1)
        r = randn((M, N), 6)
        assert torch.equal(ops.linear_add(x, w, r), r + ops.linear_variant(x, w, 0))
    separate = ops.silu_mul(ops.linear_variant(x, w, 0), ops.linear_variant(x, up, 0), True)
    assert torch.equal(ops.gate_up_silu(x, w, up), separate)
