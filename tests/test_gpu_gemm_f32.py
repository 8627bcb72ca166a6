"""The fp32 GEMM over its tile shapes, through the operator."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# one shape or more for each tile the cost rule picks (1 x 1 .. 4 x 4 blocks, one round of workgroups and several), ragged
# rows and columns, outputs whose rows are not 16-byte aligned (N = 7, 2815), K at the edges of the split kernel's range:
# 224 (below it), 252 and 260 (no whole slabs), 256 (two slabs a wave), 288 and 544 (an uneven share)
@pytest.mark.parametrize("M,N,K", [(1, 1, 256), (5, 7, 288), (16, 2816, 256), (17, 33, 544), (50, 2815, 1024),
                                   (128, 1024, 2816), (128, 2816, 1024), (131, 2816, 512), (128, 5632, 288),
                                   (256, 5632, 512), (300, 2000, 544), (1000, 2047, 256), (1024, 5632, 512),
                                   (64, 64, 224), (64, 64, 252), (70, 65, 260)])
def test_gemm_f32_tiles(M, N, K):
    """|error| <= K 2^-24 (|A| |W|^T) element by element: what any order of K fp32 products and sums stays within."""
    from dynaflow_amd import ops

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g, device="cuda")
    w = torch.randn(N, K, generator=g, device="cuda")
    got = ops.linear(a, w)
    bound = K * 2.0 ** -24 * (a.double().abs() @ w.double().abs().t())
    assert bool(((got.double() - a.double() @ w.double().t()).abs() <= bound).all())
    assert torch.equal(ops.linear(a, w), got)


# (rows, columns, K, launches side by side, whether the 128 x 128 tiles take it): both sides of the line between them
@pytest.mark.parametrize("M,N,K,share,tile128", [(8192, 2816, 512, 1, True), (3000, 2816, 512, 1, True),
                                                 (3000, 5632, 1024, 1, True), (2816, 2816, 1024, 2, True),
                                                 (1024, 5632, 1024, 2, True), (3000, 2816, 1024, 1, False),
                                                 (512, 5632, 2048, 2, False), (256, 2816, 1024, 2, False)])
def test_gemm_f32_of_many_rows(M, N, K, share, tile128):
    """Against float64 as above.  The 128 x 128 kernel is known by its bits: it also takes a K that is no multiple of 32,
    and four columns of zeros at the end of K change none of its sums."""
    from dynaflow_amd import ops

    g = torch.Generator(device="cuda").manual_seed(M + K)
    a = torch.randn(M, K, generator=g, device="cuda")
    w = torch.randn(N, K, generator=g, device="cuda")
    with ops.launch_options(share):
        got = ops.linear(a, w)
    bound = K * 2.0 ** -24 * (a[::97].double().abs() @ w.double().abs().t())
    assert bool(((got[::97].double() - a[::97].double() @ w.double().t()).abs() <= bound).all())
    padded = ops.linear(*(torch.nn.functional.pad(t, (0, 4)) for t in (a, w)))
    assert torch.equal(got, padded) == tile128


# one round of each tile, ragged in both directions, with the shortest K, an uneven share of the waves, and rows that are not contiguous
@pytest.mark.parametrize("share", [1, 2, 16])
@pytest.mark.parametrize("M,N,K", [(1, 9, 256), (17, 1409, 512), (33, 2817, 1056), (100, 1030, 2816), (130, 520, 288), (200, 2810, 1024),
                                   (250, 4090, 800), (515, 2040, 544)])
def test_gemm_f32_lanes_in_pairs(M, N, K, share):
    """Against the product in float64: a wave sums K / 4 products (and up to a slab more than the others) and the four sums meet, each
    rounding off by no more than 2^-24 of a partial sum of the magnitudes."""
    from dynaflow_amd import ops

    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn((M, K + 4), generator=g, device="cuda")[:, :K]
    w = torch.randn((N, K + 8), generator=g, device="cuda")[:, :K]
    with ops.launch_options(share):
        got = ops.linear(x, w)
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    assert ((got.double() - want).abs() <= (K // 4 + 36) * 2.0 ** -24 * size).all()
