"""The fp8 ring tiles of 256, 192 and 128 rows, and K cut into parts that meet in a workspace."""
import ctypes

import pytest
import torch

from dynaflow_amd import _cabi

F8 = torch.float8_e4m3fn


def randn(shape, seed, std=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(shape, generator=g, device="cuda") * std).bfloat16()


def operands(M, N, K):
    from dynaflow_amd import ops
    from dynaflow_amd.fp8_mlp import quantize_weight_per_channel

    xq, xs = ops.quant_fp8(randn((M, K), 1))
    return (xq, *quantize_weight_per_channel(randn((N, K), 2, 0.05)), xs)


def test_planned_fp8_splits_are_launchable():
    """Every plan names a kernel and a split that the entry points take, and only projections with K > N are cut."""
    lib, v, s = _cabi.load(), ctypes.c_int(), ctypes.c_int()
    cut = 0
    for M in (1, 16, 64, 65, 128, 129, 192, 193, 350, 700, 1024, 2048, 5000):
        for N, K in ((8192, 28672), (28672, 8192), (4096, 14336), (14336, 4096), (8, 128), (264, 1152), (2048, 4096)):
            for share in (1, 2, 4, 16):
                assert lib.dfhip_gemm_fp8_plan_shared(M, N, K, share, ctypes.byref(v), ctypes.byref(s)) == 0
                assert v.value in (-1, 0, 1, 2, 3, 4) and 1 <= s.value <= 16
                if s.value > 1:
                    cut += 1
                    assert K > N and K // 128 >= 8 * s.value
                    assert lib.dfhip_gemm_fp8_splitk_workspace_bytes(M, N, v.value, s.value) > 0
    assert cut > 20
    assert lib.dfhip_gemm_fp8_splitk_workspace_bytes(100, 256, 1, 2) == 0       # a kernel that does not split
    args = (16, 1024, 16, 1024, 16, 8, 16, 16, 1, 8, 1024)
    assert lib.dfhip_gemm_fp8_nt_splitk(*args, 4, 2, None, 0, None) == -1       # no workspace
    assert lib.dfhip_gemm_fp8_nt_splitk(*args, 4, 2, 16, 100, None) == -7       # too small
    assert lib.dfhip_gemm_fp8_nt_splitk(*args, 1, 2, 16, 1 << 30, None) == -7   # not a ring tile
    assert lib.dfhip_gemm_fp8_nt_splitk(*args, 4, 5, 16, 1 << 30, None) == -7   # less than two slabs a part


# rows at the edges of 128, 192 and 256-row tiles, ragged columns, 1 slab of K, an odd number, an even one
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 8, 128), (65, 264, 384), (128, 256, 256), (129, 520, 640), (192, 1032, 1152),
                                   (193, 264, 384), (385, 1544, 1024)])
@pytest.mark.parametrize("variant", [0, 3, 4])
def test_fp8_tile_heights_add_in_one_order(M, N, K, variant):
    from dynaflow_amd import ops

    xq, wq, ws, xs = operands(M, N, K)
    got = ops.linear_fp8_variant(xq, wq, xs, ws, variant)
    want = (xq.float() * xs) @ (wq.float() * ws[:, None]).t()
    assert (got.float() - want).abs().max().item() <= 2.0 ** -7 * want.abs().max().item()
    assert torch.equal(got, ops.linear_fp8_variant(xq, wq, xs, ws, 1))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(65, 264, 384), (193, 520, 640), (385, 1544, 1024), (300, 4032, 4096)])
def test_fp8_ring_tiles_have_one_order_of_sums(M, N, K):
    """Operands over many binades: fp32 sums of narrow e4m3 data are nearly exact in any order and would not tell."""
    from dynaflow_amd import ops
    from dynaflow_amd.fp8_mlp import quantize_weight_per_channel

    xq, xs = ops.quant_fp8(randn((M, K), 1) * torch.exp2(randn((M, K), 2, 4.0)))
    wq, ws = quantize_weight_per_channel(randn((N, K), 3) * torch.exp2(randn((N, K), 4, 4.0)))
    tall = ops.linear_fp8_variant(xq, wq, xs, ws, 0)
    for variant in (2, 3, 4):
        assert torch.equal(ops.linear_fp8_variant(xq, wq, xs, ws, variant), tall), variant


# parts of two slabs (the shortest), of uneven lengths (9 slabs in 2 and 4 parts, 37 in 16), ragged tiles
@pytest.mark.gpu
@pytest.mark.parametrize("variant", [0, 3, 4])
@pytest.mark.parametrize("M,N,K,split", [(1, 8, 512, 2), (200, 264, 1152, 2), (130, 520, 1152, 4), (390, 1032, 4736, 16),
                                         (512, 2048, 4096, 3)])
def test_fp8_split_launch(M, N, K, split, variant):
    """Against the fp32 product: bf16 rounding of the result (2^-8 of it) and the fp32 sums; the same bits in every run,
    with counters left at zero in between."""
    lib = _cabi.load()
    xq, wq, ws, xs = operands(M, N, K)
    nbytes = lib.dfhip_gemm_fp8_splitk_workspace_bytes(M, N, variant, split)
    workspace = torch.zeros(nbytes, dtype=torch.uint8, device="cuda")
    want = (xq.float() * xs) @ (wq.float() * ws[:, None]).t()
    runs = []
    for _ in range(3):
        out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert lib.dfhip_gemm_fp8_nt_splitk(
            xq.data_ptr(), K, wq.data_ptr(), K, out.data_ptr(), N, xs.data_ptr(), ws.data_ptr(), M, N, K, variant, split,
            workspace.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream) == 0
        runs.append(out)
    assert (runs[0].float() - want).abs().max().item() <= 2.0 ** -7 * want.abs().max().item()
    assert torch.equal(runs[0], runs[1]) and torch.equal(runs[0], runs[2])


@pytest.mark.gpu
@pytest.mark.parametrize("M,I,K", [(65, 1024, 2048), (128, 3592, 512), (180, 2048, 1024), (350, 7168, 384), (600, 264, 640)])
def test_fused_fp8_tile_heights(M, I, K):
    """The fused launch with tiles of 128, 192 and 256 rows: codes and scale of the separate operators."""
    from dynaflow_amd import ops
    from dynaflow_amd.fp8_mlp import quantize_weight_per_channel

    xq, wq, ws, xs = operands(M, I, K)
    uq, us = quantize_weight_per_channel(randn((I, K), 3, 0.05))
    q, scale = ops.gate_up_silu_quant_fp8(xq, wq, uq, xs, ws, us)
    want_q, want_scale = ops.silu_mul_quant_fp8(ops.linear_fp8_variant(xq, wq, xs, ws, 1),
                                                ops.linear_fp8_variant(xq, uq, xs, us, 1))
    assert torch.equal(scale, want_scale) and torch.equal(q.view(torch.uint8), want_q.view(torch.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("M,I,K", [(128, 1024, 4096), (256, 4096, 8192), (350, 1536, 7168)])
def test_fused_fp8_launch_with_an_intermediate_width_below_the_model_width(M, I, K):
    """The planned gate and up launches, whose K > N could be cut, keep the order of sums of the fused one: the same codes
    and scale, alone and side by side, and the same block output.  Operands over many binades, so that the order of the
    fp32 sums shows in some of the results."""
    from dynaflow_amd import ops
    from dynaflow_amd.fp8_mlp import Fp8SwiGLU, quantize_weight_per_channel

    spread = lambda shape, seed: randn(shape, seed) * torch.exp2(randn(shape, seed + 50, 4.0))
    xq, xs = ops.quant_fp8(spread((M, K), 1))
    (wq, ws), (uq, us) = (quantize_weight_per_channel(spread((I, K), seed)) for seed in (2, 3))
    whole = [ops.linear_fp8_variant(xq, w, xs, s, 0) for w, s in ((wq, ws), (uq, us))]
    for share in (1, 2):
        with ops.launch_options(share):
            q, scale = ops.gate_up_silu_quant_fp8(xq, wq, uq, xs, ws, us)
            gate, up = ops.linear_fp8(xq, wq, xs, ws), ops.linear_fp8(xq, uq, xs, us)
        assert torch.equal(gate, whole[0]) and torch.equal(up, whole[1])
        want_q, want_scale = ops.silu_mul_quant_fp8(gate, up)
        assert torch.equal(scale, want_scale) and torch.equal(q.view(torch.uint8), want_q.view(torch.uint8))
    outs = [Fp8SwiGLU.from_weights(spread((I, K), 6), spread((I, K), 7), spread((K, I), 8), fuse_gate_up=fused)(
        spread((M, K), 9)) for fused in (False, True)]
    assert torch.equal(*outs)


# 2^25 weights are 2048 x 16384, 2^27 are 8192 x 16384
@pytest.mark.parametrize("M,N,K,share,may_split,streamed", [
    # whole K: up to 32 rows; alone up to 64 while the weights are fewer than 2^27
    (32, 28672, 8192, 1, 0, True), (33, 28672, 8192, 1, 0, False), (32, 28672, 8192, 2, 0, True), (33, 28672, 8192, 2, 0, False),
    (64, 16376, 8192, 1, 0, True), (64, 16384, 8192, 1, 0, False), (64, 14336, 4096, 1, 0, True), (65, 14336, 4096, 1, 0, False),
    (33, 14336, 4096, 2, 0, False), (64, 4096, 14336, 1, 0, True),
    # K that may be cut, but is not where the output is as wide
    (64, 14336, 4096, 1, 1, True), (32, 8192, 8192, 2, 1, True), (33, 8192, 8192, 2, 1, False),
    # K that is cut: alone up to 32 rows, in pairs up to 16, or 8 from 2^27 weights on; few weights up to 32, alone up to 64
    (32, 8192, 28672, 1, 1, True), (33, 8192, 28672, 1, 1, False), (8, 8192, 28672, 2, 1, True), (9, 8192, 28672, 2, 1, False),
    (8, 8192, 16384, 2, 1, True), (9, 8192, 16384, 2, 1, False), (16, 8184, 16384, 2, 1, True), (17, 8184, 16384, 2, 1, False),
    (16, 4096, 14336, 2, 1, True), (17, 4096, 14336, 2, 1, False), (32, 2040, 16384, 2, 1, True), (33, 2040, 16384, 2, 1, False),
    (64, 2040, 16384, 1, 1, True), (17, 2048, 16384, 2, 1, False), (64, 1536, 7168, 1, 1, True),
    # a short K from 16 rows on
    (15, 8192, 3968, 1, 0, True), (16, 8192, 3968, 1, 0, False), (16, 8192, 4096, 1, 0, True)])
def test_few_rows_are_streamed(M, N, K, share, may_split, streamed):
    """Both sides of every boundary, in the plan that is launched and in the one without the three-slab tiles."""
    lib, v, s = _cabi.load(), ctypes.c_int(), ctypes.c_int()
    assert lib.dfhip_gemm_fp8_plan_tiles(M, N, K, share, may_split, ctypes.byref(v), ctypes.byref(s)) == 0
    assert (v.value < 0) == streamed
    if may_split:
        assert lib.dfhip_gemm_fp8_plan_shared(M, N, K, share, ctypes.byref(v), ctypes.byref(s)) == 0
        assert (v.value < 0) == streamed


def test_fp8_launches_side_by_side_are_planned_as_such():
    """A pair of large launches takes tiles where a lone one streams its weights, and the other way round nowhere."""
    lib, v, s = _cabi.load(), ctypes.c_int(), ctypes.c_int()
    for M, N, K, alone, paired in ((24, 8192, 28672, True, False), (12, 8192, 28672, True, False), (40, 14336, 4096, True, False),
                                   (20, 4096, 14336, True, False), (32, 28672, 8192, True, True), (40, 28672, 8192, False, False)):
        for share, streamed in ((1, alone), (2, paired)):
            assert lib.dfhip_gemm_fp8_plan_tiles(M, N, K, share, K > N, ctypes.byref(v), ctypes.byref(s)) == 0
            assert (v.value < 0) == streamed, (M, N, K, share)
    args = (16, 1024, 16, 1024, 16, 8, 16, 16, 1, 8, 1024)
    assert lib.dfhip_gemm_fp8_nt_shared(*args, 0, None) == -7 and lib.dfhip_gemm_fp8_nt_shared(*args, 17, None) == -7


# streamed, at its edge and beyond; one round of tall tiles instead of two of short ones; an intermediate width below the
# model width on both sides of 2^27 weights
@pytest.mark.gpu
@pytest.mark.parametrize("M,I,K", [(32, 17408, 8192), (33, 17408, 8192), (64, 17408, 8192), (192, 14336, 4096),
                                   (256, 14336, 4096), (40, 8192, 17408), (40, 4096, 8192)])
@pytest.mark.parametrize("share", [1, 2, 16])
def test_fused_fp8_launch_beside_others(M, I, K, share):
    from dynaflow_amd import ops
    from dynaflow_amd.fp8_mlp import quantize_weight_per_channel

    spread = lambda shape, seed: randn(shape, seed) * torch.exp2(randn(shape, seed + 50, 4.0))
    xq, xs = ops.quant_fp8(spread((M, K), 1))
    (wq, ws), (uq, us) = (quantize_weight_per_channel(spread((I, K), seed)) for seed in (2, 3))
    with ops.launch_options(share):
        q, scale = ops.gate_up_silu_quant_fp8(xq, wq, uq, xs, ws, us)
        gate, up = ops.linear_fp8(xq, wq, xs, ws), ops.linear_fp8(xq, uq, xs, us)
    want_q, want_scale = ops.silu_mul_quant_fp8(gate, up)
    assert torch.equal(scale, want_scale) and torch.equal(q.view(torch.uint8), want_q.view(torch.uint8))
    want = (xq.float() * xs) @ (wq.float() * ws[:, None]).t()
    assert (gate.float() - want).abs().max().item() <= 2.0 ** -6 * want.abs().max().item()


@pytest.mark.gpu
def test_fp8_block_cuts_the_projection_back_to_the_model_width():
    """The block's down projection is the launch in parts (which takes the workspace), the caller's plain one is not."""
    from dynaflow_amd import ops
    from dynaflow_amd.fp8_mlp import Fp8SwiGLU

    hidden, inter, x = 1024, 4096, randn((130, 1024), 9)
    model = Fp8SwiGLU.from_weights(randn((inter, hidden), 6, 0.05), randn((inter, hidden), 7, 0.05),
                                   randn((hidden, inter), 8, 0.05))
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    taken = lambda: sum(key[-1] == stream.cuda_stream for key in ops._splitk_workspaces)
    with torch.cuda.stream(stream):
        xq, xs = ops.quant_fp8(x)
        aq, scale = ops.gate_up_silu_quant_fp8(xq, model.w_gate_q, model.w_up_q, xs, model.w_gate_s, model.w_up_s)
        before = taken()
        whole = ops.linear_fp8(aq, model.w_down_q, scale, model.w_down_s)
        assert taken() == before
        y = model(x)
        cut = ops.linear_fp8(aq, model.w_down_q, scale, model.w_down_s, True)
    stream.synchronize()
    assert before == 0 and taken() == 1
    assert torch.equal(y, cut)
    assert (cut.float() - whole.float()).abs().max().item() <= 2.0 ** -7 * whole.float().abs().max().item()


@pytest.mark.gpu
def test_split_launches_of_both_types_share_a_workspace():
    """What an fp8 launch leaves in the workspace of a stream is nothing a bf16 launch takes for a counter."""
    from dynaflow_amd import ops

    xq, wq, ws, xs = operands(130, 1032, 4096)
    x, w = randn((17, 4096), 4), randn((4096, 4096), 5, 0.05)      # 2 parts, up to 256 counters
    want8, want16 = (xq.float() * xs) @ (wq.float() * ws[:, None]).t(), x.float() @ w.float().t()
    for _ in range(2):
        got8, got16 = ops.linear_fp8(xq, wq, xs, ws, True), ops.linear(x, w)
        assert (got8.float() - want8).abs().max().item() <= 2.0 ** -7 * want8.abs().max().item()
        assert (got16.float() - want16).abs().max().item() <= 2.0 ** -7 * want16.abs().max().item()


@pytest.mark.gpu
def test_split_launches_of_more_tiles_than_the_common_counters_share_a_workspace():
    """More than 1024 tiles: their counters lie where a launch of few tiles leaves its partial sums."""
    lib, stream = _cabi.load(), torch.cuda.current_stream().cuda_stream
    few, many = (130, 1032, 4096, 4), (4, 256 * 1030, 512, 2)
    x, w, g = randn((20, 1024), 4), randn((128 * 1030, 1024), 5, 0.05), torch.Generator(device="cuda").manual_seed(6)
    nbytes = max([lib.dfhip_gemm_fp8_splitk_workspace_bytes(M, N, 4, s) for M, N, _, s in (few, many)]
                 + [lib.dfhip_gemm_bf16_splitk_workspace_bytes(20, 128 * 1030, 2)])
    workspace = torch.zeros(nbytes, dtype=torch.uint8, device="cuda")
    for _ in range(2):
        for M, N, K, split in (few, many):
            xq, wq = ((torch.randn(s, generator=g, device="cuda") * 16).to(F8) for s in ((M, K), (N, K)))
            xs, ws = torch.full((1,), 0.01, device="cuda"), torch.full((N,), 0.01, device="cuda")
            out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
            assert lib.dfhip_gemm_fp8_nt_splitk(
                xq.data_ptr(), K, wq.data_ptr(), K, out.data_ptr(), N, xs.data_ptr(), ws.data_ptr(), M, N, K, 4, split,
                workspace.data_ptr(), nbytes, stream) == 0
            want = (xq.float() @ wq.float().t()) * 1e-4
            assert (out.float() - want).abs().max().item() <= 2.0 ** -7 * want.abs().max().item()
        out = torch.full((20, 128 * 1030), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert lib.dfhip_gemm_bf16_nt_splitk(x.data_ptr(), 1024, w.data_ptr(), 1024, out.data_ptr(), 128 * 1030, 20,
                                             128 * 1030, 1024, 2, workspace.data_ptr(), nbytes, stream) == 0
        want = x.float() @ w.float().t()
        assert (out.float() - want).abs().max().item() <= 2.0 ** -7 * want.abs().max().item()


# side by side and cut from 9 to 32 rows: whole K on either side of them, parts of 16 slabs, more parts for narrow outputs, K too short
@pytest.mark.parametrize("M,N,K,share,parts", [
    (8, 8192, 28672, 2, 1), (9, 8192, 28672, 2, 2), (32, 8192, 28672, 2, 2), (33, 8192, 28672, 2, 1), (9, 8192, 28672, 1, 1),
    (12, 4096, 14336, 2, 2), (24, 4096, 4224, 2, 2), (24, 2560, 4096, 2, 2), (24, 2528, 8192, 2, 4), (24, 2048, 4096, 2, 1),
    (24, 1280, 16384, 4, 4), (24, 1248, 16384, 2, 8), (24, 608, 65536, 2, 1), (24, 16384, 16512, 2, 2), (24, 16392, 28672, 2, 1)])
def test_few_rows_in_parts(M, N, K, share, parts):
    lib, v, s = _cabi.load(), ctypes.c_int(), ctypes.c_int()
    assert lib.dfhip_gemm_fp8_plan_tiles(M, N, K, share, 1, ctypes.byref(v), ctypes.byref(s)) == 0
    streamed = v.value < 0 or v.value == 8
    assert s.value == parts if streamed else parts == 1
    if parts > 1:
        assert streamed and lib.dfhip_gemm_fp8_splitk_workspace_bytes(M, N, v.value, parts) > 0
    args = (16, 65536, 16, 65536, 16, 16392, 16, 16)
    assert lib.dfhip_gemm_fp8_nt_splitk(*args, 33, 8192, 28672, 8, 2, 16, 1 << 30, None) == -7     # more than 32 rows
    assert lib.dfhip_gemm_fp8_nt_splitk(*args, 9, 8192, 3968, 8, 2, 16, 1 << 30, None) == -7       # fewer than 16 slabs a part
    assert lib.dfhip_gemm_fp8_nt_splitk(*args, 9, 16392, 28672, 8, 2, 16, 1 << 30, None) == -7     # more tiles than counters
    assert lib.dfhip_gemm_fp8_nt_splitk(*args, 9, 8192, 28672, 8, 2, 16, 4096, None) == -7         # no room for the parts


# rows whose launches are streamed in parts although they stay two: four parts and more all of them, two where whole K would be
# streamed in fewer than 160 workgroups of 32 columns
@pytest.mark.parametrize("N,K,rows", [(8192, 28672, ()), (8192, 16384, ()), (5120, 25600, ()), (5088, 25600, (12, 16)),
                                      (4096, 14336, (12, 16)), (3072, 8192, (12, 16, 17, 24, 32)), (3072, 24576, (12, 16)),
                                      (2048, 16384, (9, 12, 16, 17, 24, 32)), (1280, 16384, (9, 12, 16, 17, 24, 32))])
def test_launches_that_stay_two_are_streamed_in_parts_where_that_pays(N, K, rows):
    """All other plans are those of launches that may become one."""
    lib, v, s = _cabi.load(), ctypes.c_int(), ctypes.c_int()

    def plan(M, share, may_split):
        assert lib.dfhip_gemm_fp8_plan_tiles(M, N, K, share, may_split, ctypes.byref(v), ctypes.byref(s)) == 0
        return v.value, s.value

    for M in (8, 9, 12, 16, 17, 24, 32, 33, 64, 350):
        for share in (1, 2, 4):
            variant, parts = plan(M, share, 2)
            assert ((variant < 0 or variant == 8) and parts > 1) == (share > 1 and M in rows)
            if not (share > 1 and 9 <= M <= 32) or M in rows:
                assert (variant, parts) == plan(M, share, 1)
            else:
                assert plan(M, share, 1)[0] in (-1, 8) and plan(M, share, 1)[1] > 1


# one and two row blocks; tiles of 16, 32 and 64 columns, ragged ones; parts of 16 slabs, of uneven lengths, 16 of them
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,split", [(1, 8, 4096, 2), (16, 1032, 4224, 2), (17, 1032, 8320, 4), (32, 2568, 4224, 2), (9, 5128, 4224, 2),
                                         (31, 264, 33024, 16), (12, 16384, 4096, 2)])
def test_fp8_streamed_in_parts(M, N, K, split):
    """Against the product in float64: half an ulp of the bf16 result (2^-8 of it) and the fp32 sums.  A sum goes through an instruction
    of 128 products, as many of those as a part has slabs, the four waves' sums and those of the parts: at most 128 + K / 128 + 4 +
    `split` roundings, each off by no more than 2^-24 of a partial sum, and none of those larger than the sum of the magnitudes.  The
    same bits in every run."""
    lib = _cabi.load()
    xq, wq, ws, xs = operands(M, N, K)
    want = ((xq.double() * xs.double()) @ (wq.double() * ws.double()[:, None]).t())
    nbytes = lib.dfhip_gemm_fp8_splitk_workspace_bytes(M, N, 8, split)
    workspace = torch.zeros(nbytes, dtype=torch.uint8, device="cuda")
    runs = []
    for variant in (8, -1, 8):
        out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert lib.dfhip_gemm_fp8_nt_splitk(
            xq.data_ptr(), K, wq.data_ptr(), K, out.data_ptr(), N, xs.data_ptr(), ws.data_ptr(), M, N, K, variant, split,
            workspace.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream) == 0
        runs.append(out)
    size = (xq.double().abs() * xs.double()) @ (wq.double().abs() * ws.double()[:, None]).t()
    off = (runs[0].double() - want).abs()
    assert (off <= 2.0 ** -8 * want.abs() + (132 + K // 128 + split) * 2.0 ** -24 * size).all()
    assert torch.equal(runs[0], runs[1]) and torch.equal(runs[0], runs[2])
    assert not workspace[:4096].any()
