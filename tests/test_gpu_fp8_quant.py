"""Quantisation without a cell to clear: the codes and scales of the maximum and the quantisation launched one by one, at the
sizes where the kernels change."""
import pytest
import torch

from dynaflow_amd import _cabi

pytestmark = pytest.mark.gpu


def rows(M, D, gap, seed, special=False):
    """[M, D] bf16 whose rows lie `gap` elements apart from another; optionally with infinities, NaN and the largest values."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    t = (torch.randn((M, D + gap), generator=g, device="cuda") * torch.exp2(torch.randn((M, 1), generator=g, device="cuda") * 4))
    t = t.bfloat16()
    if special:
        t.view(-1)[:: max(1, t.numel() // 3)] = float("nan")
    return t[:, :D]


def one_by_one(x):
    lib, s, (M, D) = _cabi.load(), torch.cuda.current_stream().cuda_stream, x.shape
    amax, scale = torch.zeros(1, device="cuda"), torch.zeros(1, device="cuda")
    q = torch.zeros((M, D), dtype=torch.uint8, device="cuda")
    assert lib.dfhip_absmax_bf16(x.data_ptr(), x.stride(0), M, D, amax.data_ptr(), s) == 0
    assert lib.dfhip_quant_fp8_bf16(x.data_ptr(), x.stride(0), q.data_ptr(), D, M, D, amax.data_ptr(), scale.data_ptr(), s) == 0
    return q, scale, amax


# one group; an odd count; a whole block and one group more; as many blocks as count their readers and one more; more than parts
SIZES = [(1, 8), (3, 40), (1, 8192), (1, 8200), (128, 8192), (129, 8192), (4097, 2056)]


@pytest.mark.parametrize("M,D", SIZES)
@pytest.mark.parametrize("gap", [0, 8])
@pytest.mark.parametrize("special", [False, True])
def test_quant_dynamic(M, D, gap, special):
    lib, s = _cabi.load(), torch.cuda.current_stream().cuda_stream
    x = rows(M, D, gap, 1, special)
    want_q, want_scale, _ = one_by_one(x)
    parts = torch.full((1024,), float("inf"), device="cuda")
    scale, q = torch.zeros(1, device="cuda"), torch.zeros((M, D + gap), dtype=torch.uint8, device="cuda")
    assert lib.dfhip_quant_fp8_dynamic_bf16(x.data_ptr(), D + gap, q.data_ptr(), D + gap, M, D, parts.data_ptr(),
                                            scale.data_ptr(), s) == 0
    assert torch.equal(scale, want_scale) and torch.equal(q[:, :D], want_q) and not q[:, D:].any()
    # the same behind a cell, which is zero again afterwards
    cells = torch.zeros(2, device="cuda")
    assert lib.dfhip_absmax_bf16(x.data_ptr(), D + gap, M, D, cells.data_ptr(), s) == 0
    q.zero_()
    assert lib.dfhip_requant_fp8_bf16(x.data_ptr(), D + gap, q.data_ptr(), D + gap, M, D, cells.data_ptr(), scale.data_ptr(),
                                      s) == 0
    assert torch.equal(scale, want_scale) and torch.equal(q[:, :D], want_q) and not cells.view(torch.int32).any()


@pytest.mark.parametrize("M,D", SIZES)
@pytest.mark.parametrize("gap", [0, 16])
def test_silu_mul_quant(M, D, gap):
    lib, s = _cabi.load(), torch.cuda.current_stream().cuda_stream
    g, u = rows(M, D, gap, 2), rows(M, D, gap, 3)
    act, amax = torch.zeros((M, D), dtype=torch.bfloat16, device="cuda"), torch.zeros(1, device="cuda")
    assert lib.dfhip_silu_mul_absmax_bf16(g.data_ptr(), D + gap, u.data_ptr(), D + gap, act.data_ptr(), D, M, D,
                                          amax.data_ptr(), s) == 0
    want_q, want_scale, _ = one_by_one(act)
    got, q = torch.zeros((M, D + gap), dtype=torch.bfloat16, device="cuda"), torch.zeros((M, D), dtype=torch.uint8, device="cuda")
    scale, parts = torch.zeros(1, device="cuda"), torch.full((1024,), float("inf"), device="cuda")
    assert lib.dfhip_silu_mul_quant_fp8_bf16(g.data_ptr(), D + gap, u.data_ptr(), D + gap, got.data_ptr(), D + gap, q.data_ptr(),
                                             D, M, D, parts.data_ptr(), scale.data_ptr(), s) == 0
    assert torch.equal(got[:, :D], act) and not got[:, D:].any()
    assert torch.equal(scale, want_scale) and torch.equal(q, want_q)


def test_fused_launches_of_two_threads_on_one_stream():
    """The maximum of one thread's launch is not another's: the cell is theirs from the fold to the quantisation."""
    import threading

    from dynaflow_amd import ops

    g = torch.Generator(device="cuda").manual_seed(5)
    wq = [(torch.randn((1024, 2048), generator=g, device="cuda") * 50).to(torch.float8_e4m3fn) for _ in range(2)]
    ws, xs = torch.full((1024,), 0.01, device="cuda"), torch.full((1,), 0.01, device="cuda")
    xq = [(torch.randn((M, 2048), generator=g, device="cuda") * 10.0 ** i).to(torch.float8_e4m3fn) for i, M in enumerate((9, 40))]
    want = [ops.gate_up_silu_quant_fp8(x, *wq, xs, ws, ws) for x in xq]
    got = [[], []]

    def work(i):
        got[i] = [ops.gate_up_silu_quant_fp8(xq[i], *wq, xs, ws, ws) for _ in range(40)]

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for i in range(2):
        assert len(got[i]) == 40
        for q, scale in got[i]:
            assert torch.equal(scale, want[i][1]) and torch.equal(q.view(torch.uint8), want[i][0].view(torch.uint8))


# one slab of K and few, where no wave of the launch leaves its maximum apart, and the shortest K where they do
@pytest.mark.parametrize("M,I,K", [(1, 8, 128), (64, 264, 256), (128, 2816, 768), (12, 2816, 896), (24, 1408, 1024), (128, 4104, 1152)])
def test_gate_up_of_few_rows_and_a_short_k(M, I, K):
    """On both sides of the K from which it is one call: the codes and scale of the separate operators, and the entry point by itself."""
    from dynaflow_amd import ops
    from dynaflow_amd.fp8_mlp import quantize_weight_per_channel

    def randn(shape, seed):
        return torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda").bfloat16()

    xq, xs = ops.quant_fp8(randn((M, K), 1))
    (wq, ws), (uq, us) = (quantize_weight_per_channel(randn((I, K), seed)) for seed in (2, 3))
    q, scale = ops.gate_up_silu_quant_fp8(xq, wq, uq, xs, ws, us)
    want_q, want_scale = ops.silu_mul_quant_fp8(ops.linear_fp8(xq, wq, xs, ws), ops.linear_fp8(xq, uq, xs, us))
    assert torch.equal(scale, want_scale) and torch.equal(q.view(torch.uint8), want_q.view(torch.uint8))
    test_gate_up_with_maxima_side_by_side(M, I, K, 1)


# streamed in 16, 32 and 64 columns a workgroup, ragged; three-slab tiles; more workgroups than parts have room for; a ring tile
@pytest.mark.parametrize("M,I,K,share", [(1, 136, 2048, 1), (17, 5120, 4096, 2), (32, 16392, 4096, 1), (128, 14336, 4096, 1), (40, 7176, 4096, 2),
                                         (16, 65544, 2048, 1), (128, 1032, 2048, 16)])
def test_gate_up_with_maxima_side_by_side(M, I, K, share):
    """The codes and the scale of the launch that folds into a cell and the quantisation behind it; parts that hold infinities before."""
    lib, s = _cabi.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device="cuda").manual_seed(M + I)
    x, wg, wu = ((torch.randn(shape, generator=g, device="cuda") * 20).to(torch.float8_e4m3fn) for shape in ((M, K), (I, K), (I, K)))
    xs, ws = torch.full((1,), 0.01, device="cuda"), torch.rand(I, generator=g, device="cuda") * 0.01
    act, amax, scale = torch.empty((M, I), dtype=torch.bfloat16, device="cuda"), torch.zeros(1, device="cuda"), torch.empty(1, device="cuda")
    want, q = (torch.zeros((M, I), dtype=torch.uint8, device="cuda") for _ in range(2))
    weights = (wg.data_ptr(), wu.data_ptr(), K, act.data_ptr(), I)
    scales = (xs.data_ptr(), ws.data_ptr(), ws.data_ptr())
    assert lib.dfhip_gemm_fp8_gate_up_silu_absmax_shared(x.data_ptr(), K, *weights, *scales, amax.data_ptr(), M, I, K, share, s) == 0
    assert lib.dfhip_quant_fp8_bf16(act.data_ptr(), I, want.data_ptr(), I, M, I, amax.data_ptr(), scale.data_ptr(), s) == 0
    want_act, want_scale = act.clone(), scale.clone()
    parts = torch.full((4096,), float("inf"), device="cuda")
    for _ in range(2):
        act.zero_(), scale.zero_()
        assert lib.dfhip_gemm_fp8_gate_up_silu_quant_shared(x.data_ptr(), K, *weights, q.data_ptr(), I, *scales, parts.data_ptr(),
                                                            scale.data_ptr(), M, I, K, share, s) == 0
        assert torch.equal(act, want_act) and torch.equal(scale, want_scale) and torch.equal(q, want)
    assert lib.dfhip_gemm_fp8_gate_up_silu_quant_shared(x.data_ptr(), K, *weights, None, I, *scales, parts.data_ptr(), scale.data_ptr(),
                                                        M, I, K, share, s) == -1
    assert lib.dfhip_gemm_fp8_gate_up_silu_quant_shared(x.data_ptr(), K, *weights, q.data_ptr(), I, *scales, None, scale.data_ptr(),
                                                        M, I, K, share, s) == -1
