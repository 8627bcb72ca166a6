"""The cell that the fused fp8 launch folds its maximum into belongs to one call: launches on other streams, other forwards of the
same model and other graphs neither fold into it nor clear it."""
import pytest
import torch

from dynaflow_amd import ops
from dynaflow_amd.interface import OperatorHandle
from dynaflow_amd.runtime.env import set_op_handle


class Recorder:
    """Stands in for the kernel library: notes the calls."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        return lambda *args: self.calls.append((name, args)) or 0


def test_every_call_clears_and_folds_into_memory_of_its_own(monkeypatch):
    """Two unsplit forwards of one model, which have the same engine and nano-batch, on two streams."""
    lib, streams = Recorder(), iter((11, 12))
    monkeypatch.setattr(ops._cabi, "load", lambda: lib)
    monkeypatch.setattr(ops, "_require_device", lambda *tensors: None)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    current = [0]
    monkeypatch.setattr(ops, "_stream", lambda: current[0])
    fp8 = lambda *shape: torch.zeros(shape, dtype=torch.uint8).view(ops.FP8_DTYPE)
    one, scales = torch.ones(1), torch.ones(64)
    kept = []
    for current[0] in streams:
        handle = OperatorHandle(module_name="m", batch_idx=0, batch_size=3, tag=set(), _is_dryrun=False,
                                _use_cudagraph=False, _owner=5)
        with set_op_handle(handle):
            kept.append(ops._gate_up_silu_quant_fp8_impl(fp8(3, 128), fp8(64, 128), fp8(64, 128), one, scales, scales))
    per_call = [lib.calls[:len(lib.calls) // 2], lib.calls[len(lib.calls) // 2:]]
    cells = []
    for stream, calls in zip((11, 12), per_call):
        assert all(args[-1] == stream for _, args in calls)
        names = [name for name, _ in calls]
        gemm = names.index("dfhip_gemm_fp8_gate_up_silu_absmax_shared")
        cell = calls[gemm][1][10]
        assert names[:gemm] == ["dfhip_fill_u32"] and calls[0][1][:3] == (cell, 0, 1)     # cleared in front of the fold
        assert [args[6] for name, args in calls[gemm + 1:]] == [cell]                    # read behind it, by one launch
        cells.append(cell)
    assert cells[0] != cells[1]
    inside = [(scale.untyped_storage().data_ptr(), scale.untyped_storage().nbytes()) for _, scale in kept]
    for cell, (at, size) in zip(cells, inside):      # part of a result: it lives as long as that, in a graph's pool too
        assert at <= cell and cell + 4 <= at + size


@pytest.mark.gpu
@pytest.mark.parametrize("M", [9, 40, 300])
def test_graphs_of_one_stream_replayed_on_two(M):
    """Operands whose maxima differ by a factor of 1000: a foreign or an early cleared maximum would show."""
    g = torch.Generator(device="cuda").manual_seed(5)
    wq = [(torch.randn((1024, 2048), generator=g, device="cuda") * 50).to(ops.FP8_DTYPE) for _ in range(2)]
    ws, xs = torch.full((1024,), 0.01, device="cuda"), [torch.full((1,), s, device="cuda") for s in (0.01, 0.0003)]
    xq = [(torch.randn((M + i, 2048), generator=g, device="cuda") * 20).to(ops.FP8_DTYPE) for i in range(2)]
    want = [ops.gate_up_silu_quant_fp8(x, *wq, s, ws, ws) for x, s in zip(xq, xs)]
    graphs, outs = [torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()], []
    for graph, x, s in zip(graphs, xq, xs):
        with torch.cuda.graph(graph):
            outs.append(ops.gate_up_silu_quant_fp8(x, *wq, s, ws, ws))
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for _ in range(20):
        for q, scale in outs:
            q.view(torch.uint8).zero_()
            scale.zero_()
        torch.cuda.synchronize()
        for graph, stream in zip(graphs, streams):
            with torch.cuda.stream(stream):
                for _ in range(3):
                    graph.replay()
        eager = ops.gate_up_silu_quant_fp8(xq[0], *wq, xs[0], ws, ws)       # beside both, on a third stream
        torch.cuda.synchronize()
        for (q, scale), (want_q, want_scale) in zip([*outs, eager], [*want, want[0]]):
            assert torch.equal(scale, want_scale) and torch.equal(q.view(torch.uint8), want_q.view(torch.uint8))
