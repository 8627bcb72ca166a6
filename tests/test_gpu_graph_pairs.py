"""Launches of two nano-batches against the same weights as one, in a schedule captured as one graph: every replay has the bits
of the eager schedule, and a schedule that is not all of such launches is left as it is."""
import ctypes
import re

import pytest
import torch

from dynaflow_amd import _cabi
from dynaflow_amd.backend import make_backend
from dynaflow_amd.config import CUDAGraphConfig, DynaFlowConfig, InductorConfig
from dynaflow_amd.decode import DecodeModel
from dynaflow_amd.fp8_mlp import Fp8SwiGLU
from dynaflow_amd.manager import DynaFlowManager
from dynaflow_amd.mlp import SwiGLUMLP
from dynaflow_amd.schedulers import MLPOverlapScheduler


def test_arguments():
    pairs = ctypes.c_int(5)
    assert _cabi.load().dfhip_graph_pair_launches(None, 0, ctypes.byref(pairs)) == -1
    assert _cabi.load().dfhip_graph_pair_launches(16, 0, None) == -1


def randn(shape, seed, std=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(shape, generator=g, device="cuda") * std).bfloat16()


def program(model, tokens, scheduler="dynaflow_amd.schedulers:MLPOverlapScheduler", **knobs):
    manager = DynaFlowManager()
    cfg = DynaFlowConfig(scheduler, 4, InductorConfig(enabled=True),
                         CUDAGraphConfig(enabled=False, capture_sizes=[tokens]),
                         {"min_nano_split_tokens": 1, "num_nano_batches": 2, "dump_graph": False, "whole_graph": True,
                          "streams": "by_nano_batch", "fuse_silu_epilogue": True, **knobs})
    x = randn((tokens, model.hidden), 1)
    torch._dynamo.mark_dynamic(x, 0)
    torch._dynamo.reset()
    compiled = torch.compile(model, backend=make_backend(manager, cfg), fullgraph=True)
    with torch.no_grad():
        manager.prepare(tokens, [tokens])
        compiled(x)
    return manager, compiled


def forward(manager, compiled, x, graph):
    with torch.no_grad():
        manager.prepare(len(x), [1] * len(x), use_cudagraph=graph)
        return compiled(x)


def mlp(kind, hidden, inter):
    weights = randn((inter, hidden), 2, 0.03), randn((inter, hidden), 3, 0.03), randn((hidden, inter), 4, 0.03)
    if kind == "fp8":
        model = Fp8SwiGLU.from_weights(*weights, fuse_gate_up=True)
    else:
        model = SwiGLUMLP(hidden, inter, dtype=torch.bfloat16, device="cuda")
        with torch.no_grad():
            for layer, w in zip((model.gate_proj, model.up_proj, model.down_proj), weights):
                layer.weight.copy_(w)
    model.hidden = hidden
    return model


# separate gate and up projections pair like the fused one: their product is a short launch; and streams by kind, whose
# order of the launches of a kind is nobody's need
@pytest.mark.gpu
@pytest.mark.parametrize("knobs", [{"fuse_silu_epilogue": False}, {"streams": "by_kind"},
                                   {"streams": "by_kind", "fuse_silu_epilogue": False}])
def test_short_launches_between_pairs_and_streams_by_kind(knobs):
    manager, compiled = program(mlp("bf16", 2048, 5632), 64, **knobs)
    x = randn((64, 2048), 5)
    want = forward(manager, compiled, x, False).clone()
    for _ in range(3):
        assert torch.equal(forward(manager, compiled, x, True), want)
    assert list(manager.paired_launches.values()) == [2]


# streamed weights, the rows of both in one to four blocks of 16; rows of the two nano-batches that differ; tiles of 64 and 128 rows; a grid that is no multiple of eight
@pytest.mark.gpu
@pytest.mark.parametrize("kind,tokens,hidden,inter", [
    ("bf16", 2, 2048, 5632), ("bf16", 16, 2048, 5632), ("bf16", 25, 2048, 5696), ("bf16", 35, 2048, 5632),
    ("bf16", 48, 4096, 14336), ("bf16", 64, 4096, 14336), ("bf16", 96, 2048, 5696),
    ("bf16", 255, 4096, 14336), ("fp8", 9, 4096, 14336), ("fp8", 24, 4096, 14336), ("fp8", 29, 2048, 5760), ("fp8", 80, 8192, 8192),
    ("fp8", 190, 4096, 14336)])
def test_paired_replays_have_the_bits_of_the_eager_schedule(kind, tokens, hidden, inter):
    manager, compiled = program(mlp(kind, hidden, inter), tokens)
    x = randn((tokens, hidden), 5)
    forward(manager, compiled, x, True)
    assert list(manager.paired_launches.values()) == [2], manager.paired_launches
    for seed in (6, 7, 8):
        x = randn((tokens, hidden), seed, 2.0 ** (seed - 6))
        want = forward(manager, compiled, x, False).clone()
        torch.cuda.synchronize()
        for _ in range(2):
            got = forward(manager, compiled, x, True)
            assert torch.equal(got, want)


class LongBeside(torch.nn.Module):
    """An fp8 layer beside a kernel of many workgroups that has no launch of two."""

    def __init__(self, hidden, inter):
        super().__init__()
        self.layer, self.hidden = mlp("fp8", hidden, inter), hidden
        self.register_buffer("table", randn((4096, hidden), 9).float())

    def forward(self, x):
        return self.layer(x) + (self.table * 2)[7].bfloat16()


@pytest.mark.gpu
def test_launches_that_turn_out_to_stay_two_are_planned_as_such():
    """The first capture finds no pairs: the schedule is captured again with the plans of launches that stay apart."""
    manager, compiled = program(LongBeside(4096, 14336), 24)
    x = randn((24, 4096), 5)
    split = manager.prepare(24, [1] * 24)
    assert manager.launches_join(split)
    forward(manager, compiled, x, True)
    assert list(manager.paired_launches.values()) == [0] and not manager.launches_join(split)
    want = forward(manager, compiled, x, False).clone()
    for _ in range(3):
        assert torch.equal(forward(manager, compiled, x, True), want)


@pytest.mark.gpu
def test_ranks_keep_their_schedule(monkeypatch):
    """Collectives are kernels of few workgroups: with several ranks nothing is put in line."""
    monkeypatch.setattr(torch.distributed, "is_initialized", lambda: True)
    monkeypatch.setattr(torch.distributed, "get_world_size", lambda: 2)
    manager, compiled = program(mlp("bf16", 2048, 5632), 64)
    x = randn((64, 2048), 5)
    want = forward(manager, compiled, x, False).clone()
    assert torch.equal(forward(manager, compiled, x, True), want)
    assert list(manager.paired_launches.values()) == [0]


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,knobs", [(64, {"pair_launches": False}), (64, {"streams": "by_kind", "pair_launches": False}),
                                          (64, {"streams": "by_kind", "serialize": True}), (1024, {}),
                                          (1024, {"streams": "by_kind"}), (96, {"num_nano_batches": 3})])
def test_other_schedules_stay_as_they_are(tokens, knobs):
    """Switched off, one stream, many rows, a launch without a partner."""
    manager, compiled = program(mlp("bf16", 2048, 5632), tokens, **knobs)
    x = randn((tokens, 2048), 5)
    want = forward(manager, compiled, x, False).clone()
    for _ in range(3):
        assert torch.equal(forward(manager, compiled, x, True), want)
    assert list(manager.paired_launches.values()) == [0]


class WritesBetween(SwiGLUMLP):
    """Each nano-batch leaves its first row in one buffer and adds it to its result."""

    def __init__(self, hidden, inter):
        super().__init__(hidden, inter, dtype=torch.bfloat16, device="cuda")
        self.hidden = hidden
        self.register_buffer("first", torch.zeros(hidden, dtype=torch.bfloat16, device="cuda"))

    def forward(self, x):
        y = super().forward(x)
        self.first.copy_(x[0])
        return y + self.first


@pytest.mark.gpu
def test_a_buffer_of_both_nano_batches_keeps_the_order_of_the_schedule():
    """Streams by kind run the two writers one after the other, each in front of its reader; so does the captured schedule."""
    model = WritesBetween(2048, 5632)
    with torch.no_grad():
        for p, (shape, seed) in zip(model.parameters(), (((5632, 2048), 2), ((5632, 2048), 3), ((2048, 5632), 4))):
            assert tuple(p.shape) == shape
            p.copy_(randn(shape, seed, 0.03))
    manager, compiled = program(model, 64, streams="by_kind")
    for seed in (5, 6):
        x = randn((64, 2048), seed)
        want = forward(manager, compiled, x, False).clone()
        for _ in range(3):
            assert torch.equal(forward(manager, compiled, x, True), want)
    assert list(manager.paired_launches.values()) == [0]


class OwnSchedule(MLPOverlapScheduler):
    async def schedule(self, context):
        await super().schedule(context)


@pytest.mark.gpu
@pytest.mark.parametrize("streams", ["by_kind", "by_nano_batch"])
def test_a_scheduler_of_its_own_keeps_its_schedule(streams):
    manager, compiled = program(mlp("bf16", 2048, 5632), 64, "test_gpu_graph_pairs:OwnSchedule", streams=streams)
    x = randn((64, 2048), 5)
    want = forward(manager, compiled, x, False).clone()
    assert torch.equal(forward(manager, compiled, x, True), want)
    assert list(manager.paired_launches.values()) == [0]


# ------------------------------------------------------------------------------------------------ decode steps
def decode_program(T, capacity, streams, hidden=4096, heads=32, kv_heads=8, inter=4096, layers=2):
    model = DecodeModel(layers=layers, vocab=512, hidden=hidden, heads=heads, kv_heads=kv_heads, inter=inter, slots=T + 3,
                        capacity=capacity, dtype=torch.bfloat16, device="cuda")
    with torch.no_grad():
        for seed, p in enumerate(model.parameters()):
            if p.dim() > 1:
                p.copy_(randn(p.shape, 20 + seed, 1.0 if p is model.embed else 0.03))
        for block in model.attn:
            block.k_cache.copy_(randn(block.k_cache.shape, 60))
            block.v_cache.copy_(randn(block.v_cache.shape, 61))
    manager = DynaFlowManager()
    cfg = DynaFlowConfig("dynaflow_amd.schedulers:DecoderOverlapScheduler", 2, InductorConfig(enabled=True),
                         CUDAGraphConfig(enabled=False, capture_sizes=[T // 2, T - T // 2, T]),
                         {"min_nano_split_tokens": 1, "dump_graph": False, "whole_graph": True, "streams": streams,
                          "fuse_silu_epilogue": True})
    step = step_inputs(T, capacity, 1)
    torch._dynamo.reset()
    for t in step:
        torch._dynamo.mark_dynamic(t, 0)
    compiled = torch.compile(model, backend=make_backend(manager, cfg), fullgraph=True)
    with torch.no_grad():
        manager.prepare(T, [1] * T)
        compiled(*step)
    return model, manager, compiled


def step_inputs(T, capacity, seed):
    """Sequences of 1 to `capacity` positions, the shortest and the longest among them, in slots of any order."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    lengths = torch.randint(1, capacity + 1, (T,), generator=g, device="cuda").int()
    lengths[T // 3], lengths[-1] = 1, capacity
    return [torch.randint(0, 512, (T,), generator=g, device="cuda"),
            torch.randperm(T + 3, generator=g, device="cuda")[:T].int(), lengths]


def step(manager, compiled, inputs, graph):
    with torch.no_grad():
        manager.prepare(len(inputs[0]), [1] * len(inputs[0]), use_cudagraph=graph)
        return compiled(*inputs).clone()


def launches(manager, tmp_path):
    """The kernels of the one captured schedule, by name."""
    (entry,) = manager._schedule_graphs.values()
    entry.graph.debug_dump(str(tmp_path / "graph.dot"))
    return (tmp_path / "graph.dot").read_text()


# attention uncut on both sides; cut on both, in 8 and 7 parts (8 and 9 tokens) and in 3 and 4 (21 and 22 tokens: o and down
# projections of both sides with their residuals and K in parts, as one launch); 64 rows on tiles
@pytest.mark.gpu
@pytest.mark.parametrize("T,capacity,cut", [(43, 512, False), (17, 2048, True), (43, 4096, True), (2, 2048, True), (128, 256, False)])
@pytest.mark.parametrize("streams", ["by_kind", "by_nano_batch"])
def test_decode_steps_in_pairs(T, capacity, cut, streams, tmp_path):
    """Results and caches of every replay are those of the eager schedule: projections, norms and attention of the two
    nano-batches in one launch each."""
    model, manager, compiled = decode_program(T, capacity, streams)
    caches = [c for block in model.attn for c in (block.k_cache, block.v_cache)]
    step(manager, compiled, step_inputs(T, capacity, 2), True)
    assert list(manager.paired_launches.values()) == [4 * 2], manager.paired_launches
    names = launches(manager, tmp_path)
    assert names.count(f"DecodeAttentionOfILb1ELb{int(cut)}E") == 2 and len(re.findall(r"beside_kernel\w+7RmsNorm", names)) == 4
    if T == 43:          # K in parts and the rows of both sides: q/k/v, o and down of both layers
        assert len(re.findall(r"gemm_stream_kernelILb0ELi\dELi\dELi\dELb0ELb1ELb1E", names)) >= 4
    for seed in (3, 4):
        inputs = step_inputs(T, capacity, seed)
        before = [c.clone() for c in caches]
        want = step(manager, compiled, inputs, False)
        after = [c.clone() for c in caches]
        for _ in range(2):
            for c, b in zip(caches, before):
                c.copy_(b)
            got = step(manager, compiled, inputs, True)
            assert torch.equal(got, want)
            assert all(torch.equal(c, a) for c, a in zip(caches, after))


# 26 sequences with 20 kv heads are 520 workgroups of attention, the other 25 of 51 are 500
@pytest.mark.gpu
@pytest.mark.parametrize("T,joined", [(50, True), (51, False), (52, False)])
def test_long_attention_of_either_side_keeps_a_schedule_with_a_stream_per_nano_batch(T, joined):
    model, manager, compiled = decode_program(T, 128, "by_nano_batch", hidden=2048, heads=20, kv_heads=20, inter=2048)
    inputs = step_inputs(T, 128, 2)
    want = step(manager, compiled, inputs, False)
    for _ in range(2):
        assert torch.equal(step(manager, compiled, inputs, True), want)
    assert [n > 0 for n in manager.paired_launches.values()] == [joined]


# ------------------------------------------------------------------------------------- graphs that a program captured itself
def captured(first, second):
    """`first` and `second` (lists of calls) on two streams of one graph: its handle, to be replayed after the pairing."""
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for s, calls in zip(streams, (first, second)):           # workspaces are made outside of the capture
        with torch.cuda.stream(s):
            for call in calls:
                call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        start = torch.cuda.current_stream().record_event()
        for s, calls in zip(streams, (first, second)):
            with torch.cuda.stream(s):
                s.wait_event(start)
                for call in calls:
                    call()
                end = s.record_event()
            torch.cuda.current_stream().wait_event(end)
    pairs = ctypes.c_int(-1)
    assert _cabi.load().dfhip_graph_pair_launches(graph.raw_cuda_graph(), 0, ctypes.byref(pairs)) == 0
    graph.instantiate()
    return graph, pairs.value


@pytest.mark.gpu
@pytest.mark.parametrize("order,found", [((0, 1), 2), ((1, 0), 0)])
def test_pairs_that_wait_for_each_other_crosswise_stay(order, found):
    """Two chains through the same two weights: in the same order they pair, in opposite orders no order of two joined launches
    exists."""
    from dynaflow_amd import ops

    w = [randn((1024, 1024), 1 + i, 0.03) for i in range(2)]
    x = [randn((8, 1024), 3 + i) for i in range(2)]
    got = [torch.empty((8, 1024), dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    kept = [[], []]

    def chain(i, way):
        return [lambda: kept[i].append(ops.linear_variant(x[i], w[way[0]], 8)),
                lambda: kept[i].append(ops.linear_variant(kept[i][-1], w[way[1]], 8)),
                lambda: torch.mul(kept[i][-1], 1, out=got[i])]

    want = [ops.linear_variant(ops.linear_variant(x[i], w[way[0]], 8), w[way[1]], 8) for i, way in enumerate(((0, 1), order))]
    graph, pairs = captured(chain(0, (0, 1)), chain(1, order))
    assert pairs == found
    for _ in range(3):
        for g in got:
            g.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.gpu
@pytest.mark.parametrize("between", ["ring", "fp32"])
def test_a_gemm_without_a_launch_of_two_keeps_the_graph(between):
    """However few its workgroups are."""
    from dynaflow_amd import ops

    w, x = randn((1024, 1024), 1, 0.03), [randn((8, 1024), 3 + i) for i in range(2)]
    other = (lambda: ops.linear_variant(x[0], w, 0)) if between == "ring" else (lambda: ops.linear(x[0].float(), w.float()))
    kept = []
    calls = [[lambda i=i: kept.append(ops.linear_variant(x[i], w, 8))] for i in range(2)]
    assert captured(*calls)[1] == 1
    assert captured(calls[0] + [lambda: kept.append(other())], calls[1])[1] == 0
