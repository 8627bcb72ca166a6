"""From which stream a schedule can be captured as one graph: the event logs of the shipped schedules on the
recording device, and what the plan makes of them.

A capture dies at its end when a stream other than the one the capture started on waits for an event it
recorded itself, or when two such streams wait for each other's events.  The schedules below are the ones that
were captured successfully on an MI355X (no such cycle from the caller's side) and the ones whose capture
ended in a segmentation fault (each has one)."""
import pytest
import torch

from dynaflow_amd.runtime import capture_plan as plan

from test_decode_cpu import decode_inputs, small_model
from test_engine_cpu import compile_mlp, make_config


def mlp_log(host_device, splits, **knobs):
    cfg = make_config(splits, num_nano_batches=splits, **knobs)
    model, manager, compiled, x = compile_mlp(cfg, tokens=96)
    manager.prepare(96, [96])
    host_device.log.clear()
    with torch.no_grad():
        compiled(x)
    return [e for e in host_device.log if e[0] in ("record", "wait")]


def decode_log(host_device, **knobs):
    from dynaflow_amd.backend import make_backend
    from dynaflow_amd.config import CUDAGraphConfig, DynaFlowConfig, InductorConfig
    from dynaflow_amd.manager import DynaFlowManager

    model, T = small_model(), 6
    inputs = decode_inputs(T)
    cfg = DynaFlowConfig("dynaflow_amd.schedulers:DecoderOverlapScheduler", 2, InductorConfig(enabled=False),
                         CUDAGraphConfig(enabled=False, capture_sizes=[T]),
                         {"min_nano_split_tokens": 1, "dump_graph": False, "hip_backend": False, **knobs})
    manager = DynaFlowManager()
    torch._dynamo.reset()
    for t in inputs:
        torch._dynamo.mark_dynamic(t, 0)
    compiled = torch.compile(model, backend=make_backend(manager, cfg), fullgraph=True)
    with torch.no_grad():
        manager.prepare(T, [1] * T)
        compiled(*inputs)
        manager.prepare(T, [1] * T)
        host_device.log.clear()
        compiled(*inputs)
    return [e for e in host_device.log if e[0] in ("record", "wait")]


def test_hand_made_logs():
    # origin O, streams A and B
    fork_join = [("record", 1, "O"), ("wait", 1, "A"), ("record", 2, "A"), ("wait", 2, "B"), ("record", 3, "B"),
                 ("wait", 3, "O")]
    assert plan.wait_edges(fork_join) == [("O", "A"), ("A", "B"), ("B", "O")]
    assert plan.join_cycle(fork_join, "O", "O") is None and plan.choose_origin(fork_join, "O") == "O"
    # A and B wait for each other: a cycle from O, none when the capture starts on A or on B
    ping_pong = fork_join[:5] + [("wait", 3, "A"), ("record", 4, "A"), ("wait", 4, "O")]
    assert plan.join_cycle(ping_pong, "O", "O") == ["A", "B", "A"]
    assert plan.join_cycle(ping_pong, "O", "A") is None and plan.join_cycle(ping_pong, "O", "B") is None
    assert plan.choose_origin(ping_pong, "O") == "A"
    # a wait on the recording stream is never issued, so it is no edge
    own = [("record", 1, "O"), ("wait", 1, "A"), ("record", 2, "A"), ("wait", 2, "A"), ("record", 3, "A"),
           ("wait", 3, "O")]
    assert plan.join_cycle(own, "O", "O") is None
    # a ring of three streams is cut open by starting on any of them
    ring = [("record", 1, "O"), ("wait", 1, "A"), ("record", 2, "A"), ("wait", 2, "B"), ("record", 3, "B"),
            ("wait", 3, "C"), ("record", 4, "C"), ("wait", 4, "A"), ("record", 5, "A"), ("wait", 5, "O")]
    assert plan.join_cycle(ring, "O", "O") == ["A", "B", "C", "A"] and plan.choose_origin(ring, "O") == "A"
    # two pairs that each wait for each other: whichever stream the capture starts on, one pair remains
    pairs = [("record", 1, "O"), ("wait", 1, "A"), ("wait", 1, "C"),
             ("record", 2, "A"), ("wait", 2, "B"), ("record", 3, "B"), ("wait", 3, "A"),
             ("record", 4, "C"), ("wait", 4, "D"), ("record", 5, "D"), ("wait", 5, "C"),
             ("record", 6, "A"), ("wait", 6, "O"), ("record", 7, "C"), ("wait", 7, "O")]
    assert plan.choose_origin(pairs, "O") is None
    # a wait for an event that was never recorded orders nothing
    assert plan.wait_edges([("wait", 9, "A")]) == []


@pytest.mark.parametrize("splits", [2, 3, 4])
def test_two_segment_schedules_capture_from_the_callers_side(host_device, splits):
    log = mlp_log(host_device, splits)
    assert sorted(set(plan.wait_edges(log))) == [("default", "main"), ("main", "side"), ("side", "default")]
    assert plan.choose_origin(log, "default") == "default"


@pytest.mark.parametrize("knobs", [dict(serialize=True), dict(streams="by_nano_batch")])
def test_schedules_that_keep_a_nano_batch_on_one_stream(host_device, knobs):
    """Their only offence is the wait on the recording stream, which the GPU seam does not issue."""
    log = mlp_log(host_device, 2, **knobs)
    own = [(a, b) for a, b in plan.wait_edges(log) if a == b]
    assert own and all(a != "default" for a, _ in own)
    assert plan.choose_origin(log, "default") == "default"


def test_by_nano_batch_with_four_nano_batches(host_device):
    log = mlp_log(host_device, 4, streams="by_nano_batch")
    assert plan.choose_origin(log, "default") == "default"


def test_multi_layer_schedule_by_kind_is_captured_from_its_main_stream(host_device):
    """Attention sub-graphs on one stream, MLP sub-graphs on the other, layer after layer: the two streams wait
    for each other, so neither may be a bystander of a capture started elsewhere."""
    log = decode_log(host_device)
    edges = set(plan.wait_edges(log))
    assert ("main", "side") in edges and ("side", "main") in edges
    assert plan.join_cycle(log, "default", "default") == ["main", "side", "main"]
    assert plan.choose_origin(log, "default") == "main"


def test_multi_layer_schedule_by_nano_batch(host_device):
    log = decode_log(host_device, streams="by_nano_batch")
    assert plan.choose_origin(log, "default") == "default"


# ------------------------------------------------------------ which schedules may be put in another order
class Scratch(torch.nn.Module):
    """Both nano-batches write to one buffer and read it again."""

    def __init__(self):
        super().__init__()
        self.weight = torch.nn.Parameter(torch.ones(8, 8))
        self.register_buffer("last", torch.zeros(8))

    def forward(self, x):
        self.last.copy_(x[0])
        return torch.nn.functional.silu(x) + self.last


def split_graph_of(fn, lowered=False):
    """A split graph as the manager leaves it: its sub-graph calls run what stands in their backends."""
    from types import SimpleNamespace

    from dynaflow_amd.executor.hip_lowering import lower_to_hip

    inner = fn if isinstance(fn, torch.fx.GraphModule) else torch.fx.symbolic_trace(fn)
    if lowered:
        inner = lower_to_hip(inner)[0]
    graph = torch.fx.Graph()
    x = graph.placeholder("x")
    graph.output(graph.call_module("submod_0", (x,)))
    outer = torch.fx.GraphModule({"submod_0": torch.nn.Identity()}, graph)
    del outer._modules["submod_0"]
    outer.__dict__["submod_0"] = SimpleNamespace(callable_dynamic=inner, callables_per_size={})
    return outer


@pytest.mark.parametrize("fn,kept", [
    (lambda x: torch.nn.functional.rms_norm(x, (8,)) + x.view(2, 4).reshape(8) * 2, False),
    (lambda x: torch.cat([x.split(4, -1)[0], x.float()], dim=-1), False),
    (lambda x: torch.nn.functional.embedding(x, x), False),
    (lambda x: torch.nn.functional.embedding(x, x, None, 1.0), True),            # renormalises the table in place
    (lambda x: torch.nn.functional.embedding(x, x, max_norm=1.0), True),
    (lambda x: torch.nn.functional.silu(x, True), True),
    (lambda x: torch.add(x, 1, out=x), True),
    (lambda x: x.mul_(2), True),
    (lambda x: torch.relu_(x), True),
    (lambda x: torch.sort(x)[0], True),                                          # a launch of unknown length
    (lambda x: torch.nn.functional.linear(x, x), True),
    (lambda x: torch.nn.functional.dropout(x), True),
    (Scratch(), True),
])
def test_what_needs_its_order(fn, kept):
    assert (plan.needs_its_order(split_graph_of(fn)) is not None) == kept


def test_in_place_operators_and_opaque_callables_keep_their_order():
    import operator
    from types import SimpleNamespace

    for target in (operator.iadd, operator.setitem, lambda x: x):
        graph = torch.fx.Graph()
        x = graph.placeholder("x")
        graph.output(graph.call_function(target, (x, x, x)))
        assert plan.needs_its_order(split_graph_of(torch.fx.GraphModule({}, graph))) is not None
    outer = split_graph_of(lambda x: x + 1)
    outer.__dict__["submod_0"] = SimpleNamespace(callable_dynamic=lambda x: x, callables_per_size={})
    assert plan.needs_its_order(outer) is not None
    # a callable for one size, and what a graph wrapper runs
    outer.__dict__["submod_0"] = SimpleNamespace(callable_dynamic=torch.fx.symbolic_trace(lambda x: x + 1),
                                                 callables_per_size={4: torch.fx.symbolic_trace(lambda x: x.mul_(2))})
    assert plan.needs_its_order(outer) is not None
    outer.__dict__["submod_0"] = SimpleNamespace(
        callable_dynamic=SimpleNamespace(runnable=torch.fx.symbolic_trace(lambda x: x + 1)), callables_per_size={})
    assert plan.needs_its_order(outer) is None


def test_lowered_models_do_not_need_their_order():
    """The decode model: embedding, norms, projections, the attention that writes to the slots of its tokens."""
    from dynaflow_amd.decode import DecodeModel

    captured = {}
    model = DecodeModel(layers=2, vocab=100, hidden=512, heads=4, kv_heads=2, inter=256, slots=6, capacity=64, dtype=torch.bfloat16)
    model.init_weights()
    inputs = [torch.arange(6), torch.arange(6).int(), torch.full((6,), 5).int()]

    def backend(gm, example_inputs):
        captured["gm"] = gm
        return gm

    torch._dynamo.reset()
    for t in inputs:
        torch._dynamo.mark_dynamic(t, 0)
    torch.compile(model, backend=backend, fullgraph=True)(*inputs)
    assert plan.needs_its_order(split_graph_of(captured["gm"], lowered=True)) is None
    # the same on torch's own kernels
    assert plan.needs_its_order(split_graph_of(captured["gm"])) is not None
