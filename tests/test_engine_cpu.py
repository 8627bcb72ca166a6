"""Host logic of a forward on the recording device seam: the engine + shipped
schedulers must produce the launch order and event chain the oracle derives,
and the results of eager PyTorch on the unsplit input."""
import asyncio

import pytest
import torch

from dynaflow_amd.backend import make_backend
from dynaflow_amd.config import CUDAGraphConfig, DynaFlowConfig, InductorConfig
from dynaflow_amd.executor.compiler import SubgraphBackend
from dynaflow_amd.interface import ExecutionContext, OpSchedulerBase, SplitConfig
from dynaflow_amd.manager import DynaFlowManager
from dynaflow_amd.mlp import SwiGLUMLP
from dynaflow_amd.schedulers import MLPOverlapScheduler, NanoFlowScheduler, StaggeredScheduler
from dynaflow_amd.schedulers.mlp_overlap import mlp_split_rules, mlp_tag_rules
from oracle import schedule_trace as ref


def make_config(splits=2, **extra):
    knobs = {"min_nano_split_tokens": 8, "dump_graph": False}
    knobs.update(extra)
    return DynaFlowConfig("dynaflow_amd.schedulers:MLPOverlapScheduler", splits,
                          InductorConfig(enabled=False), CUDAGraphConfig(enabled=False, capture_sizes=[64, 128]), knobs)


def compile_mlp(cfg, tokens=64, hidden=32, inter=96, scheduler=None):
    torch._dynamo.reset()
    torch.manual_seed(0)
    model = SwiGLUMLP(hidden, inter, dtype=torch.float32)
    manager = DynaFlowManager()
    x = torch.randn(tokens, hidden)
    torch._dynamo.mark_dynamic(x, 0)
    compiled = torch.compile(model, backend=make_backend(manager, cfg, scheduler), fullgraph=True)
    manager.prepare(tokens, [tokens])  # not initialised yet: trivial split, used by the tracing call
    with torch.no_grad():
        compiled(x)
    return model, manager, compiled, x


def top_level(manager):
    top = []
    for node in manager.graph_module.graph.nodes:
        if node.op == "placeholder":
            top.append("in")
        elif node.op == "call_module":
            top.append(("mod", node.target))
        elif node.op == "output":
            top.append("out")
        else:
            top.append("fn")
    return top


@pytest.mark.parametrize("order,splits", [("staggered", 2), ("round_robin", 2), ("staggered", 4), ("round_robin", 3)])
def test_launch_order_and_streams_match_oracle(host_device, order, splits):
    cfg = make_config(splits, schedule=order, num_nano_batches=splits)
    model, manager, compiled, x = compile_mlp(cfg, tokens=96)
    split = manager.prepare(96, [96])
    assert split.num_nano_batches == splits
    host_device.log.clear()
    with torch.no_grad():
        y = compiled(x)
    assert manager.cached_config is None, "the split is consumed by the forward"
    torch.testing.assert_close(y, model(x), rtol=0, atol=0)

    want = ref.simulate(top_level(manager), splits, order,
                        lambda m: "side" if "tail" in getattr(manager.graph_module, m).tag else "main",
                        caller_stream="default")
    ranges = [(e[1], e[2]) for e in host_device.log if e[0] == "range"]
    got_launches = [(name.rsplit("_", 1)[0][3:], int(name.rsplit("_", 1)[1]), stream) for name, stream in ranges]
    assert got_launches == ref.launches(want)
    assert manager.engine.issue_trace == [(m, b) for m, b, _ in ref.launches(want)]

    # the full event chain: map event uids to nano-batches through the order of creation
    kinds = [(e[0], e[2]) for e in host_device.log if e[0] in ("record", "wait")]
    want_kinds = [("record" if e[0] == "record" else "wait", e[2]) for e in want if e[0] in ("record", "wait", "join")]
    assert kinds == want_kinds
    # a wait always refers to the event its nano-batch recorded last
    last_record = {}
    launch_iter = iter(ref.launches(want))
    for e in host_device.log:
        if e[0] == "record":
            last_record[e[1]] = e[2]
        elif e[0] == "wait":
            assert e[1] in last_record, "waited on an event that was never recorded"


def test_environment_is_drained(host_device):
    cfg = make_config(2)
    model, manager, compiled, x = compile_mlp(cfg)
    manager.prepare(64, [64])
    with torch.no_grad():
        compiled(x)
    assert manager.engine.last_env.live_entries() == []


def test_single_batch_takes_fast_path_and_bypasses_scheduler(host_device):
    cfg = make_config(2, min_nano_split_tokens=1000)
    model, manager, compiled, x = compile_mlp(cfg)
    split = manager.prepare(64, [64])
    assert split.num_nano_batches == 1
    host_device.log.clear()
    with torch.no_grad():
        y = compiled(x)
    assert [e for e in host_device.log if e[0] == "range"] == []
    torch.testing.assert_close(y, model(x), rtol=0, atol=0)


def test_single_batch_graph_replay_without_a_capturing_dry_run_is_refused(host_device):
    cfg = make_config(2, min_nano_split_tokens=1000)
    model, manager, compiled, x = compile_mlp(cfg)
    manager.prepare(64, [64], use_cudagraph=True)
    with torch.no_grad(), pytest.raises(RuntimeError, match="static input buffer missing"):
        compiled(x)


def test_single_batch_through_scheduler_when_fallback_disallowed(host_device):
    cfg = make_config(2, min_nano_split_tokens=1000)
    model, manager, compiled, x = compile_mlp(cfg)
    split = manager.prepare(64, [64])
    split.allow_fallback = False
    manager.override_split_config(split)
    with torch.no_grad():
        y = compiled(x)
    assert manager.engine.issue_trace == [("submod_0", 0), ("submod_1", 0)]
    torch.testing.assert_close(y, model(x), rtol=0, atol=0)


def test_forward_without_prepare_fails(host_device):
    cfg = make_config(2)
    model, manager, compiled, x = compile_mlp(cfg)
    with pytest.raises(AssertionError):
        compiled(x)


def test_uneven_split_rows_land_in_order(host_device):
    cfg = make_config(2)
    model, manager, compiled, x = compile_mlp(cfg, tokens=50)
    manager.override_split_config(SplitConfig(2, [13, 37], [0, 13, 50], [13, 37], [13, 37], [0, 13, 50], False, False))
    with torch.no_grad():
        y = compiled(x)
    torch.testing.assert_close(y, model(x), rtol=0, atol=0)


def test_dryrun_returns_whole_batch(host_device):
    cfg = make_config(2)
    model, manager, compiled, x = compile_mlp(cfg)
    split = manager.prepare(64, [64], is_dryrun=True)
    assert split.is_dryrun and split.num_nano_batches == 1
    with torch.no_grad():
        y = compiled(x)
    torch.testing.assert_close(y, model(x), rtol=0, atol=0)


class _OutOfOrder(MLPOverlapScheduler):
    async def schedule(self, context: ExecutionContext) -> None:
        first = await context.pop(0)
        await context.execute((first,))
        second = await context.pop(0)
        # executing the first handle again violates the per-nano-batch FIFO
        await context.execute((first,))


def test_out_of_order_execution_is_caught(host_device):
    cfg = make_config(2)
    model, manager, compiled, x = compile_mlp(cfg, scheduler=_OutOfOrder(cfg))
    manager.prepare(64, [64])
    with pytest.raises((AssertionError, KeyError)):
        compiled(x)


class _Substituting(MLPOverlapScheduler):
    calls = 0

    async def schedule(self, context: ExecutionContext) -> None:
        live = list(range(context.split_config.num_nano_batches))
        while live:
            for b in list(live):
                op = await context.pop(b)
                if op is None:
                    live.remove(b)
                    continue
                if "tail" in op.tag:
                    def tail(gate, size, up, w_down):
                        _Substituting.calls += 1
                        assert isinstance(size, int) and gate.shape[0] == size
                        return torch.nn.functional.linear(torch.nn.functional.silu(gate) * up, w_down)
                    await context.execute((op,), tail)
                else:
                    await context.execute(op)  # a bare handle is accepted too


def test_operator_substitution_gets_node_inputs_in_graph_order(host_device):
    cfg = make_config(2)
    model, manager, compiled, x = compile_mlp(cfg, scheduler=_Substituting(cfg))
    manager.prepare(64, [64])
    _Substituting.calls = 0
    with torch.no_grad():
        y = compiled(x)
    assert _Substituting.calls == 2
    torch.testing.assert_close(y, model(x), rtol=1e-6, atol=1e-6)


class _Quitter(MLPOverlapScheduler):
    async def schedule(self, context: ExecutionContext) -> None:
        op = await context.pop(0)
        await context.execute((op,))


def test_scheduler_that_returns_early_leaves_engine_waiting(host_device):
    """Failure detection on the host: the engine blocks on the execute queue; a
    caller that bounds the forward with a time-out sees it."""
    cfg = make_config(2)
    model, manager, compiled, x = compile_mlp(cfg, scheduler=_Quitter(cfg))
    split = manager.prepare(64, [64])

    async def bounded():
        args = (model.gate_proj.weight, 64, x, model.up_proj.weight, model.down_proj.weight)
        placeholders = [n.name for n in manager.engine.placeholder_nodes]
        assert len(placeholders) == len(args)
        await asyncio.wait_for(manager._forward_async(args, {}, split), timeout=0.5)

    with pytest.raises(asyncio.TimeoutError):
        asyncio.run(bounded())


def test_join_results_skips_the_copy_for_consecutive_rows_of_one_buffer():
    from dynaflow_amd.manager import join_results

    buf = torch.arange(24.0).reshape(6, 4).clone()
    parts = {0: buf[0:2], 1: buf[2:5], 2: buf[5:6]}
    joined = join_results(parts, 3, buf)
    assert joined.data_ptr() == buf.data_ptr() and torch.equal(joined, buf)
    # views with more dimensions (sequences x positions x hidden) of the same rows
    joined3 = join_results({0: buf[0:4].view(2, 2, 4), 1: buf[4:6].view(1, 2, 4)}, 2, buf)
    assert joined3.data_ptr() == buf.data_ptr() and joined3.shape == (3, 2, 4)
    # a one-element tuple per nano-batch (what a dynamo graph returns)
    (field,) = join_results({0: (buf[0:3],), 1: (buf[3:6],)}, 2, buf)
    assert field.data_ptr() == buf.data_ptr()
    # rows of a buffer that is not the engine's own (say, views of an input) are copied like torch.cat does
    assert join_results({0: buf[0:3], 1: buf[3:6]}, 2).data_ptr() != buf.data_ptr()
    # anything else is concatenated: a gap, a wrong order, separate tensors, part of a larger buffer
    for parts in ({0: buf[0:2], 1: buf[3:6]}, {0: buf[3:6], 1: buf[0:3]}, {0: buf[0:3].clone(), 1: buf[3:6].clone()},
                  {0: buf[0:2], 1: buf[2:4]}):
        joined = join_results(parts, 2, buf)
        assert joined.data_ptr() != buf.data_ptr()
        assert torch.equal(joined, torch.cat([parts[0], parts[1]], dim=0))


_REFERENCE_STYLE_POLICY = '''
"""A policy file written against the reference package's import names (not this build's)."""
from typing_extensions import override

from dynaflow.config import DynaFlowConfig
from dynaflow.interface import ExecutionContext, InputInfo, OpSchedulerBase, SplitConfig
from dynaflow.matching import MatchingRule, Op
from dynaflow.utils import pack_tokens


class TwoWay(OpSchedulerBase):
    def __init__(self, config: DynaFlowConfig) -> None:
        super().__init__(policy_name="two_way")
        self.capture_sizes = config.cudagraph_config.capture_sizes

    @override
    def get_split_rules(self) -> list[MatchingRule]:
        return [MatchingRule(condition=(Op("silu"), Op("mul"), Op("linear")))]

    @override
    def get_tag_rules(self) -> dict[MatchingRule, set[str]]:
        return {MatchingRule(condition=Op("mul")): {"tail"}}

    @override
    def get_split_config(self, input_info: InputInfo, use_cudagraph: bool = False) -> SplitConfig:
        total = sum(input_info.num_tokens)
        left = total // 2
        padded, fits = pack_tokens(left, self.capture_sizes)
        assert fits and padded >= left
        return SplitConfig(num_nano_batches=2, batch_sizes=[1, 1], batch_indices=[0, 1, 2],
                           num_tokens=[left, total - left], num_tokens_padded=[left, total - left],
                           split_indices=[0, left, total], is_dryrun=False, use_cudagraph=False)

    @override
    async def schedule(self, context: ExecutionContext) -> None:
        live = [0, 1]
        while live:
            for b in list(live):
                op = await context.pop(b)
                if op is None:
                    live.remove(b)
                    continue
                await context.execute((op,))
'''


def test_policy_file_written_against_the_reference_package_names_runs_unmodified(host_device, tmp_path):
    import sys

    import dynaflow_amd

    path = tmp_path / "two_way_policy.py"
    path.write_text(_REFERENCE_STYLE_POLICY)
    dynaflow_amd.install_as_dynaflow()
    try:
        import dynaflow.executor.cudagraph as graphs  # the reference's module name for the graph wrapper

        assert hasattr(graphs, "CUDAGraphWrapper")
        cfg = DynaFlowConfig(f"{path}:TwoWay", 2, InductorConfig(enabled=False),
                             CUDAGraphConfig(enabled=False, capture_sizes=[64, 128]),
                             {"min_nano_split_tokens": 8, "dump_graph": False})
        model, manager, compiled, x = compile_mlp(cfg, tokens=96)
        assert type(manager.scheduler).__name__ == "TwoWay" and manager.scheduler.policy_name == "two_way"
        split = manager.prepare(96, [96])
        assert split.split_indices == [0, 48, 96]
        with torch.no_grad():
            got = compiled(x)
            want = model(x)
        assert torch.allclose(got, want, atol=1e-6)
        assert manager.engine.issue_trace == [("submod_0", 0), ("submod_0", 1), ("submod_1", 0), ("submod_1", 1)]
    finally:
        for name in [n for n in sys.modules if n == "dynaflow" or n.startswith("dynaflow.")]:
            del sys.modules[name]


def test_one_stream_per_nano_batch_policy(host_device):
    """``streams="by_nano_batch"``: every launch of nano-batch 0 on the main stream, of nano-batch 1 on the side
    stream, whatever the sub-graph's tag; the issue order stays the staggered one and the result the same."""
    cfg = make_config(2, streams="by_nano_batch")
    model, manager, compiled, x = compile_mlp(cfg, tokens=96)
    manager.prepare(96, [96])
    host_device.log.clear()
    with torch.no_grad():
        y = compiled(x)
    torch.testing.assert_close(y, model(x), rtol=0, atol=0)
    ranges = [(e[1], e[2]) for e in host_device.log if e[0] == "range"]
    launches = [(name.rsplit("_", 1)[0][3:], int(name.rsplit("_", 1)[1]), stream) for name, stream in ranges]
    assert launches == [("submod_0", 0, "main"), ("submod_1", 0, "main"), ("submod_0", 1, "side"),
                        ("submod_1", 1, "side")]
    with pytest.raises(ValueError):
        MLPOverlapScheduler(make_config(2, streams="per_kernel"))


def test_compute_unit_split_gives_the_two_streams_disjoint_masks(host_device):
    """``cu_split=n``: the side stream gets compute units 0 .. n-1, the main stream the others (the counterpart of
    the reference's green contexts, examples/ae/up-silu-overlap.cu:236-264); unset, the streams carry no mask."""
    from dynaflow_amd.runtime.device import cu_mask_words

    assert cu_mask_words(0, 32, 256) == [0xFFFFFFFF, 0, 0, 0, 0, 0, 0, 0]
    assert cu_mask_words(40, 24, 256) == [0, 0xFFFFFF00, 0, 0, 0, 0, 0, 0]
    assert cu_mask_words(224, 32, 256)[7] == 0xFFFFFFFF
    with pytest.raises(ValueError):
        cu_mask_words(250, 16, 256)
    plain = MLPOverlapScheduler(make_config(2))
    assert plain.comm_stream.cu_mask is None and plain.comp_stream.cu_mask is None
    split = MLPOverlapScheduler(make_config(2, cu_split=48))
    side, main = split.comm_stream.cu_mask, split.comp_stream.cu_mask
    assert len(side) == len(main) == 8
    as_int = lambda words: sum(w << (32 * i) for i, w in enumerate(words))
    assert as_int(side) == (1 << 48) - 1
    assert as_int(side) & as_int(main) == 0 and as_int(side) | as_int(main) == (1 << 256) - 1


def test_listed_sizes_get_their_own_callable_in_a_dry_run(host_device):
    """``InductorConfig.compile_sizes`` (dynaflow/executor/compiler.py:69-85): a dry-run at a listed size builds
    that size's callable; scheduled forwards whose nano-batches have that size dispatch to it, other sizes go to
    the dynamic callable; outside a dry-run an unbuilt listed size is an error."""
    cfg = make_config(2)
    cfg.inductor_config.compile_sizes = {48}
    model, manager, compiled, x = compile_mlp(cfg, tokens=96)
    backends = [manager.graph_module.__dict__[n.target] for n in manager.graph_module.graph.nodes
                if n.op == "call_module"]
    assert all(b.callables_per_size == {} for b in backends)

    # a scheduled forward with nano-batches of the listed size before any dry-run: refused
    manager.prepare(96, [96])
    with pytest.raises(AssertionError, match="dry-run"):
        with torch.no_grad():
            compiled(x)

    # the dry-run at 48 tokens builds the callable of that size in every sub-graph
    small = x[:48].clone()
    manager.prepare(48, [48], is_dryrun=True)
    with torch.no_grad():
        dry = compiled(small)
    torch.testing.assert_close(dry, model(small), rtol=0, atol=0)
    assert all(sorted(b.callables_per_size) == [48] for b in backends)

    # count the calls each callable gets from now on
    calls = {"sized": 0, "dynamic": 0}
    for b in backends:
        sized, dynamic = b.callables_per_size[48], b.callable_dynamic

        def counted(fn, key):
            def call(*a, **k):
                calls[key] += 1
                return fn(*a, **k)
            return call

        b.callables_per_size[48] = counted(sized, "sized")
        b.callable_dynamic = counted(dynamic, "dynamic")

    split = manager.prepare(96, [96])
    assert split.num_tokens == [48, 48]
    with torch.no_grad():
        y = compiled(x)
    torch.testing.assert_close(y, model(x), rtol=0, atol=0)
    assert calls == {"sized": 2 * len(backends), "dynamic": 0}

    # another split of the same input: sizes that are not listed use the dynamic callable
    calls.update(sized=0, dynamic=0)
    manager.override_split_config(SplitConfig(num_nano_batches=2, batch_sizes=[40, 56], batch_indices=[0, 40, 96],
                                              num_tokens=[40, 56], num_tokens_padded=[40, 56],
                                              split_indices=[0, 40, 96], is_dryrun=False, use_cudagraph=False))
    with torch.no_grad():
        y = compiled(x)
    torch.testing.assert_close(y, model(x), rtol=0, atol=0)
    assert calls == {"sized": 0, "dynamic": 2 * len(backends)}


@pytest.mark.parametrize("knobs,splits,want", [
    ({"streams": "by_nano_batch"}, 2, 2),                        # the same sub-graph of both nano-batches at once
    ({"streams": "by_nano_batch"}, 4, 2),                        # four nano-batches take the two streams in turn
    ({"streams": "by_kind"}, 2, 1),                              # launches of one kind queue on one stream
    ({"streams": "by_nano_batch", "serialize": True}, 2, 1),     # one stream
    ({"streams": "by_nano_batch", "side_by_side": 1}, 2, 1),     # override downwards: planned as lone launches
    ({"streams": "by_kind", "serialize": True, "side_by_side": 2}, 2, 2),   # the one-stream baseline of a pair plan
])
def test_kernel_plans_follow_the_schedule_not_a_promise(host_device, monkeypatch, knobs, splits, want):
    """``side_by_side`` - how many launches of one sub-graph share the GPU, what the GEMM plans are made for - is
    derived from the stream policy and the split of each forward; the knob only overrides it downwards."""
    import contextlib

    from dynaflow_amd import ops

    seen = []
    real = ops.launch_options

    @contextlib.contextmanager
    def recording(side_by_side=1):
        seen.append(side_by_side)
        with real(side_by_side=side_by_side):
            yield

    monkeypatch.setattr(ops, "launch_options", recording)
    cfg = make_config(splits, num_nano_batches=splits, **knobs)
    model, manager, compiled, x = compile_mlp(cfg, tokens=96)
    split = manager.prepare(96, [96])
    assert split.num_nano_batches == splits
    assert manager.launches_side_by_side(split) == want
    seen.clear()
    with torch.no_grad():
        y = compiled(x)
    assert seen == [want]
    torch.testing.assert_close(y, model(x), rtol=0, atol=0)
    # a forward that is not split has nothing beside it, whatever the stream policy
    single = manager.prepare(4, [4])
    assert single.num_nano_batches == 1
    if "side_by_side" not in knobs:
        assert manager.launches_side_by_side(single) == 1


@pytest.mark.parametrize("knobs,splits,ranks,tokens,join", [
    ({"streams": "by_nano_batch", "whole_graph": True}, 2, 1, 96, True),
    ({"streams": "by_nano_batch", "whole_graph": True}, 4, 1, 96, True),
    ({"streams": "by_nano_batch", "whole_graph": True}, 2, 1, 258, False),     # more rows than two launches of one take
    ({"streams": "by_nano_batch", "whole_graph": True}, 3, 1, 96, False),      # one without a partner
    ({"streams": "by_nano_batch", "whole_graph": True}, 2, 2, 96, False),
    ({"streams": "by_nano_batch", "whole_graph": True, "pair_launches": False}, 2, 1, 96, False),
    ({"streams": "by_nano_batch", "whole_graph": True, "serialize": True}, 2, 1, 96, False),
    ({"streams": "by_nano_batch"}, 2, 1, 96, False),                           # launched one by one, or a graph a sub-graph
    ({"streams": "by_kind", "whole_graph": True}, 2, 1, 96, False),            # captured in pairs, but planned as lone launches
])
def test_kernel_plans_know_which_launches_become_one(host_device, monkeypatch, knobs, splits, ranks, tokens, join):
    """A kernel that pays where two launches become one is not planned where they stay two; an eager forward has the plans of
    the graph of its manager."""
    from dynaflow_amd import ops

    monkeypatch.setattr(torch.distributed, "is_initialized", lambda: ranks > 1)
    monkeypatch.setattr(torch.distributed, "get_world_size", lambda: ranks)
    cfg = make_config(splits, num_nano_batches=splits, **knobs)
    model, manager, compiled, x = compile_mlp(cfg, tokens=tokens)
    monkeypatch.setattr("dynaflow_amd.runtime.capture_plan.needs_its_order", lambda graph: None)   # (not lowered here)
    split, seen = manager.prepare(tokens, [1] * tokens), []
    assert split.num_nano_batches == splits and manager.launches_join(split) == join
    manager.engine.graph_module.submod_0.callable_dynamic.register_forward_pre_hook(lambda *_: seen.append(ops._join()))
    with torch.no_grad():
        compiled(x)
    assert seen == [join] * splits and not ops._join()
    monkeypatch.setattr("dynaflow_amd.runtime.capture_plan.needs_its_order", lambda graph: "something")
    assert not manager.launches_join(split)


@pytest.mark.parametrize("knobs", [{"streams": "by_kind", "side_by_side": 2},
                                   {"streams": "by_nano_batch", "side_by_side": 3},
                                   {"streams": "by_nano_batch", "side_by_side": 0}])
def test_a_side_by_side_override_that_contradicts_the_schedule_is_refused(host_device, knobs):
    """Streams by sub-graph kind with kernels planned for a pair would queue two half-chip launches on one stream;
    such a configuration raises instead of running slowly."""
    cfg = make_config(2, num_nano_batches=2, **knobs)
    model, manager, compiled, x = compile_mlp(cfg, tokens=96)
    manager.prepare(96, [96])
    with torch.no_grad(), pytest.raises(ValueError, match="side_by_side"):
        compiled(x)


def test_engine_coroutine_behind_queues_issues_what_the_manager_issues(host_device):
    """``engine.execute`` with a context of two queues - for callers that run engine and scheduler side by side
    themselves - against the manager's own forward: the same launches, events and result."""
    cfg = make_config(2)
    model, manager, compiled, x = compile_mlp(cfg)
    split = manager.prepare(64, [64])
    args = (model.gate_proj.weight, 64, x, model.up_proj.weight, model.down_proj.weight)

    def log_of(forward):
        host_device.log.clear()
        with torch.no_grad():
            y = asyncio.run(forward())
        first = min(e[1] for e in host_device.log if e[0] == "record")     # events are numbered process-wide
        return y, [(kind, n - first, where) if kind != "range" else (kind, n, where) for kind, n, where in host_device.log]

    async def queues():
        op_queue = {b: asyncio.Queue(maxsize=10) for b in range(2)}
        execute_queue = asyncio.Queue()
        (results, events), _ = await asyncio.gather(
            manager.engine.execute(args, {}, op_queue, execute_queue, split),
            manager.scheduler.schedule(ExecutionContext(split, op_queue, execute_queue)))
        for event in events:
            event.wait()
        return torch.cat([results[0], results[1]]) if isinstance(results[0], torch.Tensor) else results

    async def direct():
        return await manager._forward_async(args, {}, split)

    y_direct, log_direct = log_of(direct)
    trace = list(manager.engine.issue_trace)
    y_queues, log_queues = log_of(queues)
    assert manager.engine.issue_trace == trace and log_queues == log_direct
    if isinstance(y_queues, dict):
        y_queues = tuple(torch.cat([y_queues[0][i], y_queues[1][i]]) for i in range(len(y_queues[0])))
    for got, want in zip(y_queues if isinstance(y_queues, tuple) else (y_queues,),
                         y_direct if isinstance(y_direct, tuple) else (y_direct,)):
        assert torch.equal(got, want)


class LaneScheduler(MLPOverlapScheduler):
    """One coroutine per nano-batch, each on a stream of its own."""

    async def schedule(self, context):
        from dynaflow_amd.runtime.device import get_device

        async def lane(b, stream):
            while (op := await context.pop(b)) is not None:
                with get_device().stream(stream):
                    await context.execute((op,))

        lanes = range(context.split_config.num_nano_batches)
        await asyncio.gather(*(lane(b, self.lane_streams[b]) for b in lanes))


class TwoLayers(torch.nn.Module):
    def __init__(self):
        super().__init__()
        self.layers = torch.nn.ModuleList(SwiGLUMLP(32, 96, dtype=torch.float32) for _ in range(2))

    def forward(self, x):
        for layer in self.layers:
            x = layer(x)
        return x


@pytest.mark.parametrize("lanes", [2, 3])
def test_a_coroutine_per_nano_batch_is_launched_in_turn(host_device, lanes):
    """Schedulers that run one coroutine per nano-batch: every launch lets the other coroutines have their turn, as the
    hand-over to an engine coroutine does, and a coroutine that waits inside its ``with device.stream`` neither lends its
    stream to another one's launch nor leaves it behind."""
    torch._dynamo.reset()
    cfg = make_config(lanes, num_nano_batches=lanes)
    scheduler = LaneScheduler(cfg)
    scheduler.lane_streams = [host_device.new_stream(f"lane{b}") for b in range(lanes)]
    torch.manual_seed(0)
    model, manager, x = TwoLayers(), DynaFlowManager(), torch.randn(96, 32)
    torch._dynamo.mark_dynamic(x, 0)
    compiled = torch.compile(model, backend=make_backend(manager, cfg, scheduler), fullgraph=True)
    manager.prepare(96, [96])
    with torch.no_grad():
        compiled(x)
        assert manager.prepare(96, [96]).num_nano_batches == lanes
        host_device.log.clear()
        y = compiled(x)
    torch.testing.assert_close(y, model(x), rtol=0, atol=0)
    subgraphs = [name for name in top_level(manager) if isinstance(name, tuple)]
    assert len(subgraphs) >= 4
    assert manager.engine.issue_trace == [(name, b) for _, name in subgraphs for b in range(lanes)]
    assert [e[2] for e in host_device.log if e[0] == "range"] == [f"lane{b}" for _ in subgraphs for b in range(lanes)]
    assert host_device.current_stream().name == "default"


@pytest.mark.parametrize("policy", ["dynaflow_amd.schedulers:MLPOverlapScheduler", "test_engine_cpu:OwnWay"])
def test_a_forward_inside_an_operator_is_refused(host_device, policy):
    """Under every scheduler: a nested forward would take over the engine's state in the middle of the outer one."""
    cfg = make_config(2)
    cfg.scheduler_path = policy
    model, manager, compiled, x = compile_mlp(cfg)
    refused = []

    def operator(*_):
        manager.prepare(64, [64])
        with pytest.raises(RuntimeError, match="running event loop"):
            compiled(x)
        refused.append(1)

    hook = manager.engine.graph_module.submod_0.callable_dynamic.register_forward_pre_hook(operator)
    for _ in range(2):
        manager.prepare(64, [64])
        with torch.no_grad():
            torch.testing.assert_close(compiled(x), model(x), rtol=0, atol=0)
    hook.remove()
    assert len(refused) == 4


class OwnWay(MLPOverlapScheduler):
    async def schedule(self, context):
        await super().schedule(context)


class Waits(StaggeredScheduler):
    async def schedule(self, context):
        await asyncio.sleep(0)
        await super().schedule(context)


class WaitsBehindTheShippedOne(MLPOverlapScheduler, Waits):
    pass


def plain(patch):
    return MLPOverlapScheduler


def patched(home):
    async def schedule(self, context):
        await asyncio.sleep(0)
        await shipped(self, context)

    shipped = home.schedule

    def patch(monkeypatch):
        monkeypatch.setattr(home, "schedule", schedule)
        return MLPOverlapScheduler

    return patch


@pytest.mark.parametrize("kind,order,as_shipped", [
    (plain, "staggered", True), (plain, "round_robin", True), (lambda patch: WaitsBehindTheShippedOne, "staggered", False),
    (patched(StaggeredScheduler), "staggered", False), (patched(MLPOverlapScheduler), "staggered", False),
    (patched(NanoFlowScheduler), "round_robin", False)])
def test_a_schedule_that_waits_gets_a_loop(host_device, monkeypatch, kind, order, as_shipped):
    """Whichever class on the way to the shipped schedule waits, and whoever has put it there."""
    cfg = make_config(2, schedule=order)
    model, manager, compiled, x = compile_mlp(cfg, scheduler=kind(monkeypatch)(cfg))
    assert manager._schedules_plainly() == as_shipped
    manager.prepare(64, [64])
    with torch.no_grad():
        torch.testing.assert_close(compiled(x), model(x), rtol=0, atol=0)


@pytest.mark.parametrize("register", [
    lambda module, hook: module.register_forward_hook(hook),
    lambda module, hook: module.register_forward_pre_hook(hook),
    lambda module, hook: torch.nn.modules.module.register_module_forward_hook(hook),
    lambda module, hook: torch.nn.modules.module.register_module_forward_pre_hook(hook),
], ids=["forward", "forward_pre", "all_modules_forward", "all_modules_forward_pre"])
def test_hooks_see_a_subgraph_that_is_called_past_module_call(register):
    class Twice(torch.nn.Module):
        def forward(self, tokens, x):
            return x * 2

    gm = torch.fx.symbolic_trace(Twice())
    backend = SubgraphBackend(gm, 0, InductorConfig(enabled=False), CUDAGraphConfig(enabled=False, capture_sizes=[]),
                              use_inductor=False, use_cudagraph=False)
    backend.callable_dynamic = gm
    seen = []
    handle = register(gm, lambda module, *rest: seen.append(module))
    try:
        backend(3, torch.ones(3))
    finally:
        handle.remove()
    assert any(module is gm for module in seen)
    assert torch.equal(backend(3, torch.ones(3)), torch.full((3,), 2.0)) and len(seen) == 1


@pytest.mark.parametrize("how", ["compiled in place", "another __call__"])
def test_a_subgraph_module_that_is_called_otherwise_is_not_called_past_that(monkeypatch, how):
    class Twice(torch.nn.Module):
        def forward(self, tokens, x):
            return x * 2

    gm, seen = torch.fx.symbolic_trace(Twice()), []
    backend = SubgraphBackend(gm, 0, InductorConfig(enabled=False), CUDAGraphConfig(enabled=False, capture_sizes=[]),
                              use_inductor=False, use_cudagraph=False)
    backend.callable_dynamic = gm
    if how == "compiled in place":
        def compiler(graph, inputs):
            seen.append(gm)
            return graph.forward

        torch._dynamo.reset()
        gm.compile(backend=compiler)
    else:
        call = torch.nn.Module.__call__

        def watched(module, *args, **kwargs):
            seen.append(module)
            return call(module, *args, **kwargs)

        monkeypatch.setattr(torch.nn.Module, "__call__", watched)
    assert torch.equal(backend(3, torch.ones(3)), torch.full((3,), 2.0))
    assert any(module is gm for module in seen)
