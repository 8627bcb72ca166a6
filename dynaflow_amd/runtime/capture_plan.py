"""From which stream a multi-stream schedule can be captured into one hipGraph, and which schedules the capture may put in
another order (``needs_its_order``).

Stream capture starts on one stream (the origin); every other stream joins the capture when it first
waits for an event that a capturing stream recorded.  The HIP runtime books that as "the waiting
stream is a child of the recording stream" - again at every later wait, whichever streams are involved,
unless the waiting stream is the origin - and the end of the capture walks the children of the origin,
their children and so on.  A schedule in which a stream other than the origin waits for an event that it
recorded itself, or in which two such streams wait for each other's events, makes that walk endless: the
process dies with a segmentation fault inside the end-of-capture call.  That is what five captures of
this package did (the one-stream schedule, one stream per nano-batch, the six-segment decode schedule),
and no capture that worked had such a cycle.

Two things keep a schedule clear of it, neither of which changes what the graph computes:

* a wait for an event on the very stream that recorded it orders nothing that stream order does not
  order already, so the device seam never issues it (``HipEvent.wait``);
* the origin is exempt, so a schedule whose two streams wait for each other is captured FROM one of them
  (``choose_origin``) instead of from a third stream.

The functions below work on the (``"record"`` | ``"wait"``, event id, stream) log that both device seams
write, so the plan for a schedule can be made - and tested - without a GPU.
"""
from __future__ import annotations

import operator
from collections.abc import Hashable, Iterable

import torch
import torch.fx
import torch.nn.functional as F

LogEntry = tuple

_FUNCTION_NAMES = (
    "getitem", "add", "sub", "mul", "div", "truediv", "floordiv", "mod", "neg", "pow", "eq", "ne", "lt", "le", "gt", "ge", "abs",
    "sigmoid", "tanh", "silu", "gelu", "relu", "exp", "rsqrt", "sqrt", "square", "clamp", "where", "cat", "split", "chunk",
    "reshape", "flatten", "transpose", "permute", "unsqueeze", "squeeze", "embedding", "rms_norm", "layer_norm",
    "sym_size", "sym_int")
#: Functions that write to none of their arguments and make a few passes over a nano-batch's activations at most.
_PLAIN_FUNCTIONS = {f for home in (operator, torch, F) for name in _FUNCTION_NAMES
                    if callable(f := getattr(home, name, None))}
#: Tensor methods of the same kind.
_PLAIN_METHODS = {
    "view", "reshape", "flatten", "transpose", "permute", "unsqueeze", "squeeze", "expand", "contiguous", "size", "dim", "numel",
    "split", "chunk", "t", "to", "type_as", "float", "bfloat16", "half", "add", "sub", "mul", "div", "neg", "pow", "rsqrt", "sigmoid",
    "tanh", "clamp", "mean", "sum"}


def _is_plain(node: torch.fx.Node) -> bool:
    if node.op in ("placeholder", "get_attr", "output"):
        return True
    if node.op == "call_method":
        return node.target in _PLAIN_METHODS
    if node.op != "call_function":
        return False
    packet = getattr(node.target, "overloadpacket", node.target)
    if isinstance(packet, torch._ops.OpOverloadPacket):
        return str(packet).startswith("dynaflow_hip.")
    if packet not in _PLAIN_FUNCTIONS or any(node.kwargs.get(k) for k in ("out", "inplace", "max_norm")):
        return False
    # the same given by position: silu(x, True), embedding(ids, weight, padding_idx, max_norm)
    name = packet.__name__
    return not (name in ("silu", "relu") and any(a is True for a in node.args)) and \
        not (name == "embedding" and len(node.args) > 3 and node.args[3] is not None)


def needs_its_order(split_graph: torch.fx.GraphModule) -> str | None:
    """The first node of a split graph or of what its sub-graph calls run for which it may matter in which order, or beside what,
    a schedule launches it; None if there is none.

    Launches of two nano-batches that no data flow orders may change places when only operators of this package and plain torch
    functions are launched: those write to nothing but their results.  (Of this package ``decode_attention`` writes to the caches:
    to the slots of its tokens, of which every sequence has one per forward.)  Any other operator - one that writes to a buffer
    which both nano-batches use, one that nobody knows here - stays where the schedule has it; also because it may take long, and
    what the schedule runs beside it would not be beside it any more."""
    for node in split_graph.graph.nodes:
        if node.op != "call_module":
            if not _is_plain(node):
                return f"{node.op} {node.target}"
            continue
        backend = getattr(split_graph, node.target)
        for fn in (backend.callable_dynamic, *backend.callables_per_size.values()):
            fn = getattr(fn, "runnable", fn)         # (a graph wrapper runs it as it is under this capture)
            if not isinstance(fn, torch.fx.GraphModule):
                return f"{node.target}: {type(fn).__name__}"
            for inner in fn.graph.nodes:
                if not _is_plain(inner):
                    return f"{node.target}: {inner.op} {inner.target}"
    return None


def wait_edges(log: Iterable[LogEntry]) -> list[tuple[Hashable, Hashable]]:
    """(recording stream, waiting stream) of every wait for an event that has been recorded, in log order."""
    recorded_on: dict[Hashable, Hashable] = {}
    edges = []
    for entry in log:
        kind = entry[0]
        if kind == "record":
            recorded_on[entry[1]] = entry[2]
        elif kind == "wait" and entry[1] in recorded_on:
            edges.append((recorded_on[entry[1]], entry[2]))
    return edges


def join_cycle(log: Iterable[LogEntry], caller: Hashable, origin: Hashable) -> list | None:
    """A cycle in the child-of relation that capturing ``log`` from ``origin`` would build, or None.

    ``log`` was written with ``caller`` as the current stream of the forward; under capture the origin takes
    that part.  Waits on the recording stream are left out (the seam does not issue them), and so are the
    waits of the origin (it is never made anybody's child).
    """
    children: dict[Hashable, set] = {}
    for src, dst in wait_edges(log):
        src = origin if src == caller else src
        dst = origin if dst == caller else dst
        if src == dst or dst == origin:
            continue
        children.setdefault(src, set()).add(dst)
    state: dict[Hashable, int] = {}

    def walk(node: Hashable, path: list) -> list | None:
        state[node] = 1
        for child in sorted(children.get(node, ()), key=repr):
            if state.get(child) == 1:
                loop = path + [node, child]
                return loop[loop.index(child):]          # the cycle itself, without the way that led to it
            if child not in state:
                found = walk(child, path + [node])
                if found:
                    return found
        state[node] = 2
        return None

    for node in sorted(children, key=repr):
        if node not in state:
            found = walk(node, [])
            if found:
                return found
    return None


def choose_origin(log: Iterable[LogEntry], caller: Hashable) -> Hashable | None:
    """The stream to start the capture on: ``caller`` if that is safe, else the first stream of the log
    (in order of appearance) from which the schedule has no cycle, else None."""
    log = list(log)
    candidates = [caller]
    for entry in log:
        if entry[0] in ("record", "wait") and entry[2] not in candidates:
            candidates.append(entry[2])
    for origin in candidates:
        if join_cycle(log, caller, origin) is None:
            return origin
    return None
