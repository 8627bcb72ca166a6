"""Scheduling policies shipped with the package."""
from dynaflow_amd.interface import OpSchedulerBase
from dynaflow_amd.schedulers.nanoflow import NanoFlowScheduler  # noqa: F401
from dynaflow_amd.schedulers.staggered import StaggeredScheduler  # noqa: F401
from dynaflow_amd.schedulers.mlp_overlap import MLPOverlapScheduler  # noqa: F401
from dynaflow_amd.schedulers.decoder_overlap import DecoderOverlapScheduler  # noqa: F401

_PARTS = ("schedule", "_issue", "_stream_for")
#: How the staggered policies issue their operators, as they are shipped: what each class on the way has of that.
_SHIPPED = {home: [(name, vars(home).get(name)) for name in _PARTS]
            for home in (StaggeredScheduler, MLPOverlapScheduler, DecoderOverlapScheduler, OpSchedulerBase)}
_ROUND_ROBIN = NanoFlowScheduler.schedule


def issues_as_shipped(scheduler: OpSchedulerBase) -> bool:
    """Whether ``scheduler`` is a staggered policy that issues its operators, and waits for nothing else, the way the shipped ones
    do: no class that has a part in it (a call of ``super()`` goes to the next one, whichever that is), and nobody afterwards, has
    put something else in the place of what does that."""
    staggered = False
    for home in type(scheduler).__mro__:
        parts, shipped = home.__dict__, _SHIPPED.get(home)
        if shipped is None:
            if "schedule" in parts or "_issue" in parts or "_stream_for" in parts:
                return False
            continue
        staggered |= home is StaggeredScheduler
        for name, function in shipped:
            if parts.get(name) is not function:
                return False
    return staggered and NanoFlowScheduler.schedule is _ROUND_ROBIN and not any(name in scheduler.__dict__ for name in _PARTS)
