"""Scheduling policies shipped with the package."""
from dynaflow_amd.interface import OpSchedulerBase
from dynaflow_amd.schedulers.nanoflow import NanoFlowScheduler  # noqa: F401
from dynaflow_amd.schedulers.staggered import StaggeredScheduler  # noqa: F401
from dynaflow_amd.schedulers.mlp_overlap import MLPOverlapScheduler  # noqa: F401
from dynaflow_amd.schedulers.decoder_overlap import DecoderOverlapScheduler  # noqa: F401

def _parts(home: type) -> tuple:
    """What a class itself has of how operators are issued."""
    own = home.__dict__
    return own.get("schedule"), own.get("_issue"), own.get("_stream_for")


#: The staggered policies' as they are shipped; any other class has none of it.
_SHIPPED = {home: _parts(home) for home in (StaggeredScheduler, MLPOverlapScheduler, OpSchedulerBase)}
_NOTHING = (None, None, None)
_ROUND_ROBIN = NanoFlowScheduler.schedule


def issues_as_shipped(scheduler: OpSchedulerBase) -> bool:
    """Whether ``scheduler`` is a staggered policy that issues its operators, and waits for nothing else, the way the shipped ones
    do: no class that has a part in it (a call of ``super()`` goes to the next one, whichever that is), and nobody afterwards, has
    put something else in the place of what does that."""
    staggered = False
    for home in type(scheduler).__mro__:
        if _parts(home) != _SHIPPED.get(home, _NOTHING):
            return False
        staggered |= home is StaggeredScheduler
    own = scheduler.__dict__
    return staggered and NanoFlowScheduler.schedule is _ROUND_ROBIN and not (
        "schedule" in own or "_issue" in own or "_stream_for" in own)
