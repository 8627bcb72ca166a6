"""One event loop per thread for the scheduler coroutines.

A forward runs one coroutine to its end (dynaflow/manager.py:161-190 starts a fresh loop with ``asyncio.run`` for it).
Opening and closing a loop costs more than the schedule it runs, so a thread keeps the loop of its first forward; the
loop is closed with the thread.
"""
from __future__ import annotations

import asyncio
import ctypes
import os
import threading
from collections.abc import Coroutine
from typing import Any


class _TaskFactory:
    """Makes a loop's tasks and counts the ones of a run."""

    def __init__(self) -> None:
        self.made = 0

    def __call__(self, loop: asyncio.AbstractEventLoop, coroutine: Coroutine, **kwargs: Any) -> asyncio.Task:
        self.made += 1
        return asyncio.Task(coroutine, loop=loop, **kwargs)


#: A loop of a parent process that a fork has brought here shares the parent's epoll object: closing it (its own ``__del__``
#: does that too, at the end of the process at the latest) would take the parent's wake-up descriptor out of it.  One
#: reference that nobody gives back leaves it as it is.
_keep_forever = ctypes.PYFUNCTYPE(None, ctypes.py_object)(("Py_IncRef", ctypes.pythonapi))


class _KeptLoop:
    """A loop and whoever closes it: the thread's locals hold this object and the loop does not, so it goes, and the loop
    is closed, when they are dropped at the end of the thread.  (A loop by itself is part of reference cycles and would
    keep its descriptors until the collector finds it.)"""

    def __init__(self) -> None:
        self.loop = asyncio.new_event_loop()
        self.tasks = _TaskFactory()
        self.loop.set_task_factory(self.tasks)
        self.process = os.getpid()
        self.forks = _forks

    def __del__(self, _process: Any = os.getpid, _keep_forever: Any = _keep_forever) -> None:   # (also at the very end)
        loop = getattr(self, "loop", None)
        if loop is None or loop.is_closed() or loop.is_running():
            return
        if self.process != _process():
            _keep_forever(loop)
        else:
            loop.close()


_thread = threading.local()

#: Forks of this process so far.  A loop from before one shares its epoll object with the child, whatever that does with
#: its copy: the next forward takes a new loop.
_forks = 0


def _count_fork() -> None:
    global _forks
    _forks += 1


os.register_at_fork(after_in_parent=_count_fork)


def _kept_loop() -> _KeptLoop:
    kept = getattr(_thread, "kept", None)
    if kept is None or kept.process != os.getpid() or kept.forks != _forks or kept.loop.is_closed():
        kept = _thread.kept = _KeptLoop()
    return kept


def may_have_other_tasks() -> bool:
    """False if the coroutine of ``run_coroutine`` that runs now is the only one: it has started no task.  (Half a
    microsecond where a turn of the loop takes three.)"""
    loop = asyncio.get_running_loop()
    if loop is _on_demand:
        return False                                   # run_without_loop
    kept = getattr(_thread, "kept", None)
    if kept is None or kept.loop is not loop or loop.get_task_factory() is not kept.tasks:
        return True
    return kept.tasks.made > 1


def _refuse_running_loop(coroutine: Coroutine) -> None:
    if asyncio._get_running_loop() is not None:
        coroutine.close()
        raise RuntimeError("a forward cannot be called from a running event loop")


class _LoopOnDemand(asyncio.AbstractEventLoop):
    """The running loop while a coroutine is run without one: what looks for a running loop finds one (another forward and
    ``asyncio.run`` refuse to start inside it), and what uses it uses the thread's."""

    def __getattribute__(self, name: str) -> Any:
        return getattr(_kept_loop().loop, name)


_on_demand = _LoopOnDemand()


def _cancel_left(loop: asyncio.AbstractEventLoop) -> None:
    left = asyncio.all_tasks(loop)
    if left:
        for task in left:
            task.cancel()
        loop.run_until_complete(asyncio.gather(*left, return_exceptions=True))
        for task in left:
            if not task.cancelled() and task.exception() is not None:
                loop.call_exception_handler({"message": "a task that outlived its forward failed while it was cancelled",
                                             "exception": task.exception(), "task": task})


def run_without_loop(coroutine: Coroutine) -> Any:
    """Run a coroutine that waits for nothing (a forward under a scheduler that issues one operator after the other) to its end.
    A turn of the loop and the task around the coroutine cost 30 us of a forward's 400.  Tasks that something inside it starts are
    cancelled at its end."""
    _refuse_running_loop(coroutine)
    kept = getattr(_thread, "kept", None)
    if kept is not None:
        kept.tasks.made = 0
    asyncio._set_running_loop(_on_demand)
    try:
        coroutine.send(None)
    except StopIteration as done:
        return done.value
    finally:
        asyncio._set_running_loop(None)
        kept = getattr(_thread, "kept", None)
        if kept is not None and kept.tasks.made and not kept.loop.is_closed():
            _cancel_left(kept.loop)
    coroutine.close()
    raise RuntimeError("a schedule that was taken to wait for nothing waits")


def run_coroutine(coroutine: Coroutine) -> Any:
    """Run ``coroutine`` to its end; whatever tasks it leaves behind are cancelled, as ``asyncio.run`` does."""
    _refuse_running_loop(coroutine)
    kept = _kept_loop()
    loop, kept.tasks.made = kept.loop, 0
    try:
        return loop.run_until_complete(coroutine)
    finally:
        _cancel_left(loop)
