"""One event loop per thread for the scheduler coroutines.

A forward runs one coroutine to its end (dynaflow/manager.py:161-190 starts a fresh loop with ``asyncio.run`` for it).
Opening and closing a loop costs more than the schedule it runs, so a thread keeps the loop of its first forward; the
loop is closed with the thread.
"""
from __future__ import annotations

import asyncio
import threading
from collections.abc import Coroutine
from typing import Any


class _ThreadLoop(threading.local):
    def __init__(self) -> None:
        self.loop: asyncio.AbstractEventLoop | None = None

    def get(self) -> asyncio.AbstractEventLoop:
        if self.loop is None or self.loop.is_closed():
            self.loop = asyncio.new_event_loop()
        return self.loop

    def __del__(self) -> None:
        if self.loop is not None and not self.loop.is_closed() and not self.loop.is_running():
            self.loop.close()


_thread = _ThreadLoop()


def run_coroutine(coroutine: Coroutine) -> Any:
    """Run ``coroutine`` to its end; whatever tasks it leaves behind are cancelled, as ``asyncio.run`` does."""
    try:
        asyncio.get_running_loop()
    except RuntimeError:
        pass
    else:
        coroutine.close()
        raise RuntimeError("a forward cannot be called from a running event loop")
    loop = _thread.get()
    try:
        return loop.run_until_complete(coroutine)
    finally:
        left = asyncio.all_tasks(loop)
        if left:
            for task in left:
                task.cancel()
            loop.run_until_complete(asyncio.gather(*left, return_exceptions=True))
