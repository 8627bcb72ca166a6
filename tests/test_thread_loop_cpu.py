"""The event loop that a thread keeps for its forwards: what ``asyncio.run`` did for each of them is still done."""
import asyncio
import gc
import logging
import multiprocessing
import os
import subprocess
import sys
import threading
import time
import warnings

import pytest

from dynaflow_amd.runtime.loop import run_coroutine, run_without_loop

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


async def nothing():
    return 7


def open_descriptors():
    return len(os.listdir("/proc/self/fd"))


def test_a_loop_is_closed_with_its_thread_without_the_collector():
    def forward():
        assert run_coroutine(nothing()) == 7

    gc.collect()
    gc.disable()
    try:
        before = open_descriptors()
        with warnings.catch_warnings():
            warnings.simplefilter("error", ResourceWarning)
            for _ in range(20):
                thread = threading.Thread(target=forward)
                thread.start()
                thread.join()
            assert open_descriptors() == before
    finally:
        gc.enable()


def test_a_loop_is_closed_at_the_end_of_the_process():
    code = ("from dynaflow_amd.runtime.loop import run_coroutine\n"
            "async def nothing(): return 7\n"
            "assert run_coroutine(nothing()) == 7\n")
    done = subprocess.run([sys.executable, "-X", "dev", "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=120)
    assert done.returncode == 0 and "event loop" not in done.stderr and "loop.py" not in done.stderr, done.stderr


def _in_a_forked_child():
    from dynaflow_amd.runtime import loop

    assert run_coroutine(nothing()) == 7
    loop._thread.__dict__.clear()            # what the end of a thread does
    gc.collect()


def _closes_what_it_inherits():
    from dynaflow_amd.runtime import loop

    loop._thread.kept.loop.close()


@pytest.mark.parametrize("child", [_in_a_forked_child, _closes_what_it_inherits])
def test_a_forked_child_leaves_its_parents_loop_alone(child):
    """A child shares the parent's epoll object.  One that closes the inherited loop takes the parent's wake-up descriptor
    out of it, and the parent's coroutines then sleep through what other threads finish for them."""
    async def other_thread():
        started = time.monotonic()
        await asyncio.wait_for(asyncio.get_running_loop().run_in_executor(None, time.sleep, 0.02), 10)
        return time.monotonic() - started

    assert run_coroutine(nothing()) == 7
    with warnings.catch_warnings():
        warnings.simplefilter("ignore", DeprecationWarning)      # a fork beside torch's threads
        child = multiprocessing.get_context("fork").Process(target=child)
        child.start()
    child.join(60)
    assert child.exitcode == 0
    assert run_coroutine(other_thread()) < 5


@pytest.mark.parametrize("forward", [False, True])
def test_a_forked_child_that_ends_like_any_process_leaves_its_parents_loop_alone(forward):
    """Through the interpreter's end, where modules are already taken apart, with and without a forward of its own."""
    code = (f"import asyncio, os, sys, time\n"
            f"from dynaflow_amd.runtime import loop\n"
            f"run_coroutine = loop.run_coroutine\n"
            f"async def nothing(): return 7\n"
            f"async def other_thread():\n"
            f"    started = time.monotonic()\n"
            f"    await asyncio.wait_for(asyncio.get_running_loop().run_in_executor(None, time.sleep, 0.02), 10)\n"
            f"    return time.monotonic() - started\n"
            f"assert run_coroutine(nothing()) == 7\n"
            f"child = os.fork()\n"
            f"if child == 0:\n"
            f"    if {forward}: assert run_coroutine(nothing()) == 7\n"
            f"    sys.exit(0)\n"
            f"assert os.waitpid(child, 0)[1] == 0\n"
            f"assert run_coroutine(other_thread()) < 5\n")
    done = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=120)
    assert done.returncode == 0 and not done.stderr, done.stderr


def test_a_left_over_task_that_fails_while_it_is_cancelled_is_reported(caplog):
    async def fails_on_cancel():
        try:
            await asyncio.sleep(60)
        finally:
            raise ValueError("lost work")

    async def leaves_it():
        asyncio.get_running_loop().create_task(fails_on_cancel())
        await asyncio.sleep(0)

    with caplog.at_level(logging.ERROR, "asyncio"):
        run_coroutine(leaves_it())
    assert any(r.exc_info and "lost work" in str(r.exc_info[1]) for r in caplog.records)


def test_a_forward_that_waits_for_nothing_needs_no_loop(monkeypatch):
    made = []
    monkeypatch.setattr(asyncio, "new_event_loop", lambda: made.append(1))
    assert run_without_loop(nothing()) == 7 and not made

    async def fails():
        raise KeyError("its own")

    with pytest.raises(KeyError, match="its own"):
        run_without_loop(fails())
    closed = []

    async def waits():
        try:
            await asyncio.sleep(0)
        finally:
            closed.append(1)

    with pytest.raises(RuntimeError, match="waits"):
        run_without_loop(waits())
    assert closed == [1]


def test_a_forward_without_a_loop_is_refused_inside_one():
    async def inside():
        with pytest.raises(RuntimeError, match="running event loop"):
            run_without_loop(nothing())
        return 3

    assert run_coroutine(inside()) == 3


@pytest.mark.parametrize("inner", [run_without_loop, run_coroutine, asyncio.run])
def test_a_forward_without_a_loop_refuses_what_one_with_a_loop_refuses(inner):
    """An operator cannot start another forward, or a loop of its own, in the middle of a schedule."""
    async def operator():
        coroutine = nothing()
        with pytest.raises(RuntimeError, match="running event loop"):
            inner(coroutine)
        coroutine.close()
        return 3

    assert run_without_loop(operator()) == run_coroutine(operator()) == 3
    assert run_without_loop(nothing()) == asyncio.run(nothing()) == 7


def test_an_operator_finds_a_running_loop_without_one():
    ended = []

    async def other():
        try:
            await asyncio.sleep(60)
        finally:
            ended.append(asyncio.current_task().get_loop())

    async def operator():
        task = asyncio.get_running_loop().create_task(other())
        task.get_loop().call_soon(ended.append, "called")
        return task

    task = run_without_loop(operator())
    assert task.cancelled() and ended == ["called"]
    assert asyncio._get_running_loop() is None
    assert run_coroutine(nothing()) == 7
