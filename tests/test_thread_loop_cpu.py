"""The event loop that a thread keeps for its forwards: what ``asyncio.run`` did for each of them is still done."""
import gc
import os
import subprocess
import sys
import threading
import warnings

from dynaflow_amd.runtime.loop import run_coroutine

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
