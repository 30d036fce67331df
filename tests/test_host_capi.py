"""The C ABI's host code on a stand-in HIP runtime (tests/host): what the host
does beside another thread, and with a device short of memory."""
import os
import subprocess

import pytest

HOST = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host")


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host"))
    r = subprocess.run(["make", "-C", HOST, f"OUT={out}", "-j4"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    return out


def _run(built, exe, what):
    env = dict(os.environ, TSAN_OPTIONS="halt_on_error=1 exitcode=66")
    r = subprocess.run([os.path.join(built, exe), what], capture_output=True, text=True, env=env, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr[-3000:]


def test_counters_read_beside_another_threads_calls(built):
    """bgpq_item_count and its like correct the host's count of keys while
    another thread inserts and pops: no data race."""
    _run(built, "capi_host_threads", "counters")


def test_heap_that_fills_the_memory(built):
    """A heap whose slots just fit is made, without the bulk calls' lookback
    words and without bulk calls; one whose slots do not is refused, and
    nothing stays allocated."""
    _run(built, "capi_host", "memory")


def test_calls_start_no_idle_workgroups(built):
    """A call of a few batches starts as many workgroups as it has calls, and
    the counters share no more memory with the bulk calls' words than a page."""
    _run(built, "capi_host", "grids")
