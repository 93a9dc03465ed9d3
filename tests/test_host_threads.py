"""Plan construction where no thread can be started (CPU, no GPU).

The sanitizer driver of plan construction's host stage runs under a stack
limit, from which a new thread takes its stack's size, that no thread's
allocation meets: every range of the threaded passes runs on the one thread.
"""
import os
import resource
import subprocess

import pytest

from test_host_sanitize import SAN_DIR, SUPP, test_plan_host_stage_under_host_sanitizers as _built

STACK = 100 << 40  # bytes; more than the address space holds


def test_plan_host_stage_without_threads():
    hard = resource.getrlimit(resource.RLIMIT_STACK)[1]
    if hard != resource.RLIM_INFINITY and hard < STACK:
        pytest.skip("the stack limit cannot be raised here")
    exe = os.path.join(SAN_DIR, "_build", "plan_host")
    if not os.path.exists(exe):
        _built()  # builds the driver

    def limit():
        resource.setrlimit(resource.RLIMIT_STACK, (STACK, hard))

    env = dict(os.environ, LSAN_OPTIONS=f"suppressions={SUPP}:print_suppressions=0")
    r = subprocess.run([exe], env=env, preexec_fn=limit, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    assert "plan_host ok" in r.stdout
