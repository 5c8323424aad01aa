"""Whole fields through the pinned ring, on the CPU: smx_ring.h over a stand-in for the runtime
(ring_check.cpp) that makes queued copies only when something waits for them."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def ring_check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("ring") / "ring_check")
    subprocess.run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-Wall", "-pthread", "-D__HIP_PLATFORM_AMD__",
                    "-I", "/opt/rocm/include", os.path.join(HERE, "ring_check.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("scenario", ["bytes", "errors", "nomemory", "known"])
def test_ring(ring_check, scenario):
    """bytes: every byte arrives, at sizes about the thresholds, with one and several workers.  errors: after a
    call of the runtime failed, no copy is in flight that still uses the slots or the caller's array.
    nomemory: without the ring's memory the runtime's copy is taken.  known: memory that the runtime knows
    (pinned, managed, device) goes in one copy of its own."""
    r = subprocess.run([ring_check, scenario], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
