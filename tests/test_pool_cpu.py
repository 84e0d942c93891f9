"""CPU: the buffers that host-pointer calls keep, in the library's own host code with
the HIP calls replaced (tests/fakehip): they are bounded, giving them back neither
touches other users' buffers nor waits nor blocks the pool, and memory that is short
gets them back; and a call that fails leaves no copy of the caller's memory under way.
The native server's thread works on the server's device."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DIR = os.path.join(ROOT, "tests", "fakehip")

pytestmark = pytest.mark.skipif(not os.path.exists("/opt/rocm/bin/hipcc"), reason="no hipcc")


@pytest.fixture(scope="module")
def driver():
    p = subprocess.run(["make", "-s", "-C", DIR], capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stdout[-2000:] + p.stderr[-2000:]
    return os.path.join(DIR, "_build", "pool_driver")


@pytest.mark.parametrize("scenario", ["bounded", "unblocked", "shortage", "drained", "server"])
def test_pool(driver, scenario):
    p = subprocess.run([driver, scenario], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0 and p.stdout.strip().endswith("ok"), p.stdout[-2000:] + p.stderr[-2000:]
