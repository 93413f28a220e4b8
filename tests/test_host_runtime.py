"""The library's host code over a HIP runtime of host memory (tests/hostrt/):
the order of launches, waits and frees, error paths among them.  CPU only; no
kernel runs."""
import shutil
import subprocess
from pathlib import Path

import pytest

HOSTRT = Path(__file__).resolve().parent / "hostrt"

CASES = ["failed_launch_joins_the_side_stream", "misaligned_buffers_are_refused",
         "no_stream_outlives_a_device_reset", "streams_stay_with_their_device",
         "prepared_graphs_serve_logged_runs", "branched_replicas_take_the_faster_path",
         "branched_systems_take_the_faster_path"]


@pytest.fixture(scope="module")
def host_rt():
    if not shutil.which("hipcc") or not shutil.which("make"):
        pytest.skip("hipcc/make not available")
    r = subprocess.run(["make", "-s", "-j8", "-C", str(HOSTRT)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    return HOSTRT / "_build" / "host_rt"


@pytest.mark.parametrize("case", CASES)
def test_host_code(host_rt, case):
    r = subprocess.run([str(host_rt), case], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
