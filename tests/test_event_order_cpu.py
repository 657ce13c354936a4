"""The order of the spikes that read_events returns, checked on the host with
tests/event_order_check.cpp under AddressSanitizer: counting events into rows may not write
before or after its counters, whatever step a generated cell logs them at."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_events_are_sorted_for_every_row(tmp_path):
    exe = tmp_path / "event_order_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address", "-I", ROOT,
                    os.path.join(ROOT, "tests", "event_order_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip() == "ok 72", out.stdout + out.stderr[:2000]
