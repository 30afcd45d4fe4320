"""CPU tests of the sorted join on the CPU build (tests/cpu_sim) with the address
and undefined-behaviour sanitizers:

* join_sorted_wide: buckets of more than 1024 spread build keys (one s_payload
  interval per key) and s_payloads over the whole int32 range; many buckets of
  few rows with one key of 4000, which the sample shows and a bucket has room for.
"""
import os
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent / "cpu_sim"


@pytest.fixture(scope="module")
def cpu_build():
    env = dict(os.environ, SIMT_VARIANT="asan")
    subprocess.run([sys.executable, str(HERE / "build.py"), "join_sorted_wide"], check=True, env=env, timeout=900)
    return HERE / "_build" / "asan"


def run(exe, *args):
    r = subprocess.run([str(exe), *args], capture_output=True, text=True, timeout=600,
                       env=dict(os.environ, SIMT_TRACE="1"))
    assert r.returncode == 0 and r.stdout.strip().endswith("PASS"), r.stdout[-2000:] + r.stderr[-2000:]
    return r.stderr


def test_one_payload_interval_per_key(cpu_build):
    assert "k_sj_finish<<<8, 1024" in run(cpu_build / "join_sorted_wide")


def test_room_for_a_hot_key_among_few_rows(cpu_build):
    trace = run(cpu_build / "join_sorted_wide", "hot")
    assert "k_sj_finish" in trace and "k_join_probe" not in trace
