"""CPU tests of the group-by's host side on the CPU build (tests/cpu_sim):

* groupby_plan: a call's workspace and launches follow one reading of the tune
  table, whatever is set in between.
* serve_budget: served group-bys within a small device-memory budget.
"""
import os
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent / "cpu_sim"


@pytest.fixture(scope="module")
def cpu_build():
    env = dict(os.environ, SIMT_VARIANT="fast")
    subprocess.run([sys.executable, str(HERE / "build.py"), "groupby_plan", "serve_budget"], check=True, env=env, timeout=900)
    return HERE / "_build" / "fast"


@pytest.mark.parametrize("driver", ["groupby_plan", "serve_budget"])
def test_driver(cpu_build, driver):
    r = subprocess.run([str(cpu_build / driver)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0 and r.stdout.strip().endswith("PASS"), r.stdout[-2000:] + r.stderr[-2000:]
