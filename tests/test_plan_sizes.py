"""Sizes and matcher choices of the plans on the CPU (tests/asan/plan_sizes: the
library's sources with AddressSanitizer on the host code): every allowed block,
step, range and group is sized without a read outside a table."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EXE = os.path.join(HERE, "asan", "plan_sizes")
CSRC = os.path.join(HERE, "..", "vapoursynth-nssfactory_amd", "csrc")


@pytest.fixture(scope="module")
def plan_sizes():
    sources = [os.path.join(HERE, "asan", "plan_sizes.cpp")] + [os.path.join(CSRC, f) for f in os.listdir(CSRC)]
    if not os.path.exists(EXE) or any(os.path.getmtime(s) > os.path.getmtime(EXE) for s in sources):
        subprocess.check_call([sys.executable, os.path.join(HERE, "asan", "build_asan.py")],
                              stdout=subprocess.DEVNULL)

    def run(*args):
        env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1")
        return subprocess.run([EXE, *map(str, args)], capture_output=True, text=True, timeout=300, env=env)
    return run


def test_every_shape_is_sized(plan_sizes):
    r = plan_sizes()
    assert r.returncode == 0, r.stdout + r.stderr[-2000:]
    assert "0 failure(s)" in r.stdout
