"""Sizes and matcher choices of the plans on the CPU (tests/asan/plan_sizes: the
library's sources with AddressSanitizer on the host code): every allowed block,
step, range and group is sized without a read outside a table, and the automatic
choice of the matcher of block 8 and of the group filters' tiles on both sides
of each of its lines."""
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


MFMA, RUN, WAVE = 3, 2, 1


@pytest.mark.parametrize("kind,step,rng,group,refs", [
    # ranges up to 9: steps up to 4, groups up to 16, 49152 references (16384 for
    # ranges up to 4 at groups up to 8)
    (RUN, 4, 4, 8, 16383), (MFMA, 4, 4, 8, 16384), (RUN, 4, 5, 8, 49151), (MFMA, 4, 5, 8, 49152),
    (MFMA, 1, 1, 16, 49152), (RUN, 1, 1, 16, 49151), (MFMA, 4, 5, 16, 49152), (RUN, 4, 5, 16, 49151),
    (RUN, 4, 6, 8, 49151), (MFMA, 4, 6, 8, 49152), (RUN, 3, 9, 16, 49151), (MFMA, 3, 9, 16, 49152),
    (RUN, 5, 5, 8, 1 << 20), (RUN, 5, 9, 8, 1 << 20), (RUN, 4, 5, 32, 1 << 20), (RUN, 3, 9, 32, 1 << 20),
    # from 10 on: windows wider than 3.3 steps, 16384; steps 7 and 8 to range 11
    # (12 at group 8), 30000
    (RUN, 6, 10, 32, 16383), (MFMA, 6, 10, 32, 16384), (RUN, 7, 10, 8, 29999), (MFMA, 7, 10, 8, 30000),
    (RUN, 8, 11, 32, 29999), (MFMA, 8, 11, 32, 30000), (RUN, 7, 11, 8, 29999), (MFMA, 7, 12, 8, 16384),
    (RUN, 8, 12, 16, 1 << 20), (RUN, 8, 12, 8, 29999), (MFMA, 8, 12, 8, 30000), (RUN, 8, 13, 16, 16383),
    (MFMA, 8, 13, 16, 16384), (RUN, 20, 10, 8, 1 << 20),
    # any range: small frames stay where the run matcher fits; groups of 64 never leave
    (RUN, 3, 18, 8, 6889), (RUN, 8, 18, 16, 1024), (MFMA, 3, 18, 8, 16384), (MFMA, 3, 40, 32, 100),
    (RUN, 3, 16, 64, 1 << 20), (WAVE, 3, 40, 64, 1 << 20)])
def test_matcher_choice(plan_sizes, kind, step, rng, group, refs):
    r = plan_sizes(step, rng, group, 1920, 1080, refs)
    assert r.returncode == 0, r.stderr[-2000:]
    assert int(r.stdout) == kind


def _over(tw, th, step, rng):
    """Tiles over a pixel: (accumulation rectangle, pixels from tile to tile)."""
    return ((tw - 1) * step + 2 * rng + 8) * ((th - 1) * step + 2 * rng + 8), tw * th * step * step


# the smallest launch of each shape's tiles, and one reference less; groups of 8
# leave the tiles where only 4 x 2 of them fit, groups of 16 where none do
@pytest.mark.parametrize("group,step,rng,tw,th,least", [
    (8, 8, 7, 8, 4, 2048), (8, 8, 27, 8, 4, 2048), (8, 2, 20, 8, 4, 100), (8, 1, 24, 8, 4, 100), (8, 1, 44, 8, 4, 100),
    (8, 8, 28, 4, 4, 480), (8, 8, 34, 4, 4, 480), (8, 4, 40, 4, 4, 480), (8, 2, 42, 4, 4, 480),
    (8, 8, 35, 0, 0, 0), (8, 4, 42, 0, 0, 0), (8, 2, 44, 0, 0, 0), (8, 8, 39, 0, 0, 0),
    (16, 8, 7, 4, 4, 30), (16, 1, 34, 4, 4, 30), (16, 8, 34, 4, 4, 30), (16, 8, 35, 4, 2, 30), (16, 2, 44, 4, 2, 30),
    (16, 8, 40, 0, 0, 0), (32, 8, 7, 0, 0, 0), (4, 8, 7, 0, 0, 0)])
def test_group_filter_tiles(plan_sizes, group, step, rng, tw, th, least):
    if not tw:
        r = plan_sizes("tiles", group, step, rng, 1 << 24)
        assert r.stdout == "0 0\n", r.stdout + r.stderr[-2000:]
        return
    area, pitch = _over(tw, th, step, rng)
    refs = least if least == 2048 else -(-least * area // pitch)
    r = plan_sizes("tiles", group, step, rng, refs, group, step, rng, refs - 1)
    assert r.stdout == f"{tw} {th}\n0 0\n", r.stdout + r.stderr[-2000:]
