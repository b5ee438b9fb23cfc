"""WNNM and NCSR instances on a device without room for the tiles' partials: the
atomic path's smaller sums are allocated instead, with the same output. And a
refused memory limit names the least one that is accepted, whichever of the two
paths it is for."""
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

W, H = 333, 251


def _make(gpu, kind, **kw):
    return getattr(gpu, kind)("GRAYS", W, H, sigma=[10.0], block_step=3, bm_range=9, **kw)


def _frame():
    r = np.random.default_rng(3)
    y, x = np.mgrid[0:H, 0:W]
    return (0.5 + 0.3 * np.sin(x / 6.0) * np.cos(y / 4.5) + r.normal(0, 10 / 255, (H, W))).astype(np.float32)


@pytest.mark.parametrize("group", [8, 16])
@pytest.mark.parametrize("kind,allocations", [("WNNM", 3), ("NCSR", 4)])
def test_a_failed_allocation_of_the_tile_path(gpu, kind, allocations, group):
    import torch
    src = [torch.from_numpy(_frame()).cuda()]
    base = gpu.debug_live_allocations()
    tiled = _make(gpu, kind, group_size=group)
    live = gpu.debug_live_allocations()
    assert live[0] - base[0] == allocations
    want = tiled(src)[0].cpu().numpy()
    tiled.close()
    try:
        for k in range(allocations):  # the matches, the counts, the partials (and the estimate)
            gpu.debug_fail_alloc(k)
            small = _make(gpu, kind, group_size=group)
            now = gpu.debug_live_allocations()
            assert now[0] - base[0] == allocations + 1  # two sums instead of the partials
            assert now[1] < live[1]
            got = small(src)[0].cpu().numpy()
            small.close()
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
            assert gpu.debug_live_allocations() == base
    finally:
        gpu.debug_fail_alloc(-1)


@pytest.mark.parametrize("kind", ["WNNM", "NCSR"])
@pytest.mark.parametrize("kw", [dict(block_step=8, bm_range=5), dict(block_step=4, bm_range=9),
                                dict(block_step=8, bm_range=9, group_size=32)])
def test_a_refused_limit_names_the_least(gpu, kind, kw):
    # at step 8 and range 5 the partials are the smaller buffer, else the sums
    make = getattr(gpu, kind)
    with pytest.raises(gpu.Error, match="memory_limit_mb is too small") as e:
        make("GRAYS", 1920, 1080, sigma=[10.0], memory_limit_mb=1, **kw)
    least = int(re.search(r"at least (\d+) MiB", str(e.value)).group(1))
    make("GRAYS", 1920, 1080, sigma=[10.0], memory_limit_mb=least, **kw).close()
    with pytest.raises(gpu.Error, match="memory_limit_mb is too small"):
        make("GRAYS", 1920, 1080, sigma=[10.0], memory_limit_mb=least - 1, **kw)
