"""The group filters' tile path (full groups of 8 or 16 blocks of 8, sums of a
tile of references in LDS) against their atomic path, which a memory limit
between the two paths' needs selects: the same arithmetic, so the same bits.
Shapes: ragged grids, one row or column of references, tiles that are not
full, steps 1-8, and planes holding a NaN and infinities (the groups of a wave
must not see a neighbour's)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _grid(n, step):
    return (n - 8 + step - 1) // step + 1


def _needs(w, h, step, rng, group, ncsr):
    """Device bytes of the atomic path and of the tile path (wnnm.cpp)."""
    nx, ny = _grid(w, step), _grid(h, step)
    both = nx * ny * (group * 16 + 4) + (w * h * 4 if ncsr else 0)
    tw, th = (8, 4) if group == 8 else (4, 4)
    aw, ah = (tw - 1) * step + 2 * rng + 8, (th - 1) * step + 2 * rng + 8
    tiles = -(-nx // tw) * -(-ny // th) * ((aw + 9) & ~3) * ah
    return both + 16 * w * h, both + 8 * (tiles + nx * ny)


@pytest.mark.parametrize("kind", ["WNNM", "NCSR"])
@pytest.mark.parametrize("w,h,step,rng,group", [
    (253, 191, 3, 9, 8),
    (251, 190, 3, 7, 16),
    (123, 117, 1, 3, 8),
    (1501, 96, 4, 5, 16),
    (96, 1501, 4, 5, 8),
    (2999, 12, 2, 7, 8),
    (9, 3001, 1, 9, 16),
    (605, 399, 5, 12, 8),
])
def test_tile_path_equals_the_atomic_path(gpu, kind, w, h, step, rng, group):
    import torch
    small, large = _needs(w, h, step, rng, group, kind == "NCSR")
    limit = -(-small // MIB)
    assert limit * MIB < large
    r = np.random.default_rng(w * h + group)
    yy, xx = np.mgrid[0:h, 0:w]
    src = (0.5 + 0.3 * np.sin(xx / 6.0) * np.cos(yy / 4.5) + r.normal(0, 10 / 255, (h, w))).astype(np.float32)
    bad = src.copy()
    bad[h // 2, w // 3] = np.nan
    bad[h // 3, w // 2] = np.inf
    bad[h - 1, w - 1] = -np.inf
    forms = [dict(residual=q, adaptive_aggregation=a) for q, a in ((0, 1), (1, 1), (1, 0))] if kind == "WNNM" else \
        [dict(iters=1), dict(iters=2)]
    for kw in forms:
        for plane in (src, bad):
            got = []
            for lim in (0, limit):
                f = getattr(gpu, kind)("GRAYS", w, h, sigma=[10.0], block_step=step, bm_range=rng, group_size=group,
                                       memory_limit_mb=lim or None, **kw)
                got.append(f([torch.from_numpy(plane).cuda()])[0].cpu().numpy())
                f.close()
            assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32)), kw
