"""The group filters' tile path at wide ranges, whose tiles hold fewer references
(4 x 4 for groups of 8, 4 x 2 for groups of 16, so waves of a workgroup stay
idle), against their atomic path, which a memory limit between the two paths'
needs selects: the same bits, with and without values that are not finite."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _needs(w, h, step, rng, group, ncsr, tw, th):
    """Device bytes of the atomic path and of the tile path (wnnm.cpp)."""
    nx, ny = (w - 8 + step - 1) // step + 1, (h - 8 + step - 1) // step + 1
    both = nx * ny * (group * 16 + 4) + (w * h * 4 if ncsr else 0)
    aw, ah = (tw - 1) * step + 2 * rng + 8, (th - 1) * step + 2 * rng + 8
    tiles = -(-nx // tw) * -(-ny // th) * ((aw + 9) & ~3) * ah
    return both + 16 * w * h, both + 8 * (tiles + nx * ny)


@pytest.mark.parametrize("kind", ["WNNM", "NCSR"])
@pytest.mark.parametrize("w,h,step,rng,group,tw,th", [
    (643, 481, 8, 34, 8, 4, 4),
    (643, 481, 8, 28, 8, 4, 4),
    (547, 551, 3, 41, 8, 4, 4),
    (405, 301, 8, 36, 16, 4, 2),
    (301, 403, 7, 38, 16, 4, 2),
    (403, 299, 8, 34, 16, 4, 4),
    (389, 177, 2, 31, 8, 8, 4),
])
def test_wide_tiles_equal_the_atomic_path(gpu, kind, w, h, step, rng, group, tw, th):
    import torch
    small, large = _needs(w, h, step, rng, group, kind == "NCSR", tw, th)
    limit = -(-small // MIB)
    assert limit * MIB < large
    r = np.random.default_rng(w * h + group)
    yy, xx = np.mgrid[0:h, 0:w]
    src = (0.5 + 0.3 * np.sin(xx / 6.0) * np.cos(yy / 4.5) + r.normal(0, 10 / 255, (h, w))).astype(np.float32)
    bad = src.copy()
    bad[h // 2, w // 3] = np.nan
    bad[h - 1, w - 1] = -np.inf
    for plane in (src, bad):
        got = []
        for lim in (None, limit):
            f = getattr(gpu, kind)("GRAYS", w, h, sigma=[10.0], block_step=step, bm_range=rng, group_size=group,
                                   memory_limit_mb=lim)
            got.append(f([torch.from_numpy(plane).cuda()])[0].cpu().numpy())
            f.close()
        assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
