"""Group filter and finish of launches of few and of many tiles.

One plane alone takes workgroups of 16 waves (filter) and one pixel per
thread (finish); the same plane three times in one launch passes the 256
tiles above which workgroups are smaller. The sums are integers, so the
planes must be the same bit for bit; odd sizes, groups of 8 and 16, both
stages, and groups of 32 (always four waves). No tolerance.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height,step,group", [
    (637, 397, 8, 8), (531, 259, 7, 16), (201, 187, 3, 16), (203, 190, 3, 32), (64, 9, 8, 8)])
@pytest.mark.parametrize("final", [0, 1])
def test_planes_alone_and_together(gpu, width, height, step, group, final):
    import torch
    rng = np.random.default_rng(width + height)
    y, x = np.mgrid[0:height, 0:width]
    plane = (0.5 + 0.3 * np.sin(x * 0.13) * np.cos(y * 0.11) + rng.normal(0, 0.04, (height, width))).astype(np.float32)
    kw = dict(sigma=10.0, final=final, block_step=step, group_size=group, bm_range=9)
    src = torch.from_numpy(plane).cuda()
    alone = gpu.BM3D("GRAYS", width, height, **kw)
    together = gpu.BM3D("RGBS", width, height, **kw)
    one = alone([src])[0].cpu().numpy()
    three = [o.cpu().numpy() for o in together([src, src.clone(), src.clone()])]
    torch.cuda.synchronize()
    alone.close()
    together.close()
    assert np.isfinite(one).all()
    assert np.abs(one - plane).max() > 0
    for p in three:
        assert np.array_equal(one, p)
