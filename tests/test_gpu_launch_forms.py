"""The forms of the group filter and of the finish that a launch's size selects,
against each other: a plane alone (up to 256 filter tiles: 16 waves each; up to
256 finish blocks: one pixel per thread) and the same plane three times in one
launch (more than 256: eight or four waves in the hard stage and four in the
Wiener stage; four pixels per thread). Each row states which of the two it
crosses, and that is checked here; the sums are integers, so the planes must be
the same bit for bit. No tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _counts(width, height, block, step):
    """Filter tiles of 4 x 4 references and finish blocks of 64 x 16 pixels."""
    nx, ny = (width - block + step - 1) // step + 1, (height - block + step - 1) // step + 1
    return -(-nx // 4) * -(-ny // 4), -(-width // 64) * -(-height // 16)


def _compare(gpu, width, height, **kw):
    import torch
    r = np.random.default_rng(width + height)
    y, x = np.mgrid[0:height, 0:width]
    plane = (0.5 + 0.3 * np.sin(x * 0.13) * np.cos(y * 0.11) + r.normal(0, 0.04, (height, width))).astype(np.float32)
    # (the group of the first stage follows group_size)
    src = torch.from_numpy(plane).cuda()
    alone = gpu.BM3D("GRAYS", width, height, sigma=10.0, **kw)
    together = gpu.BM3D("RGBS", width, height, sigma=10.0, **kw)
    one = alone([src])[0].cpu().numpy()
    three = [o.cpu().numpy() for o in together([src, src.clone(), src.clone()])]
    alone.close()
    together.close()
    assert np.isfinite(one).all()
    assert np.abs(one - plane).max() > 0
    for p in three:
        assert np.array_equal(one.view(np.uint32), p.view(np.uint32))


# (block 8 has the filter with 4 to 16 waves; the others share the finish)
@pytest.mark.parametrize("width,height,block,step,group,rng,crosses", [
    (509, 397, 8, 8, 8, 9, "both"), (509, 397, 8, 8, 16, 9, "both"), (509, 397, 8, 8, 8, 24, "both"),
    (531, 259, 8, 7, 8, 9, "both"), (261, 199, 8, 4, 8, 7, "filter"), (261, 199, 8, 4, 16, 12, "filter"),
    (131, 121, 8, 2, 8, 5, "filter"), (509, 397, 4, 4, 8, 9, "finish"), (501, 403, 12, 12, 16, 5, "finish")])
@pytest.mark.parametrize("final", [0, 1])
def test_planes_alone_and_together(gpu, width, height, block, step, group, rng, crosses, final):
    tiles, blocks = _counts(width, height, block, step)
    assert (block == 8 and tiles <= 256 < 3 * tiles) == (crosses in ("both", "filter"))
    assert (blocks <= 256 < 3 * blocks) == (crosses in ("both", "finish"))
    _compare(gpu, width, height, final=final, block_size=block, block_step=step, group_size=group, bm_range=rng)


# hard stage, more than 256 tiles: eight waves while the tiles fill the device at
# most twice (128 times the waves of a CU), then four where eight would put no
# fifth more waves on a CU: 32 either way at group 8, 16 at group 16
@pytest.mark.parametrize("width,height,step,group,rng,waves", [
    (401, 300, 2, 8, 7, 32), (361, 331, 3, 16, 12, 16)])
def test_eight_waves_and_four(gpu, width, height, step, group, rng, waves):
    tiles, _ = _counts(width, height, 8, step)
    assert 256 < tiles <= 128 * waves < 3 * tiles
    _compare(gpu, width, height, final=0, block_step=step, group_size=group, bm_range=rng)
