"""Wiener gains and fixed-point sums beyond the range of their short forms.

The gains r^2 / (r^2 + sigma^2) take a short division where the coefficients
and sigma^2 allow it, the sums a short conversion where the values do. Every
finite sigma is accepted, so both sides of each limit, and sigmas whose square
is not finite, must give what the plain division gives: against the oracle
(block matching on the same planes is exact, so the groups are the same).

Tolerance: the forward and inverse transforms are 8-point sums over x, y and
(by halves) the group, at most 64 roundings of 2^-24 of the largest value on a
pixel's path, on either side: 2^-17 of the plane's largest value.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

W, H = 61, 45


def _plane(scale):
    rng = np.random.default_rng(5)
    y, x = np.mgrid[0:H, 0:W]
    v = 0.5 + 0.3 * np.sin(x * 0.21) * np.cos(y * 0.17) + rng.normal(0, 0.04, (H, W))
    return (v * scale).astype(np.float32)


def _run(gpu, plane, **kw):
    import torch
    inst = gpu.BM3D("GRAYS", W, H, ref=True, **kw)
    src = [torch.from_numpy(plane).cuda()]
    got = inst(src, ref=src)[0].cpu().numpy()
    inst.close()
    return got


# sigma^2 of the filter (the argument times 0.75 / 255): 2^-60 and 2^61 lie
# near 3.2e-7 and 5.2e11; from 6.3e21 on it is not finite
@pytest.mark.parametrize("group", [8, 16, 32])
@pytest.mark.parametrize("sigma", [1e-20, 2.9e-7, 3.5e-7, 4.9e11, 5.5e11, 6e21, 7e21, 1e30, 3e38])
def test_sigmas(gpu, oracle, sigma, group):
    plane = _plane(1.0)
    kw = dict(sigma=sigma, group_size=group, block_step=5)
    got = _run(gpu, plane, **kw)
    want, = oracle.bm3d_frame([plane], gpu.parse("GRAYS", W, H, ref=True, **kw), ref=[plane])
    assert np.isfinite(got).all()
    assert np.abs(got - want).max() <= 2.0 ** -17 * np.abs(plane).max()


# a lane's coefficients sum to 2^30 near 2e7 (group 8), the fixed-point values
# of a patch's row to 2^19 near 3e7 (weights of 1 / 512)
@pytest.mark.parametrize("group", [8, 16, 32])
@pytest.mark.parametrize("scale", [2e6, 1.5e7, 3e7, 6e7, 2e8])
def test_values(gpu, oracle, scale, group):
    plane = _plane(scale)
    kw = dict(sigma=10.0, group_size=group, block_step=5)
    got = _run(gpu, plane, **kw)
    want, = oracle.bm3d_frame([plane], gpu.parse("GRAYS", W, H, ref=True, **kw), ref=[plane])
    assert np.abs(got - want).max() <= 2.0 ** -17 * np.abs(plane).max()


# every temporal filter (tiles of references; groups one by one where the
# tiles do not fit), at the gate of the other temporal tests: a gain that is
# not a number leaves the source, 20 dB from the groups' means
@pytest.mark.parametrize("sigma", [10.0, 5.5e11, 7e21, 3e38])
@pytest.mark.parametrize("kw", [
    dict(radius=1), dict(radius=1, group_size=16), dict(radius=1, bm_range=40), dict(radius=1, temporal_mode="legacy")])
def test_clips(gpu, oracle, sigma, kw):
    import torch
    rng = np.random.default_rng(6)
    clip = [[_plane(1.0) + rng.normal(0, 0.02, (H, W)).astype(np.float32)] for _ in range(3)]
    dev = [[torch.from_numpy(p).cuda() for p in f] for f in clip]
    inst = gpu.BM3D("GRAYS", W, H, frames=3, ref=True, sigma=sigma, **kw)
    out = inst.filter_clip(dev, dev)
    p = gpu.parse("GRAYS", W, H, 3, ref=True, sigma=sigma, **kw)
    if kw.get("temporal_mode") == "legacy":
        out = gpu.VAggregate(out, dev, 1)
        want = oracle.vaggregate(oracle.bm3d_clip_legacy(clip, p, ref_clip=clip), clip, 1)
    else:
        want = oracle.bm3d_clip(clip, p, ref_clip=clip)
    got = [f[0].cpu().numpy() for f in out]
    inst.close()
    assert len(got) == 3
    for g, w in zip(got, want):
        assert oracle.psnr(g, w[0]) >= 60.0
