"""Matcher records over the MFMA matcher's branches and the automatic choice.

Scales (planes whose values lie near their mean, far from it, or on it),
staged and unstaged regions, windows of copies that end with the first 256
places or only later, windows scored in pieces, partial 4 x 4 blocks, and a
size on each side of every line of the automatic choice. Records must equal
the FP32 matchers' bit for bit; no tolerance.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _plane(kind, width, height):
    rng = np.random.default_rng(width * 7 + height)
    y, x = np.mgrid[0:height, 0:width]
    base = 0.5 + 0.3 * np.sin(x * 0.21) * np.cos(y * 0.17)
    noise = rng.normal(0, 0.05, (height, width))
    if kind == "noise":
        v = base + noise
    elif kind == "near":  # below 2^-6 of the mean
        v = 0.25 + 0.01 * (base + noise)
    elif kind == "far":  # up to 2^5 and more
        v = 40.0 * (base + noise)
    elif kind == "period":  # copies every 16 rows and 24 columns
        v = (base + noise)[:16, :24][y % 16, x % 24]
    elif kind == "bands":  # constant, noisy, constant, one step
        v = np.where((y // 24) % 2 == 0, 0.0625, base + noise)
        v[-12:] = 0.75
    elif kind == "lowconst":  # the noise ends above: late places copy
        v = np.where(y < height // 2, base + noise, 0.5)
    return v.astype(np.float32)


def _records(gpu, plane, path, step, rng, group):
    import torch
    gpu.set_match_path(path)
    try:
        rec, cnt = gpu.spatial_match(torch.from_numpy(plane).cuda(), 8, step, rng, group)
        torch.cuda.synchronize()
        rec, cnt = rec.cpu().numpy(), cnt.cpu().numpy()
    finally:
        gpu.set_match_path(gpu.MATCH_AUTO)
    live = np.arange(rec.shape[1])[None, :] < cnt[:, None]
    return np.where(live[..., None], rec, 0), cnt


@pytest.mark.parametrize("kind", ["noise", "near", "far", "period", "bands", "lowconst"])
@pytest.mark.parametrize("step,rng,group,width,height", [
    (1, 4, 8, 61, 43), (3, 9, 16, 130, 75), (4, 9, 32, 97, 101), (8, 10, 8, 161, 90), (3, 16, 32, 133, 91),
    (2, 17, 16, 70, 150), (8, 30, 16, 201, 149), (5, 41, 32, 190, 140), (8, 64, 32, 210, 200)])
def test_mfma_records(gpu, kind, step, rng, group, width, height):
    plane = _plane(kind, width, height)
    want = _records(gpu, plane, gpu.MATCH_FP32, step, rng, group)
    got = _records(gpu, plane, gpu.MATCH_MFMA, step, rng, group)
    assert np.array_equal(want[1], got[1])
    assert np.array_equal(want[0], got[0])


@pytest.mark.parametrize("step,rng,group,width,height", [
    (8, 17, 16, 128, 96), (8, 18, 16, 128, 96), (3, 10, 16, 240, 236), (3, 10, 16, 256, 256), (3, 10, 32, 256, 256),
    (4, 9, 16, 512, 510), (4, 9, 16, 520, 528), (4, 9, 32, 520, 528), (5, 9, 16, 720, 640), (8, 10, 8, 1032, 1032),
    (20, 10, 8, 300, 200)])
def test_automatic_choice(gpu, step, rng, group, width, height):
    plane = _plane("bands", width, height)
    want = _records(gpu, plane, gpu.MATCH_FP32, step, rng, group)
    got = _records(gpu, plane, gpu.MATCH_AUTO, step, rng, group)
    assert np.array_equal(want[1], got[1])
    assert np.array_equal(want[0], got[0])
