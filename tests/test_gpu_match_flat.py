"""Matcher records over constant regions, which the MFMA matcher answers without
scoring: records equal the FP32 matchers' bit for bit (the first places of the
window). Constants at the ends of the exponent range, both zeros, planes that
leave the constant in one last place of one pixel, planes and windows smaller
than a block of references or a group, staged and unstaged regions. No
tolerance.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _planes(width, height):
    for v in (0.0, 0.25, -3.5, 1e-40, 1e-45, 65504.0, 1e30, 3e38, np.inf, np.nan):
        yield str(v), np.full((height, width), v, np.float32)
    zeros = np.zeros((height, width), np.float32)
    zeros[::2, ::3] = -0.0
    yield "both zeros", zeros
    for v in (0.25, 1e-40, 1e-45):
        for y, x in ((0, 0), (height - 1, width - 1), (height // 2, width // 2)):
            p = np.full((height, width), v, np.float32)
            p[y, x] = np.nextafter(np.float32(v), np.float32(np.inf), dtype=np.float32)
            yield f"{v}, one pixel {y} {x}", p


def _records(gpu, plane, path, *args):
    import torch
    gpu.set_match_path(path)
    try:
        rec, cnt = gpu.spatial_match(torch.from_numpy(plane).cuda(), 8, *args)
        torch.cuda.synchronize()
        rec, cnt = rec.cpu().numpy(), cnt.cpu().numpy()
    finally:
        gpu.set_match_path(gpu.MATCH_AUTO)
    live = np.arange(rec.shape[1])[None, :] < cnt[:, None]
    return np.where(live[..., None], rec, 0), cnt


@pytest.mark.parametrize("step,rng,group,width,height", [
    (3, 9, 16, 61, 43), (8, 10, 8, 64, 40), (1, 1, 32, 19, 17), (4, 3, 32, 8, 8), (5, 12, 32, 8, 41),
    (2, 17, 32, 47, 9), (8, 30, 16, 131, 77), (8, 64, 32, 190, 140)])
def test_flat_regions(gpu, step, rng, group, width, height):
    for name, plane in _planes(width, height):
        want = _records(gpu, plane, gpu.MATCH_FP32, step, rng, group)
        got = _records(gpu, plane, gpu.MATCH_MFMA, step, rng, group)
        assert np.array_equal(want[1], got[1]), name
        assert np.array_equal(want[0], got[0]), name
