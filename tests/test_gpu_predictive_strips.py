"""Predictive search layers of up to 64 strips (keys in registers) and above
(keys in LDS), around the line: on clips of exact ties every record must equal
the oracle's, entry by entry. No tolerance.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ps_num,ps_range", [(4, 2), (2, 4), (3, 3), (1, 6), (2, 5), (4, 3), (8, 1)])
@pytest.mark.parametrize("group", [8, 16])
def test_records_on_ties(gpu, oracle, ps_num, ps_range, group):
    import torch
    width, height, radius = 61, 43, 2
    y, x = np.mgrid[0:height, 0:width]
    frames = [((((x + 3 * k) // 8 + (y + k) // 8 + ps_num) % 3) * 0.25).astype(np.float32) for k in range(4)]
    dev = torch.from_numpy(np.stack(frames)).cuda()
    grid = oracle.raster_grid(width, height, 8, 7)
    for center in (0, 2):
        rec, cnt = gpu.predictive_match(dev, center, radius, block=8, step=7, bm_range=5, group=group, ps_num=ps_num,
                                        ps_range=ps_range)
        torch.cuda.synchronize()
        rec, cnt = rec.cpu().numpy(), cnt.cpu().numpy()
        n = len(frames)
        planes = [frames[center + min(max(t - radius, -center), n - 1 - center)] for t in range(2 * radius + 1)]
        begin, end = max(0, radius - center), radius + min(radius + 1, n - center)
        for i, (bx, by) in enumerate(grid):
            want = oracle.predictive_match(planes, bx, by, radius, 8, group, 5, ps_num, ps_range, radius, begin, end)
            got = [(int(a), int(b), int(t), float(np.array(d, np.int32).view(np.float32))) for a, b, t, d in rec[i, :cnt[i]]]
            assert got == [(int(a), int(b), int(t), float(d)) for a, b, t, d in want], (center, i)
