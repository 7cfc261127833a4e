"""Runs whose part of the destination's first 128-byte line is stored apart from
the rest: every place in a line a run can start at and
every place it can end at, lengths around lines, steps (1008 bytes) and pairs of
steps, nothing written beside the runs."""
import numpy as np
import pytest
import torch

from helpers import first_diff

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LENGTHS = (1, 16, 113, 127, 128, 129, 144, 255, 256, 257, 383, 895, 1007, 1008, 1025, 1400, 2015, 2016, 2017, 2144, 4100)


@pytest.mark.parametrize("src_phase", (0, 2, 7, 12))
def test_every_place_in_a_line(ctx, src_phase):
    rng = np.random.default_rng(300 + src_phase)
    size = 1 << 21
    src_h = rng.integers(0, 256, size, dtype=np.uint8)
    fill = rng.integers(0, 256, size, dtype=np.uint8)
    want = fill.copy()
    src, dst = torch.from_numpy(src_h).to(DEV), torch.from_numpy(fill).to(DEV)
    assert dst.data_ptr() % 128 == 0
    runs, so, do = [], 0, 0
    for at in range(128):
        for k in range(4):
            n = LENGTHS[(at * 4 + k * 5) % len(LENGTHS)]
            s, d = so + src_phase, do + at
            runs.append((s, d, n))
            want[d:d + n] = src_h[s:s + n]
            so, do = (s + n + 31) // 16 * 16, (d + n + 127) // 128 * 128 + 128
    assert so < size and do < size
    for k in range(0, len(runs), 500):
        part = runs[k:k + 500]
        ctx.copy_runs([src.data_ptr() + s for s, _, _ in part], [dst.data_ptr() + d for _, d, _ in part], [n for _, _, n in part])
    got = dst.cpu().numpy()
    assert np.array_equal(got, want), first_diff(got, want)
