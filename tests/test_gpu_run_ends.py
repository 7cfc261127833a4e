"""Runs whose part of the destination's first 128-byte line is stored apart from
the rest.  Apart from each other: every place in a line a run can start at,
lengths around lines, steps (1008 bytes) and pairs of steps, nothing written
beside the runs.  End to end, where two wavefronts and more write the same line
with different hints: every start with every length, and so every end."""
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


@pytest.mark.parametrize("src_phase", (0, 2, 7, 12))
def test_runs_end_to_end(ctx, src_phase):
    lens = []
    at = 0
    for start in range(128):
        for n in LENGTHS:
            gap = (start - at) % 128  # a run of its own that brings the next one to its place
            if gap:
                lens.append(gap)
            lens.append(n)
            at = (start + n) % 128
    assert {e % 128 for e in np.cumsum(lens)} == set(range(128))
    total = sum(lens)
    rng = np.random.default_rng(310 + src_phase)
    fill = rng.integers(0, 256, total + 256, dtype=np.uint8)
    want = fill.copy()
    want[:total] = rng.integers(0, 256, total, dtype=np.uint8)
    src_h = np.zeros(total + 32 * len(lens), np.uint8)
    runs, so, do = [], 0, 0
    for n in lens:
        s = so + src_phase
        src_h[s:s + n] = want[do:do + n]
        runs.append((s, do, n))
        so, do = (s + n + 15) // 16 * 16, do + n
    src, dst = torch.from_numpy(src_h).to(DEV), torch.from_numpy(fill).to(DEV)
    assert src.data_ptr() % 16 == 0 and dst.data_ptr() % 128 == 0
    for k in range(0, len(runs), 1000):
        part = runs[k:k + 1000]
        ctx.copy_runs([src.data_ptr() + s for s, _, _ in part], [dst.data_ptr() + d for _, d, _ in part], [n for _, _, n in part])
    got = dst.cpu().numpy()
    assert np.array_equal(got, want), first_diff(got, want)
