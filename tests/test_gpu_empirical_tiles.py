"""The empirical model's tile passes at the sizes where they can go wrong,
bit-exact against the CPU oracle: tiles of 2,048 records (eight per thread,
four waves), streaks that start on either side of thread, wave and tile ends,
tiles that hold one streak or no modeled record, streaks over several tiles up
to the 1,023 cap, and streams out of issue order."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_empirical import BASE, PAGE, burst_stream, check_burst, make_pair

import parity

pytestmark = pytest.mark.gpu
PAGES = (64 << 20) // PAGE


def stream(n, streak, seed, outside=0.0, writes=0.1):
    """Streaks of exactly `streak` pages from the stream's start."""
    rng = np.random.default_rng(seed)
    k = np.arange(n)
    start = rng.integers(0, PAGES - streak, n)[k // streak]
    op = (rng.random(n) < writes)[k // streak]
    rec = np.zeros((n, 4), np.uint64)
    rec[:, 0] = BASE + (start + k % streak) * PAGE
    rec[:, 1] = 4096
    rec[:, 2] = np.cumsum(rng.integers(0, 20_000_000, n))
    rec[:, 3] = op
    out = rng.random(n) < outside
    rec[out, 0] = BASE + (70 << 20)
    return rec


@pytest.mark.parametrize("n,streak,outside", [
    (2047, 8, 0.0), (2048, 8, 0.0), (2049, 7, 0.0), (8 * 2048 + 1, 512, 0.0),
    (10_000, 9, 0.3), (10_000, 64, 0.9), (6000, 2048, 0.0), (9000, 3000, 0.02),
    (4096, 1, 0.0), (5000, 4, 1.0), (1, 1, 0.0), (7, 3, 0.0)])
@pytest.mark.parametrize("mode", ["fast", "hybrid"])
def test_tiles(n, streak, outside, mode):
    p = make_pair(mode=mode)
    try:
        for k in range(2):  # the second run goes on from the first's state
            rec = stream(n, streak, n + k, outside)
            g, c = p.run(rec)
            parity.assert_same(g, c, f"n={n} streak={streak} outside={outside} run {k}")
            check_burst(p)
    finally:
        p.close()


@pytest.mark.parametrize("at", [1, 7, 8, 511, 2047, 2048, 4099])
def test_one_record_goes_back(at):
    """The record at `at` is issued before its predecessor (thread, wave and
    tile ends): timed in issue order, the state as after the sorted stream."""
    rec = burst_stream(4100, 3)
    rec[:, 2] += 1000
    rec[at, 2] = rec[at - 1, 2] - np.uint64(500)
    p = make_pair()
    try:
        g, c = p.run(rec)
        parity.assert_same(g, c, f"back at {at}")
        check_burst(p)
    finally:
        p.close()
