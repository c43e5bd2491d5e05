"""Two page registers, hits from one pass over the records, bit-exact against
the CPU oracle: a tile's first record on a plane takes its hit from the tiles
before it, all others from the pass itself.  Tiles of one, three and seventy
steps, streams that end inside a step, runs of lines that return to a few pages
per plane (whole, split and broken steps), and planes whose registers fill in
the middle of the stream."""
from __future__ import annotations

import numpy as np
import pytest

import parity
from hbfsim_amd import workloads
from test_gpu_parity import C0, C2

pytestmark = pytest.mark.gpu

PAGE = 16384


def runs_stream(n, seed, planes, pages_per_plane, shortest):
    """Runs of consecutive lines, each inside one of a few pages per plane; a
    step's 64 records share one issue time.  The second half of the stream
    reads planes that the first half leaves alone."""
    rng = np.random.default_rng(seed)
    length = rng.integers(shortest, 129, n // shortest + 2)
    length = length[: int(np.searchsorted(np.cumsum(length), n)) + 1]
    page = (rng.integers(0, planes // 2, len(length)) +
            planes * rng.integers(0, pages_per_plane, len(length)))
    first = rng.integers(0, 129 - length)
    run = np.repeat(np.arange(len(length)), length)[:n]
    at = np.arange(n) - (np.cumsum(length) - length)[run]
    late = np.where(np.arange(n) >= n // 2, planes // 2, 0)
    rec = np.zeros((n, 4), np.uint64)
    rec[:, 0] = (workloads.RANGE_BASE + (page[run] + late) * PAGE +
                 (first[run] + at) * 128).astype(np.uint64)
    rec[:, 1] = 128
    rec[:, 2] = (np.arange(n) // 64 * 50_000).astype(np.uint64)
    return rec


@pytest.mark.parametrize("profile,planes", [(C0, 64), (C2, 512)], ids=["c0", "c2"])
@pytest.mark.parametrize("tile", [64, 64 * 3, 64 * 70])
@pytest.mark.parametrize("n", [1, 63, 64, 4 * 64 + 1, 30_001])
@pytest.mark.parametrize("shortest", [1, 48])
def test_hits_from_one_pass(profile, planes, tile, n, shortest):
    ranges = [(workloads.RANGE_BASE, 1 << 30, 1)]
    p = parity.Pair(profile, ranges, page_buffers=2, tile_records=tile)
    try:
        for k in range(2):  # from empty registers, then from those it leaves
            rec = runs_stream(n, 17 * n + k, planes, 3, shortest)
            g, c = p.run(rec, k * 10**11)
            parity.assert_same(g, c, f"{profile.name} tile {tile} n {n} run {k}")
        p.check_state()
    finally:
        p.close()
