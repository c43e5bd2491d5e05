"""The report reduction and the small-run tiles at their edges, against the
oracle: tile reports of one block (up to 128 tiles), of two and of many, runs
that reuse the block counter, and automatic tiles of 64, 128 and 256 records on
either side of their limits.  Kernel times come with every run."""
from __future__ import annotations

import pytest

import parity
from hbfsim_amd import workloads as w
from test_gpu_parity import C0, C2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("profile", [C0, C2])
@pytest.mark.parametrize("n,tile", [
    (1, 64), (64 * 128, 64), (64 * 128 + 1, 64), (64 * 257 - 3, 64), (64 * 1000, 64),  # blocks
    (65_535, 0), (65_537, 0), (131_071, 0), (131_073, 0), (262_145, 0)])             # auto tiles
def test_report(profile, n, tile):
    options = {"tile_records": tile} if tile else {}
    s = w.config0(n=n, seed=n, write_fraction_per_mille=60)
    p = parity.Pair(profile, s.ranges, **options)
    try:
        for k in range(2):
            g, c = p.run_packed(s.records, base_ps=k * 10**9)
            parity.assert_same(g, c, f"n={n} tile={tile} run {k}")
        p.check_state()
        ms = p.engine.kernel_ms()
        assert len(ms) == 3 and all(0 < x < 1000 for x in ms)
    finally:
        p.close()
