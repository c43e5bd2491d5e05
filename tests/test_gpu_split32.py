"""Split steps of 32-byte records, bit-exact against the CPU oracle: the
streams of tests/test_gpu_split.py (page crossings, joined spans of one or two
ranges, broken lines, writes) with one page register, with two (given hits per
run) and in hybrid mode, on tiles that end inside batches, over two runs."""
from __future__ import annotations

import numpy as np
import pytest

import parity
from test_gpu_parity import C0, C2
from test_gpu_split import ranges_for, split_stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("profile", [C0, C2], ids=["c0", "c2"])
@pytest.mark.parametrize("options", [
    dict(), dict(page_buffers=2), dict(page_buffers=2, plane_contention=0),
    dict(plane_contention=0), dict(transfer_page=1), dict(tile_records=64 * 8),
    dict(page_buffers=2, tile_records=64 * 70), dict(page_buffers=0)])
@pytest.mark.parametrize("kinds", [None, {"cross": 1.0}, {"join": 0.5, "join_same": 0.5}])
def test_split_steps(profile, options, kinds):
    ranges = ranges_for()
    p = parity.Pair(profile, ranges, **options)
    try:
        for k in range(2):
            rec = split_stream(31 + k, 1200, ranges, kinds)
            # (above 2^18 records tiles of runs go to the batched passes)
            rec = np.concatenate([rec] * 4)
            t = rec[: len(rec) // 4, 2].copy()
            for j in range(1, 4):
                rec[j * len(t):(j + 1) * len(t), 2] = t + j * t[-1]
            g, c = p.run(rec, k * 10**11)
            parity.assert_same(g, c, f"{profile.name} {options} run {k}")
            if options.get("page_buffers") != 0:  # (without page registers nothing is batched)
                p.check_batched()
        p.check_state()
    finally:
        p.close()


def test_split_steps_hybrid(tmp_path):
    import json
    prof = json.loads(C2.read_text())
    prof.update(reference_sample_rate=0.1, reference_warmup_requests=50)
    path = tmp_path / "hybrid.json"
    path.write_text(json.dumps(prof))
    ranges = ranges_for()
    p = parity.Pair(path, ranges, mode="hybrid")
    try:
        g, c = p.run(split_stream(5, 3000, ranges))
        parity.assert_same(g, c, "hybrid")
        p.check_state()
    finally:
        p.close()
