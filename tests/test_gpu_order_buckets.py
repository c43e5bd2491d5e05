"""The bucket sort behind streams out of issue order, at the sizes and time
distributions where its forms change: bucket counts and partition chunks
(8,192 records), many records with one issue time, buckets that overflow LDS
and spans whose bucket keys need more than 32 bits (both radix-sorted), against
the same engine run on numpy's stable order, and small ones against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

import parity
from hbfsim_amd import workloads as w
from test_gpu_order import sorted_pair_run
from test_gpu_parity import C0

pytestmark = pytest.mark.gpu
RANGES = [(w.RANGE_BASE, 1 << 30, 3)]


def stream(n, shape, seed):
    rng = np.random.default_rng(seed)
    rec = np.zeros((n, 4), np.uint64)
    rec[:, 0] = np.uint64(w.RANGE_BASE) + rng.integers(0, (1 << 30) // 128, n, np.uint64) * 128
    rec[:, 1] = 128
    rec[:, 3] = rng.random(n) < 0.05
    t = {"spread": lambda: rng.integers(0, 2000 * n, n),
         "ties": lambda: rng.integers(0, max(2, n // 300), n) * 64_000,
         "two": lambda: rng.integers(0, 2, n) * 1000,                 # overflows a bucket
         "late": lambda: np.where(np.arange(n) < 3, 2**50, rng.integers(0, 2000 * n, n)),
         "wide": lambda: rng.integers(0, 2**54, n),                   # keys beyond 32 bits
         "shift": lambda: 7_777_777 + rng.integers(0, n, n)}[shape]()
    rec[:, 2] = t.astype(np.uint64)
    rec[-1, 2] = rec[:, 2].min()  # goes back at the end at least
    return rec


@pytest.mark.parametrize("packed", [True, False])
@pytest.mark.parametrize("n,shape", [
    (3, "spread"), (257, "ties"), (8191, "spread"), (8193, "shift"), (16_385, "spread"),
    (40_000, "ties"), (50_000, "two"), (20_000, "late"), (5000, "wide"), (300_001, "spread")])
def test_bucketed_order(n, shape, packed):
    rec = stream(n, shape, n)
    p, q = parity.Pair(C0, RANGES), parity.Pair(C0, RANGES)
    try:
        g, c = p.run_packed(rec) if packed else p.run(rec)
        if c is not None:
            parity.assert_same(g, c, f"{n} {shape}")
        comp, st, rep = sorted_pair_run(q, rec, packed)
        np.testing.assert_array_equal(g[0], comp)
        np.testing.assert_array_equal(g[1], st)
        assert g[2] == rep
    finally:
        p.close()
        q.close()


@pytest.mark.parametrize("packed", [True, False])
@pytest.mark.parametrize("per", [12, 48, 64, 95, 96, 97, 98, 120, 1000, 2049, 4095, 4096, 4097])
def test_many_records_of_one_time(per, packed):
    """`per` records share each issue time: told apart by comparing up to 96 in a sub-bucket, by
    the sorting network up to the 4,096 that a bucket holds, by the radix sort beyond."""
    n = 63 * 4096 + 11
    rec = stream(n, "spread", per)
    rec[:, 2] = np.random.default_rng(per).permutation(np.arange(n) // per).astype(np.uint64)
    rec[:, 2] *= np.uint64(2000 * per)
    p, q = parity.Pair(C0, RANGES), parity.Pair(C0, RANGES)
    try:
        g, c = p.run_packed(rec) if packed else p.run(rec)
        parity.assert_same(g, c, f"{per} records a time")
        comp, st, rep = sorted_pair_run(q, rec, packed)
        np.testing.assert_array_equal(g[0], comp)
        np.testing.assert_array_equal(g[1], st)
        assert g[2] == rep
    finally:
        p.close()
        q.close()
