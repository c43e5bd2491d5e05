"""The hybrid model's class table and combined sort key at the sizes where
their forms change, against the oracle: batches whose classes outgrow the
first table (2^16 slots) and the counted numbering (8,192 classes), latencies
that need 32-bit, 64-bit and split sort keys, and parts of 512 samples.
Everything but the logarithm statistics is exact; those are double sums (at
most 4e5 terms in a tree of depth 30, relative error below 30 * 2^-53 of the
largest partial sum), checked to 1e-12 as elsewhere."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_py

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hy():
    import torch
    assert torch.cuda.is_available()
    from hbfsim_amd import hybrid
    return hybrid


def classes_of(rng, n, classes, order="random"):
    pool = np.zeros((classes, 4), np.uint64)
    pool[:, 0] = np.arange(classes) % 2
    pool[:, 1] = rng.integers(0, 2**32, classes)
    pool[:, 3] = np.arange(classes)
    pick = rng.integers(0, classes, n) if order == "random" else np.arange(n) % classes
    return np.ascontiguousarray(pool[pick].astype(np.uint32))


@pytest.mark.parametrize("n,classes,top", [
    (511, 1, 200), (512, 1, 200), (1025, 2, 2**31), (4097, 4097, 1000),
    (100_000, 8192, 5000), (100_000, 8193, 5000),      # counted and sorted numbering
    (70_000, 70_000, 2**20), (400_000, 150_000, 2**40), (65_536, 7, 900),  # larger tables
    (200_000, 3, 2**63), (200_000, 5, 2**64 - 1)])       # 64-bit and split keys
def test_calibrator_forms(hy, n, classes, top):
    rng = np.random.default_rng(n + classes)
    acc = classes_of(rng, n, classes, "each" if n == classes else "random")
    lat = rng.integers(1, top, n, dtype=np.uint64)
    lat[rng.integers(0, n)] = np.uint64(top)
    c = hy.Calibrator()
    c.observe_batch(acc, lat)
    got = c.estimates()
    want = oracle_py.calibrate(acc, lat)
    assert len(got) == len(want)
    for (cls, e), r in zip(got.items(), want):
        assert cls == tuple(int(r[f]) for f in ("operation", "bytes", "queue_bucket",
                                                "locality_bucket"))
        assert (e.count, e.mean_ns, e.p50_ns, e.p95_ns, e.p99_ns) == \
            tuple(int(r[f]) for f in ("count", "mean_ns", "p50_ns", "p95_ns", "p99_ns")), cls
        assert e.log_mean == pytest.approx(float(r["log_mean"]), rel=1e-12, abs=1e-12)
        assert e.log_sigma == pytest.approx(float(r["log_sigma"]), rel=1e-12, abs=1e-12)


@pytest.mark.parametrize("n,classes", [(1, 1), (257, 256), (90_000, 80_000), (300_000, 300_000)])
def test_sampler_table_growth(hy, n, classes):
    """Two batches; the second holds old classes and new ones."""
    rng = np.random.default_rng(n)
    acc = classes_of(rng, n, classes, "each")[rng.permutation(n)]
    half = n // 2
    both = np.concatenate([acc[:half], acc])
    seq = np.arange(len(both), dtype=np.uint64)
    want = oracle_py.sampler_run(2, 0.01, 11, both, seq)
    s = hy.HybridSampler(2, 0.01, 11)
    a, ca = s.reference_batch(both[:half]) if half else (None, 0)
    b, cb = s.reference_batch(both[half:], first_sequence=half)
    got = np.concatenate([x.cpu().numpy() for x in (a, b) if x is not None])
    np.testing.assert_array_equal(got, want)
    assert ca + cb == int(want.sum())
    s.close()


@pytest.mark.parametrize("sizes,wide", [
    ([511, 512, 513, 1, 2, 1023, 1024, 1025, 3, 4096, 30], False),      # a wave per class
    ([100_000] + [1] * 30_000 + [700, 33, 1024], False),                # eight lanes, whole parts
    ([513] * 40 + [1] * 9_000, True)])                                  # split keys, both
def test_calibrator_parts_and_lanes(hy, sizes, wide):
    """Classes that begin and end anywhere within runs of 512 sorted samples, summed by a wave or
    by eight lanes each; classes of one sample, whose deviation is zero."""
    rng = np.random.default_rng(len(sizes))
    pool = np.zeros((len(sizes), 4), np.uint64)
    pool[:, 1] = 1 + np.arange(len(sizes))
    pool[:, 2] = rng.integers(0, 2**32, len(sizes))
    acc = np.repeat(pool, sizes, axis=0)[rng.permutation(sum(sizes))].astype(np.uint32)
    top = 2**63 if wide else 2**30
    lat = rng.integers(1, top, len(acc), dtype=np.uint64)
    c = hy.Calibrator()
    c.observe_batch(acc, lat)
    got = c.estimates()
    want = oracle_py.calibrate(acc, lat)
    assert len(got) == len(want) == len(sizes)
    for (cls, e), r in zip(got.items(), want):
        assert cls == tuple(int(r[f]) for f in ("operation", "bytes", "queue_bucket",
                                                "locality_bucket"))
        assert (e.count, e.mean_ns, e.p50_ns, e.p95_ns, e.p99_ns) == \
            tuple(int(r[f]) for f in ("count", "mean_ns", "p50_ns", "p95_ns", "p99_ns")), cls
        assert e.log_mean == pytest.approx(float(r["log_mean"]), rel=1e-12, abs=1e-12)
        assert e.log_sigma == pytest.approx(float(r["log_sigma"]), rel=1e-12, abs=1e-12)


@pytest.mark.parametrize("n,classes", [(70_000, 70_000), (300_000, 120_000)])
def test_zero_latency_is_found_past_the_first_table(hy, n, classes):
    """A batch whose first table is given up early still has every latency checked."""
    import ctypes

    import torch
    from hbfsim_amd import _native as nat
    rng = np.random.default_rng(n)
    acc = hy.access_tensor(classes_of(rng, n, classes))
    lat = torch.from_numpy(rng.integers(1, 1000, n)).cuda()
    lat[n - 1] = 0
    rows = torch.empty((n, 9), dtype=torch.int64, device="cuda")
    count = ctypes.c_size_t()
    rc = nat.load().hbfsim_amd_calibrate(acc.data_ptr(), lat.data_ptr(), n, rows.data_ptr(), n,
                                         ctypes.byref(count), None)
    assert rc == nat.HBFSIM_INVALID_ARGUMENT and count.value == 0
