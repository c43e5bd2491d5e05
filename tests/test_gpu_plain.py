"""The scattered-record passes (k_plain_summary, k_plain_apply) where they can
go wrong, bit-exact against the CPU oracle: runs taken whole (up to 2^18
records) and run beside the batched passes (tiles of runs of lines between
scattered ones), partial steps and tiles, byte counts that differ within a step,
page-register options, records that bypass or are refused, range tables of 1 to
129 ranges and range ends, both record forms, services beyond 32-bit steps."""
from __future__ import annotations

import numpy as np
import pytest

import parity
from hbfsim_amd import workloads as w
from test_gpu_parity import C0, C2

pytestmark = pytest.mark.gpu
PITCH = 3 << 20


def ranges_of(count):
    # odd lengths, a read-only one, neighbours that touch
    return [(w.RANGE_BASE + k * PITCH, PITCH if k % 3 == 1 else (2 << 20) + 4096 * k + 512,
             1 if k % 5 == 2 else 3) for k in range(count)]


def scattered(n, ranges, seed, sizes=(128,), writes=0.1, gap=2000, strange=0.05):
    rng = np.random.default_rng(seed)
    r = rng.integers(0, len(ranges), n)
    base = np.array([x[0] for x in ranges], np.uint64)[r]
    length = np.array([x[1] for x in ranges], np.uint64)[r]
    size = rng.choice(np.array(sizes, np.uint64), n)
    rec = np.zeros((n, 4), np.uint64)
    rec[:, 0] = base + rng.integers(0, 1 << 62, n, np.uint64) % (length // 128) * 128
    rec[:, 1] = size
    rec[:, 2] = np.cumsum(rng.integers(0, 2 * gap + 1, n))
    rec[:, 3] = rng.random(n) < writes
    odd = np.nonzero(rng.random(n) < strange)[0]
    kind = rng.integers(0, 6, len(odd))
    end = base[odd] + length[odd]
    rec[odd, 0] = np.select([kind == 0, kind == 1, kind == 2, kind == 3],
                            [end, end - 64, base[odd] - 64, base[odd] + 16384 - 64],
                            rec[odd, 0])
    rec[odd[kind == 4], 1] = 0
    rec[odd[kind == 5], 3] = 7
    return rec


def lines(n, ranges, seed):
    """Runs of 128-byte lines, 256 at one issue time."""
    k = np.arange(n, dtype=np.uint64)
    rec = np.zeros((n, 4), np.uint64)
    rec[:, 0] = np.uint64(ranges[0][0]) + (k % 8192) * 128
    rec[:, 1] = 128
    rec[:, 2] = k // 256 * 64_000
    return rec


def check(rec, ranges, profile=C0, runs=2, **options):
    for packed in (True, False):
        p = parity.Pair(profile, ranges, **options)
        try:
            for k in range(runs):
                base = k * 10**10
                g, c = (p.run_packed if packed else p.run)(rec, base)
                parity.assert_same(g, c, f"packed={packed} run {k} {options}")
            p.check_state()
        finally:
            p.close()


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 4099, (1 << 18) - 1, (1 << 18) + 63])
@pytest.mark.parametrize("profile", [C0, C2])
def test_sizes(n, profile):
    ranges = ranges_of(5)
    check(scattered(n, ranges, n), ranges, profile)


@pytest.mark.parametrize("count", [1, 2, 3, 64, 65, 127, 128, 129])
def test_range_counts(count):
    ranges = ranges_of(count)
    check(scattered(20_000, ranges, count, strange=0.2), ranges)


@pytest.mark.parametrize("options", [
    {"page_buffers": 0}, {"plane_contention": 0}, {"transfer_page": 1},
    {"program_every_write": 1}, {"xfer_quantum_ps": 1000}, {"tile_records": 16384},
    {"flat_geometry": 1}])
@pytest.mark.parametrize("sizes", [(128,), (64, 128, 100, 4096)])
def test_options_and_sizes(options, sizes):
    ranges = ranges_of(7)
    check(scattered(30_000, ranges, len(sizes), sizes, writes=0.4), ranges, C0, **options)


@pytest.mark.parametrize("gap", [1, 200_000, 30_000_000])
def test_gaps(gap):
    """Crowded, half-idle and idle resources; gaps beyond the 32-bit step."""
    ranges = ranges_of(3)
    check(scattered(20_000, ranges, gap, gap=gap), ranges, C2)


def test_tiles_of_lines_between_scattered_ones():
    """Tiles of each kind in one run, and a tile that turns from one to the
    other half way."""
    ranges = ranges_of(4)
    parts, t = [], 0
    for k, n in enumerate((70_000, 64 * 1024, 30_001, 300_000, 64 * 500, 50_000)):
        r = lines(n, ranges, k) if k % 2 else scattered(n, ranges, k)
        r[:, 2] += np.uint64(t)
        t = int(r[:, 2].max()) + 1000
        parts.append(r)
    check(np.concatenate(parts), ranges, C0)
    check(np.concatenate(parts), ranges, C0, tile_records=4096)


def test_which_passes_took_the_tiles():
    """The tile counts by pass: a short run, one of mostly scattered tiles, hybrid mode and the
    state before a run."""
    ranges = ranges_of(3)
    p = parity.Pair(C0, ranges)
    try:
        assert p.engine.last_tiles() == (0, 0)
        p.run_packed(scattered(4099, ranges, 1))
        batched, taken = p.engine.last_tiles()
        assert batched == 0 and taken == -(-4099 // 64)
        assert p.engine.apply_waves() == 4  # k_plain_apply's
    finally:
        p.close()
    p = parity.Pair(C0, ranges)  # (no run before it that mostly hit its registers)
    try:
        n = (1 << 18) + 4096
        rec = scattered(n, ranges, 2)
        rec[:65536] = lines(65536, ranges, 3)
        rec[65536:, 2] += np.uint64(int(rec[65535, 2]))
        p.run_packed(rec)
        batched, taken = p.engine.last_tiles()
        assert batched + taken == -(-n // 256) and batched == 65536 // 256
    finally:
        p.close()
    p = parity.Pair(C0, ranges_of(129))
    try:
        p.run_packed(scattered(4099, ranges, 1))
        assert p.engine.last_tiles() == (-(-4099 // 64), 0)
    finally:
        p.close()


@pytest.mark.parametrize("options", [dict(), dict(plane_contention=0), dict(transfer_page=1),
                                     dict(flat_geometry=1)])
def test_without_page_registers(options):
    """Runs of more than 2^18 records without page registers go to the scattered-record passes
    whole, lines too; with flat geometry the tiles of lines stay with the batched ones."""
    ranges = ranges_of(4)
    n = (1 << 18) + 4097
    rec = scattered(n, ranges, 5)
    rec[:131_072] = lines(131_072, ranges, 6)
    rec[131_072:, 2] += np.uint64(int(rec[131_071, 2]))
    for packed in (True, False):
        p = parity.Pair(C0, ranges, page_buffers=0, **options)
        try:
            for k in range(2):
                g, c = (p.run_packed if packed else p.run)(rec, k * 10**10)
                parity.assert_same(g, c, f"packed={packed} {options} run {k}")
                batched, taken = p.engine.last_tiles()
                assert batched + taken == -(-n // 256)
                assert batched == (131_072 // 256 if "flat_geometry" in options else 0)
            p.check_state()
        finally:
            p.close()
