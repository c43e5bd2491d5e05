"""Streams out of issue order at the sizes where the sort changes form: 8,192 buckets up to
2^23 records, 16,384 (whose histogram is 64 KB of LDS) up to 2^25, the radix sort beyond.  Each
against the same engine run on torch's stable order of the issue times."""
from __future__ import annotations

import pytest

from hbfsim_amd import workloads as w
from test_gpu_parity import C0

pytestmark = pytest.mark.gpu
LENGTH = 1 << 30


def stream(n, seed):
    """Random lines, one in twenty a write, at random times over 2 ns a record."""
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def draw(hi):
        return torch.randint(0, hi, (n,), generator=g, device="cuda", dtype=torch.int64)
    rec = torch.stack([w.RANGE_BASE + draw(LENGTH // 128) * 128, torch.full_like(draw(2), 128),
                       draw(2000 * n), (draw(20) == 0).long()], dim=1)
    rec[-1, 2] = 0  # goes back at the end at least
    return rec


def run(rec, packed):
    import torch
    from hbfsim_amd import engine as eng
    n = rec.shape[0]
    comp = torch.empty(n, dtype=torch.int64, device="cuda")
    status = torch.empty(n, dtype=torch.uint8, device="cuda")
    e = eng.Engine(str(C0))
    try:
        e.register(w.RANGE_BASE, LENGTH, 3)
        if packed:
            report = e.run_packed(eng.pack_records(rec), comp, status)
        else:
            report = e.run(rec.contiguous(), comp, status)
        return comp, status, report, e.busy_totals()
    finally:
        e.close()


@pytest.mark.parametrize("packed", [True, False])
@pytest.mark.parametrize("n", [(1 << 23) - 1, (1 << 23) + 1, (1 << 25) - 1, (1 << 25) + 17])
def test_large_streams_out_of_order(n, packed):
    import torch
    rec = stream(n, n)
    comp, status, report, busy = run(rec, packed)
    order = torch.sort(rec[:, 2], stable=True).indices
    scomp, sstatus, sreport, sbusy = run(rec[order], packed)
    assert torch.equal(comp[order], scomp)
    assert torch.equal(status[order], sstatus)
    assert report == sreport
    assert all((a == b).all() for a, b in zip(busy, sbusy))


@pytest.mark.parametrize("n,skewed", [((1 << 25) + 17, False), ((1 << 25) - 1, True)])
def test_radix_sort_within_its_memory(n, skewed):
    """The radix sort of 32-byte records needs 45 bytes of scratch a record, its keys given back
    before the sorted copy is laid out (69 side by side), whether it takes the stream by its size
    or after the bucket sort could not (half the records in a thousandth of the span)."""
    import torch
    from hbfsim_amd import engine as eng
    rec = stream(n, n)
    if skewed:
        rec[::2, 2] //= 1000
    rec = rec.contiguous()
    comp = torch.empty(n, dtype=torch.int64, device="cuda")
    status = torch.empty(n, dtype=torch.uint8, device="cuda")
    e = eng.Engine(str(C0))
    try:
        e.register(w.RANGE_BASE, LENGTH, 3)
        order = torch.sort(rec[:, 2], stable=True).indices
        in_order = rec[order]
        want = e.run(in_order, comp, status)  # also lays out the engine's own arrays
        wcomp = torch.empty_like(comp)
        wcomp[order] = comp
        del in_order, order
        e.reset()
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        room = 45 * n + (256 << 20)
        filler = torch.empty(torch.cuda.mem_get_info()[0] - room, dtype=torch.uint8, device="cuda")
        got = e.run(rec, comp, status)
        del filler
        assert torch.equal(comp, wcomp)
        assert got == want
    finally:
        e.close()
        torch.cuda.empty_cache()
