"""Allocations that fail and are recovered from leave no error behind for the next launch:
page-locked memory that is not to be had, and a device filter whose call in pieces finds
no room for the totals that it guessed."""
import numpy as np
import pytest

import saruman_amd as sa
from saruman_amd import _lib, workload as wl
from saruman_amd.batch import Context
from saruman_amd.testing import random_batch
from test_gpu_filter_batch import same

pytestmark = pytest.mark.gpu


def test_page_locked_memory_that_is_not_to_be_had(orc):
    print("[gpu] alloc errors: host", flush=True)
    lib = _lib.load()
    batch = random_batch(np.random.default_rng(41), 300, L=100, k=5)
    assert not lib.srm_host_alloc(1 << 60)
    got = sa.align_batch(batch, kernel="banded")
    assert got.records == orc.align_batch(batch).records


@pytest.mark.parametrize("after", range(8))
def test_no_room_for_guessed_totals(after):
    """Allocations of the call in pieces: its inputs, the three list arrays, the sums, the
    output, the reads' codes and mask."""
    print(f"[gpu] alloc errors: pieces {after}", flush=True)
    lib = _lib.load()
    genome = wl.synth_genome(91, [60_000], 0.5)
    reads = wl.synth_reads(92, genome, 70_000, 36, 60, 1, p_sub=0.01, p_ins=0.001, indel_max=2,
                           k_rate=0.05)
    ctx = Context(0)
    idx = wl.Index(genome, wl.needed_qs(reads))
    df = wl.DeviceFilter(ctx, idx, genome)
    try:
        lib.srm_debug_fail_filter_allocs(after, 1)
        try:
            got = df.run_both(reads, 20_000)
        finally:
            lib.srm_debug_fail_filter_allocs(0, 0)
        for dr, d in zip((0, 4), got):
            same(wl.run_filter(idx, genome, reads, dr, 20_000), d, dr)
    finally:
        df.close()
        idx.close()
        ctx.close()
