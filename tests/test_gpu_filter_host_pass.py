"""Calls whose batch pass goes to the host, with entries one after another: from the start
(separators that outweigh the reads) or once the device's list of flushes has run over,
with reads that outgrow the LDS slots and with the reads in pieces."""
import pytest

from saruman_amd import workload as wl
from saruman_amd.batch import Context
from test_gpu_filter_batch import same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,lens,families,n,chunks", [
    ("flushes", [60_000], None, 6_000, (2, 3)),
    ("flushes_overflow", [40_000], (3, 300, 600, 40, 0.5, 0.001), 6_000, (5, 20)),
    ("pieces", [60_000], None, 70_000, (25, 50)),
    ("pieces_overflow", [40_000], (2, 300, 600, 40, 0.5, 0.001), 66_000, (80,)),
    ("separators", [2_000_000, 1_000_000], None, 5_000, (7, 1_000)),
    ("separators_overflow", [2_000_000, 500_000], (8, 300, 600, 60, 0.5, 0.001), 4_000, (300,)),
])
def test_host_pass(name, lens, families, n, chunks):
    print(f"[gpu] filter host pass {name}", flush=True)
    genome = wl.synth_genome(71, lens, 0.5, families)
    reads = wl.synth_reads(72, genome, n, 40, 60, 1, p_sub=0.01, p_ins=0.001, indel_max=2, k_rate=0.05)
    ctx = Context(0)
    idx = wl.Index(genome, wl.needed_qs(reads))
    df = wl.DeviceFilter(ctx, idx, genome)
    try:
        for chunk in chunks:
            want = [wl.run_filter(idx, genome, reads, dr, chunk) for dr in (0, 4)]
            if name != "separators" and name != "separators_overflow":
                assert len(want[0].batch_end) > 256, len(want[0].batch_end)
            for w, d in zip(want, df.run_both(reads, chunk)):
                same(w, d, (name, chunk))
            if "overflow" in name:
                assert df.stats()["overflow_reads"] > 0
            same(want[1], df.run(reads, 4, chunk), (name, chunk, "one strand"))
    finally:
        df.close()
        idx.close()
        ctx.close()
