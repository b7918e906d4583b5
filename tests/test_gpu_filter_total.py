"""A call whose q-gram lists hold more entries than 32 bits count is refused, through
the upload in pieces, and the next calls on the handle are as before."""
import pytest

from saruman_amd import workload as wl
from saruman_amd.batch import Context
from test_gpu_filter_batch import same

pytestmark = pytest.mark.gpu


def test_too_many_list_entries():
    print("[gpu] filter total", flush=True)
    # q = 7: 10 lists a read of 4 Mbp / 4^7 = 244 positions
    genome = wl.synth_genome(95, [4_000_000], 0.5)
    n, L = 2_000_000, 36
    reads = wl.synth_reads(96, genome, n, L, L, 1, p_sub=0.01, p_ins=0.001, indel_max=2, k_rate=0.05)
    reads.k[:] = 4
    ctx = Context(0)
    idx = wl.Index(genome, wl.needed_qs(reads))
    df = wl.DeviceFilter(ctx, idx, genome)
    try:
        with pytest.raises(Exception, match="more than 4294967040 positions"):
            df.run_both(reads, 1_000_000)
        few = wl.Reads(reads.seq[:3_000 * L], reads.off[:3_000], reads.length[:3_000],
                       reads.true_pos[:3_000], reads.strand[:3_000], reads.k[:3_000])
        for dr, d in zip((0, 4), df.run_both(few, 1_000)):
            same(wl.run_filter(idx, genome, few, dr, 1_000), d, dr)
            assert len(d.read) > 500
    finally:
        df.close()
        idx.close()
        ctx.close()
