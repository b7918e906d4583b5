"""A device filter call that finds no device memory for both strands at once runs one
after the other, and one in pieces starts over without them: results as the host's.  Only
where the reads themselves have no room is the call refused, and the next one runs."""
import pytest

from saruman_amd import _lib, workload as wl
from saruman_amd.batch import Context
from test_gpu_filter_batch import same

pytestmark = pytest.mark.gpu

INPUTS = 3      # the reads with their plan, their codes, their mask


@pytest.mark.parametrize("n,allocs", [(3_000, range(0, 26)), (70_000, range(8, 30, 3))])
def test_one_strand_at_a_time(n, allocs):
    lib = _lib.load()
    genome = wl.synth_genome(91, [60_000], 0.5, (3, 300, 600, 40, 0.5, 0.001))
    reads = wl.synth_reads(92, genome, n, 36, 60, 1, p_sub=0.01, p_ins=0.001, indel_max=2, k_rate=0.05)
    idx = wl.Index(genome, wl.needed_qs(reads))
    want = [wl.run_filter(idx, genome, reads, dr, 1_000) for dr in (0, 4)]
    for after in allocs:
        print(f"[gpu] filter room {n} {after}", flush=True)
        ctx = Context(0)
        df = wl.DeviceFilter(ctx, idx, genome)
        try:
            lib.srm_debug_fail_filter_allocs(after, 1)
            try:
                if n < 32_768 and after < INPUTS:
                    with pytest.raises(Exception, match="hipMalloc"):
                        df.run_both(reads, 1_000)
                    got = df.run_both(reads, 1_000)
                else:
                    got = df.run_both(reads, 1_000)
            finally:
                lib.srm_debug_fail_filter_allocs(0, 0)
            for w, d in zip(want, got):
                same(w, d, (n, after))
        finally:
            df.close()
            ctx.close()
    idx.close()
