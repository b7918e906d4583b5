"""The record writers' tiles (8 to 64 candidates a wave, by the candidates of a launch):
the device's text equals the host formatter's around each change, short and long lines
mixed."""
import dataclasses

import pytest

import saruman_amd as sa
from saruman_amd import workload as wl
from test_gpu_pipeline import host_text

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def aligned():
    genome = wl.synth_genome(7, [400_000], 0.5, (4, 300, 600, 30, 0.3, 0.01))
    reads = wl.synth_reads(8, genome, 420_000, 36, 60, 1, p_sub=0.01, p_ins=0.001, indel_max=2, k_rate=0.05)
    index = wl.Index(genome, wl.needed_qs(reads))
    ctx = sa.Context(0)
    ctx.set_genome(wl.genome_words(genome))
    df = wl.DeviceFilter(ctx, index, genome)
    strands = df.run_both(reads, 1_000_000)
    df.close()
    index.close()
    yield ctx, genome, reads, wl.batches_by_reads(reads, strands, reads.n)[0][2]
    ctx.close()


# a launch of at least 4,096 tiles of 64, 32 or 16 candidates takes that size
@pytest.mark.parametrize("n", [1, 7, 8, 9, 65_535, 65_536, 131_071, 131_072, 262_143, 262_150])
def test_text(aligned, n):
    ctx, genome, reads, db = aligned
    assert db.n >= 262_150
    print(f"[gpu] record tiles {n}", flush=True)
    part = dataclasses.replace(db, cand=db.cand[:n], pos=db.pos[:n], read_id=db.read_id[:n])
    job = sa.Job(ctx)
    try:
        job.upload(0, 1, part.cand, db.read_words, None, ops_total=db.ops_total)
        job.set_records(part.pos, read_id=part.read_id.astype("int32"), prefix="r")
        job.run("banded")
        text = job.records_text()[0]
        res, ops = job.download()
    finally:
        job.close()
    assert text == host_text(sa.load(), part, reads, 0, genome, res, ops)
