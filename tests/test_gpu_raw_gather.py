"""Candidates on raw bytes whose own bytes are gathered at the upload (few of them) and
those that take the whole arrays (many), against the oracle: the last and first
candidates among them, the smallest reads, and costs whose kernel keeps the matrix."""
import numpy as np
import pytest

import saruman_amd as sa
from oracle import oracle as orc
from saruman_amd.testing import random_batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,L,k,raw,costs", [
    (600, (1, 90), 2, [0], (0, 1)), (600, (20, 250), 5, [599], (0, 1)),
    (600, (20, 250), 5, range(0, 600, 40), (0, 1)), (600, (20, 250), 5, range(0, 600, 2), (0, 1)),
    (17_000, (20, 60), 2, range(3, 17_000, 500), (0, 1)), (300, (20, 90), 3, range(0, 300, 30), (0, 20))])
def test_raw_bytes(n, L, k, raw, costs):
    print(f"[gpu] raw bytes {n} {L} {len(raw)} {costs}", flush=True)
    rng = np.random.default_rng(n + len(raw))
    batch = random_batch(rng, n, L=L, k=k, match=costs[0], mismatch=costs[1])
    for t in raw:
        for what in (batch.windows, batch.reads):
            b = bytearray(what[t])
            if b:
                b[int(rng.integers(0, len(b)))] = ord("N")
            what[t] = bytes(b)
    got, want = sa.align_batch(batch, kernel="auto"), orc.align_batch(batch)
    assert got.paths[2] >= len(raw)
    assert list(got.records) == list(want.records)


def test_beside_the_band_in_a_graph():
    """Raw candidates run on a stream of their own: a captured step replayed between eager
    work, and an eager run with the classes one after another, give the same text."""
    from saruman_amd import _lib, tune
    from saruman_amd import workload as wl
    from saruman_amd.batch import Context, Job
    print("[gpu] raw bytes beside the band", flush=True)
    genome = wl.synth_genome(3, [100_000], 0.5)
    reads = wl.synth_reads(4, genome, 20_000, 36, 250, 1, p_sub=0.01, p_ins=0.001, indel_max=2, k_rate=0.05)
    ctx = Context(0)
    idx = wl.Index(genome, wl.needed_qs(reads))
    ctx.set_genome(wl.genome_words(genome))
    strands = [wl.run_filter(idx, genome, reads, dr, 10_000) for dr in (0, 4)]
    fwd = np.frombuffer(reads.seq, np.uint8)
    comp = np.arange(256, dtype=np.uint8)
    comp[list(b"ACGT")] = list(b"TGCA")
    both = np.concatenate([fwd] + [comp[fwd[o:o + n]][::-1] for o, n in zip(reads.off.astype(int), reads.length)])
    code = np.zeros(256, np.uint32)
    code[list(b"ACGT")] = range(4)
    pad = _lib.SRM_CODE_PAD
    codes = np.zeros((2 * pad + len(both) + 15) // 16 * 16 + 16, np.uint32)
    codes[pad:pad + len(both)] = code[both]
    words = (codes.reshape(-1, 16) << np.arange(0, 32, 2, dtype=np.uint32)).sum(1).astype(np.uint32)
    db = wl.device_batch(reads, strands, words)
    raw = np.random.default_rng(5).random(db.n) < 0.03
    db.cand["bits"][raw] = _lib.SRM_CAND_BYTES
    db.cand["win_off"][raw] = db.pos[raw]
    texts = []
    for streams, graph in ((0, False), (0, True), (1, False)):
        tune.apply(ctx, {"blocks_per_cu": [0] * 9, "class_streams": streams})
        job = Job(ctx)
        job.upload(0, 1, db.cand, db.read_words, None, both.tobytes(), genome.seq, ops_total=db.ops_total)
        job.set_records(db.pos, read_id=db.read_id.astype(np.int32), prefix="r")
        job.use_graph(graph)
        for _ in range(4 if graph else 1):
            job.run("auto")
            texts.append(job.records_text()[0])
            job.download()
        job.close()
    tune.apply(ctx, None)
    idx.close()
    ctx.close()
    assert raw.sum() > 100 and len(texts[0]) > 0
    assert all(t == texts[0] for t in texts)
