"""The server's read codes from the device filter: the records of requests whose reads
hold other bytes, have lengths that end anywhere in a code word, or fill more than one
piece of the filter's upload equal those of a server that filters and packs on
the host; several requests at once, results collected in another order."""
import numpy as np
import pytest

from saruman_amd import serve
from saruman_amd import workload as wl

pytestmark = pytest.mark.gpu


def reads_with_others(genome, n, lo, hi, seed):
    r = wl.synth_reads(seed, genome, n, lo, hi, 1, p_sub=0.01, p_ins=0.001, indel_max=2, k_rate=0.05)
    rng = np.random.default_rng(seed)
    seq = np.frombuffer(r.seq, np.uint8).copy()
    at = rng.integers(0, len(seq), max(1, n // 8))
    seq[at] = rng.choice(np.frombuffer(b"NRacgt.", np.uint8), len(at))
    return wl.Reads(seq.tobytes(), r.off, r.length, r.true_pos, r.strand, r.k)


@pytest.mark.parametrize("n,lo,hi", [(1, 36, 36), (17, 36, 53), (700, 36, 250), (33_001, 36, 90)])
def test_records_equal_the_hosts(n, lo, hi):
    print(f"[gpu] serve words {n}", flush=True)
    genome = wl.synth_genome(61, [150_000], 0.5)
    reads = reads_with_others(genome, n, lo, hi, 62)
    cuts = sorted({0, n // 3, n})
    spans = list(zip(cuts[:-1], cuts[1:]))
    got = []
    for on_device in (False, True):
        S = serve.Server(genome, wl.needed_qs(reads), n_slots=2, chunk_value=5_000,
                         gpu_filter=on_device, gpu_records=True)
        try:
            ids = [S.submit(reads, a, b) for a, b in spans]
            texts = {}
            for rid in reversed(ids):
                S.wait(rid)
                texts[rid] = S.result(rid)[0]
            got.append([texts[rid] for rid in ids])
        finally:
            S.close()
    assert got[0] == got[1]
    assert n < 700 or all(got[0])
