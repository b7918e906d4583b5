"""The device filter's upload in three pieces and more (65,536 reads a piece here), which
is where a piece's staging and events are used again, against the host filter: read
counts at a piece's edges and over one; calls that stop in the third piece or later, for
a missing index, a guess of the totals that does not hold or too many parameter sets; and
a serving request whose codes the filter leaves after such an upload."""
import numpy as np
import pytest

from saruman_amd import serve, workload as wl
from saruman_amd.batch import Context
from test_gpu_filter_batch import same
from test_gpu_serve_words import reads_with_others

pytestmark = pytest.mark.gpu

PIECE = 65_536


def synth(genome, n, lo, hi, seed=92):
    return wl.synth_reads(seed, genome, n, lo, hi, 1, p_sub=0.01, p_ins=0.001, indel_max=2, k_rate=0.05)


def joined(*parts):
    """Read sets one after another."""
    base = np.cumsum([0] + [len(p.seq) for p in parts])
    cat = lambda f: np.concatenate([getattr(p, f) for p in parts])
    return wl.Reads(b"".join(p.seq for p in parts),
                    np.concatenate([p.off + np.uint64(b) for p, b in zip(parts, base)]), cat("length"),
                    cat("true_pos"), cat("strand"), cat("k"))


def check(df, idx, genome, reads, chunk, tag):
    for dr, d in zip((0, 4), df.run_both(reads, chunk)):
        same(wl.run_filter(idx, genome, reads, dr, chunk), d, (tag, dr))


@pytest.mark.parametrize("n,lo,hi", [(3 * PIECE, 36, 36), (4 * PIECE + 1, 36, 60), (3 * PIECE - 1, 36, 200),
                                     (5 * PIECE + 777, 36, 90)])
def test_many_pieces(n, lo, hi):
    print(f"[gpu] filter many pieces {n}", flush=True)
    genome = wl.synth_genome(91, [200_000], 0.5, (3, 300, 600, 10, 0.5, 0.001))
    reads = synth(genome, n, lo, hi)
    if hi == 90:
        rng = np.random.default_rng(5)
        seq = np.frombuffer(reads.seq, np.uint8).copy()
        seq[rng.integers(0, len(seq), n // 20)] = ord("N")
        reads = wl.Reads(seq.tobytes(), reads.off, reads.length, reads.true_pos, reads.strand, reads.k)
    ctx = Context(0)
    idx = wl.Index(genome, wl.needed_qs(reads))
    df = wl.DeviceFilter(ctx, idx, genome)
    try:
        for chunk in (100_000, 30_000):
            check(df, idx, genome, reads, chunk, n)
        same(wl.run_filter(idx, genome, reads, 4, 100_000), df.run(reads, 4, 100_000), (n, "one strand"))
    finally:
        df.close()
        idx.close()
        ctx.close()


@pytest.mark.parametrize("at", [2 * PIECE + 1, 2 * PIECE + 30_000, 4 * PIECE + 3])
def test_missing_index_in_a_late_piece(at):
    print(f"[gpu] filter many pieces: missing index at {at}", flush=True)
    n = 4 * PIECE + 5
    genome = wl.synth_genome(91, [60_000], 0.5)
    reads = synth(genome, n, 36, 36)
    idx = wl.Index(genome, wl.needed_qs(reads))
    ctx = Context(0)
    df = wl.DeviceFilter(ctx, idx, genome)
    try:
        k = reads.k.copy()
        k[at:] = 9
        k[np.arange(0, n, n // 512)] = reads.k[0]     # (from which the totals are guessed)
        bad = wl.Reads(reads.seq, reads.off, reads.length, reads.true_pos, reads.strand, k)
        for _ in range(2):
            with pytest.raises(Exception, match="lacks q"):
                df.run_both(bad, 100_000)
        check(df, idx, genome, reads, 100_000, at)
    finally:
        df.close()
        idx.close()
        ctx.close()


@pytest.mark.parametrize("name", ["lists", "sets"])
def test_starts_over_in_a_late_piece(name):
    print(f"[gpu] filter many pieces: starts over, {name}", flush=True)
    genome = wl.synth_genome(91, [60_000], 0.5)
    if name == "lists":
        # the reads that are not sampled get longer from the third piece on
        n, short = 3 * PIECE + 60_000, synth(genome, 3 * PIECE + 60_000, 36, 36)
        long = synth(genome, n, 200, 200, 93)
        use = np.arange(n) >= 2 * PIECE + 500
        use[np.arange(0, n, n // 512)] = False
        use[-1] = True
        both = joined(short, long)
        at = np.where(use, n + np.arange(n), np.arange(n))
        seq = b"".join(both.seq[int(both.off[t]):int(both.off[t]) + int(both.length[t])] for t in at)
        ln = both.length[at]
        off = (np.cumsum(ln.astype(np.uint64)) - ln).astype(np.uint64)
        reads = wl.Reads(seq, off, ln, both.true_pos[at], both.strand[at], both.k[at])
    else:
        # more than 16,384 lengths with their error bounds, nearly all in the third piece
        reads = joined(synth(genome, 2 * PIECE + 100, 36, 40), synth(genome, 40_000, 300, 1_000, 93))
        rng = np.random.default_rng(6)
        L = reads.length[2 * PIECE + 100:].astype(np.int64)
        reads.k[2 * PIECE + 100:] = rng.integers(L // 20, L // 8)
        assert len(set(zip(reads.length.tolist(), reads.k.tolist()))) > 16_384
    idx = wl.Index(genome, wl.needed_qs(reads))
    ctx = Context(0)
    df = wl.DeviceFilter(ctx, idx, genome)
    try:
        check(df, idx, genome, reads, 100_000, name)
        check(df, idx, genome, synth(genome, 3 * PIECE, 36, 36), 100_000, "the next call")
    finally:
        df.close()
        idx.close()
        ctx.close()


def test_one_large_request():
    print("[gpu] filter many pieces: request", flush=True)
    genome = wl.synth_genome(61, [150_000], 0.5)
    n = 2 * PIECE + 9_001
    reads = reads_with_others(genome, n, 36, 90, 62)
    got = []
    for on_device in (False, True):
        S = serve.Server(genome, wl.needed_qs(reads), n_slots=2, chunk_value=5_000, gpu_filter=on_device,
                         gpu_records=True)
        try:
            rid = S.submit(reads, 0, n)
            S.wait(rid)
            got.append(S.result(rid)[0])
        finally:
            S.close()
    assert got[0] == got[1] and got[0]
