"""Uploads of the device filter in pieces against the host filter: read counts at a
piece's edges, reads stored in other orders or with gaps between them, guesses of the
totals that do not hold (the call starts over), other bytes and repeats, one strand, and
a read without an index in the last piece."""
import numpy as np
import pytest

from saruman_amd import workload as wl
from saruman_amd.batch import Context

pytestmark = pytest.mark.gpu

FIELDS = ("read", "pos", "flag", "w", "batch_end", "perfect_read", "perfect_pos")
PIECE = 32_768


def same(h, d, tag):
    for f in FIELDS:
        a, b = getattr(h, f), getattr(d, f)
        assert a.shape == b.shape and np.array_equal(a, b), (tag, f, a.shape, b.shape)


def placed(reads, order, gap):
    """The reads stored in another order, `gap` bytes between them."""
    seq = np.frombuffer(reads.seq, np.uint8)
    ln = reads.length.astype(np.int64)
    off = np.zeros(reads.n, np.int64)
    off[order] = np.concatenate([[0], np.cumsum(ln[order] + gap)[:-1]])
    buf = np.full(int((ln + gap).sum()), ord("G"), np.uint8)
    within = np.arange(int(ln.sum())) - np.repeat(np.cumsum(ln) - ln, ln)
    buf[np.repeat(off, ln) + within] = seq[np.repeat(reads.off.astype(np.int64), ln) + within]
    return wl.Reads(buf.tobytes(), off.astype(np.uint64), reads.length, reads.true_pos, reads.strand,
                    reads.k)


@pytest.mark.parametrize("name,n,lo,hi", [
    ("below", PIECE, 36, 60), ("edge", PIECE + 1, 36, 60), ("last_full", 2 * PIECE, 36, 36),
    ("ragged", 2 * PIECE + 4_097, 36, 120), ("backwards", PIECE + 999, 36, 90),
    ("shuffled", PIECE + 999, 36, 90), ("gaps", PIECE + 999, 36, 90),
    ("by_length", PIECE * 2 + 5, 36, 200), ("bad_sample", PIECE * 2 + 5, 36, 200),
    ("others", PIECE + 7, 36, 90), ("repeats", PIECE + 7, 40, 60)])
def test_pieces(name, n, lo, hi):
    print(f"[gpu] filter pieces {name}", flush=True)
    rng = np.random.default_rng(5)
    # (the lists of "repeats" outgrow the room they are first given)
    families = {"others": (3, 300, 600, 10, 0.5, 0.001), "repeats": (3, 300, 600, 60, 0.5, 0.001)}
    genome = wl.synth_genome(91, [60_000], 0.5, families.get(name))
    reads = wl.synth_reads(92, genome, n, lo, hi, 1, p_sub=0.01, p_ins=0.001, indel_max=2, k_rate=0.05)
    if name == "others":
        seq = np.frombuffer(reads.seq, np.uint8).copy()
        seq[rng.integers(0, len(seq), n // 20)] = ord("N")
        reads = wl.Reads(seq.tobytes(), reads.off, reads.length, reads.true_pos, reads.strand, reads.k)
    if name == "backwards":
        reads = placed(reads, np.arange(n)[::-1], 0)
    elif name == "shuffled":
        reads = placed(reads, rng.permutation(n), 3)
    elif name == "gaps":
        reads = placed(reads, np.arange(n), 17)
    elif name in ("by_length", "bad_sample"):
        order = np.argsort(reads.length, kind="stable")
        if name == "bad_sample":      # every sampled read one of the shortest
            step = n // 512
            at = np.arange(0, n, step)
            rest = np.setdiff1d(np.arange(n), at)
            full = np.empty(n, np.int64)
            full[at], full[rest] = order[:len(at)], order[len(at):]
            order = full
        off, ln = reads.off[order], reads.length[order]
        reads = wl.Reads(reads.seq, off, ln, reads.true_pos[order], reads.strand[order], reads.k[order])
    ctx = Context(0)
    idx = wl.Index(genome, wl.needed_qs(reads))
    df = wl.DeviceFilter(ctx, idx, genome)
    try:
        want = {dr: wl.run_filter(idx, genome, reads, dr, 20_000) for dr in (0, 4)}
        for dr, d in zip((0, 4), df.run_both(reads, 20_000)):
            same(want[dr], d, (name, dr))
        if name == "repeats":
            assert df.stats()["list_entries"] > 2 * df.stats()["lists"] + 2048
        if name == "ragged":
            for dr in (4, 0):
                same(want[dr], df.run(reads, dr, 20_000), (name, "one strand", dr))
    finally:
        df.close()
        idx.close()
        ctx.close()


def test_last_piece_without_an_index():
    print("[gpu] filter pieces error", flush=True)
    genome = wl.synth_genome(91, [60_000], 0.5)
    reads = wl.synth_reads(92, genome, PIECE + 500, 36, 36, 1, p_sub=0.01, p_ins=0.001, indel_max=2,
                           k_rate=0.05)
    ctx = Context(0)
    idx = wl.Index(genome, wl.needed_qs(reads))
    df = wl.DeviceFilter(ctx, idx, genome)
    try:
        k = reads.k.copy()
        k[-1] = 9
        bad = wl.Reads(reads.seq, reads.off, reads.length, reads.true_pos, reads.strand, k)
        with pytest.raises(Exception, match="lacks q"):
            df.run_both(bad, 20_000)
        for dr, d in zip((0, 4), df.run_both(reads, 20_000)):
            same(wl.run_filter(idx, genome, reads, dr, 20_000), d, dr)
    finally:
        df.close()
        idx.close()
        ctx.close()
