"""Both strands of the device filter in one call, with its batch pass on the device,
against the host filter: the smallest calls (inputs and output in one copy each),
output larger than the first copy, reads that outgrow the LDS slots, flushes beyond
the device's list, separators, and entries skipped at a genome's end, whose window
lengths the next reads' entries inherit."""
import numpy as np
import pytest

from saruman_amd import workload as wl
from saruman_amd.batch import Context

pytestmark = pytest.mark.gpu

FIELDS = ("read", "pos", "flag", "w", "batch_end", "perfect_read", "perfect_pos")


def same(h, d, tag):
    for f in FIELDS:
        a, b = getattr(h, f), getattr(d, f)
        assert a.shape == b.shape and np.array_equal(a, b), (tag, f, a.shape, b.shape)


def at_ends(genome, n, L, seed):
    """Reads of the genome's last L + 12 bases, with gaps and substitutions."""
    rng = np.random.default_rng(seed)
    g = np.frombuffer(genome.seq, np.uint8)
    out = []
    for _ in range(n):
        s = len(g) - L - int(rng.integers(0, 13))
        r = g[s:s + L].copy()
        if rng.random() < 0.7:      # a base left out: the read ends with one more
            at = int(rng.integers(5, L - 5))
            r = np.concatenate([r[:at], r[at + 1:], g[s + L:s + L + 1], g[:1]])[:L]
        at = int(rng.integers(0, L))
        r[at] = ord("A") if r[at] != ord("A") else ord("C")
        out.append(r)
    return wl.Reads(np.concatenate(out).tobytes(), np.arange(n, dtype=np.uint64) * L,
                    np.full(n, L, np.uint16), np.zeros(n, np.int64), np.zeros(n, np.uint8),
                    np.full(n, 5, np.uint8))


CASES = {
    # genome lengths, repeats, reads (count, lengths), chunk values
    "one_read": ([20_000], None, (1, 36, 36), (1, 1000)),
    "few": ([20_000], None, (300, 36, 90), (3, 1000)),
    "stage_edges": ([50_000], None, (9_000, 50, 150), (40, 100_000)),
    "overflow": ([40_000], (3, 300, 600, 40, 0.5, 0.001), (6_000, 40, 40), (60, 100_000)),
    "separators": ([60_000, 30_000, 9_000], None, (12_000, 50, 250), (5, 500, 200_000)),
    "separators_on_host": ([400_000, 300_000], None, (2_000, 50, 250), (500,)),
    "large": ([300_000], None, (70_000, 36, 250), (20_000, 1_000_000)),
}


@pytest.mark.parametrize("name", list(CASES) + ["ends"])
def test_both_strands(name):
    print(f"[gpu] filter batch {name}", flush=True)
    if name == "ends":
        genome = wl.synth_genome(77, [5_000], 0.5)
        reads, chunks = at_ends(genome, 900, 60, 5), (4, 100, 100_000)
    else:
        lens, rep, (n, lo, hi), chunks = CASES[name]
        genome = wl.synth_genome(71, lens, 0.5, rep)
        kw = dict(max_err=3, k=3) if lo == hi else dict(indel_max=2, k_rate=0.05)
        reads = wl.synth_reads(72, genome, n, lo, hi, 0 if lo == hi else 1,
                               p_sub=0.8 if lo == hi else 0.01, p_ins=0.1 if lo == hi else 0.001, **kw)
    ctx = Context(0)
    idx = wl.Index(genome, wl.needed_qs(reads))
    df = wl.DeviceFilter(ctx, idx, genome)
    try:
        for chunk in chunks:
            for dr, d in zip((0, 4), df.run_both(reads, chunk)):
                same(wl.run_filter(idx, genome, reads, dr, chunk), d, (name, chunk, dr))
    finally:
        df.close()
        idx.close()
        ctx.close()


def test_results_outlive_the_filter():
    """Six calls' results held at once (more than the page-locked blocks there are) and
    read after the filter is gone."""
    import ctypes as C

    from saruman_amd import _lib
    from saruman_amd._lib import ptr
    print("[gpu] filter results held", flush=True)
    genome = wl.synth_genome(81, [200_000], 0.5)
    reads = wl.synth_reads(82, genome, 30_000, 50, 150, 1, p_sub=0.01, p_ins=0.001, indel_max=2,
                           k_rate=0.05)
    ctx = Context(0)
    idx = wl.Index(genome, wl.needed_qs(reads))
    df = wl.DeviceFilter(ctx, idx, genome)
    want = [wl.run_filter(idx, genome, reads, dr, 10_000) for dr in (0, 4)]
    rs, off, ln, kk = wl._reads_args(reads)
    held = []
    for _ in range(6):
        h = (C.c_void_p(), C.c_void_p())
        _lib.check(df.lib.srm_dfilter_run2(df.h, None, ptr(rs), ptr(off), ptr(ln), ptr(kk), reads.n,
                                           10_000, C.byref(h[0]), C.byref(h[1])), "srm_dfilter_run2")
        held.append(h)
    lib = df.lib
    df.close()
    idx.close()
    ctx.close()
    for h in held:
        for dr, x in zip((0, 1), h):
            same(want[dr], wl._collect(lib, x, 4 * dr, 0.0), dr)
