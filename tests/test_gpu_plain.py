"""The plain path's two kernels (a wave per candidate; a thread per candidate for
costs beyond its range) against the oracle at the sizes where the wave's layout
changes: columns per lane, strips of 256 columns, 16 steps per decision word, 64
rows per window load, empty and short windows."""
import numpy as np
import pytest

import saruman_amd as sa
from saruman_amd.batch import Batch
from saruman_amd.testing import ACGT, mutate

pytestmark = pytest.mark.gpu

LS = (1, 2, 63, 64, 65, 128, 129, 192, 193, 256, 257, 512, 513, 1000)


def sized_batch(rng, L, match, mismatch, raw):
    wins, reads, flags, ks = [], [], [], []
    for flag in range(9):
        for k in (0, 3, 40):
            for dw in (-L, -L + 1, -20, 0, k, 2 * k):
                w = L + dw
                if w < 0 or w > 900:
                    continue
                win = ACGT[rng.integers(0, 4, w)]
                read = mutate(rng, win[min(w, max(0, dw) // 2):], int(rng.integers(0, 6)))
                read = np.concatenate([read, ACGT[rng.integers(0, 4, L)]])[:L]
                if raw:
                    read = read.copy()
                    read[int(rng.integers(0, L))] = ord("N")
                    if w:
                        win = win.copy()
                        win[int(rng.integers(0, w))] = ord("N")
                wins.append(win.tobytes())
                reads.append(read.tobytes())
                flags.append(flag)
                ks.append(k)
    n = len(wins)
    return Batch(match, mismatch, 40, wins, reads, np.array(flags, np.uint8),
                 rng.integers(1, 1 << 24, n).astype(np.int64), [f"r{t}" for t in range(n)],
                 ks=np.array(ks, np.int64), first_row0=True)


@pytest.mark.parametrize("raw", [False, True])
@pytest.mark.parametrize("match,mismatch", [(0, 1), (0, 2), (-1, 1), (3, 0), (-15, 15), (15, -15),
                                            (0, 16), (-16, 3)])
def test_plain_sizes(orc, match, mismatch, raw):
    for L in LS:
        print(f"[gpu] plain L={L} costs {match},{mismatch} raw={raw}", flush=True)
        batch = sized_batch(np.random.default_rng(1000 * L + raw), L, match, mismatch, raw)
        got = sa.align_batch(batch, kernel="plain")
        want = orc.align_batch(batch)
        assert (got.scores == np.asarray(want.scores, np.int64)).all(), L
        bad = [t for t in range(batch.n) if got.records[t] != want.records[t]]
        assert not bad, (L, bad[0], got.records[bad[0]], want.records[bad[0]])
