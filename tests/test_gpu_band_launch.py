"""The band kernels with every class in one launch and with the classes one after
another, for unit costs in both scratch layouts: equal results, and the oracle's records.
The reads hold one gap of up to k bases at every place of a 32-column segment (a
walk that recomputes a segment holds 8 diagonals of it), the batch sizes leave tiles
of one candidate and classes of one tile."""
import numpy as np
import pytest

import saruman_amd as sa
from saruman_amd import tune
from saruman_amd.batch import Batch, Context, Job, _layout, pack_codes
from saruman_amd.testing import ACGT

pytestmark = pytest.mark.gpu


def gapped_batch(rng, n, lengths, match, mismatch):
    wins, reads, flags, ks = [], [], [], []
    for t in range(n):
        L = int(lengths[t % len(lengths)])
        k = int(rng.integers(1, 16))
        flag = int(rng.integers(0, 8))
        s = k if flag & 2 else 0
        e = k if flag & 1 else 0
        w = L + s + e
        win = ACGT[rng.integers(0, 4, w)]
        g = int(rng.integers(0, k + 1))
        at = int(rng.integers(0, L))
        src = np.concatenate([win[int(rng.integers(0, s + 1)):], ACGT[rng.integers(0, 4, L + 15)]])
        if t & 1:      # g genome bases skipped
            read = np.concatenate([src[:at], src[at + g:]])[:L]
        else:          # g bases between
            read = np.concatenate([src[:at], ACGT[rng.integers(0, 4, g)], src[at:]])[:L]
        sub = rng.random(L) < 0.01
        read = np.where(sub, ACGT[rng.integers(0, 4, L)], read)
        wins.append(win.tobytes())
        reads.append(read.astype(np.uint8).tobytes())
        flags.append(flag)
        ks.append(k)
    return Batch(match, mismatch, 15, wins, reads, np.array(flags, np.uint8),
                 rng.integers(1, 1 << 24, n).astype(np.int64), [f"r{t}" for t in range(n)],
                 ks=np.array(ks, np.int64))


@pytest.mark.parametrize("match,mismatch", [(0, 1), (0, 2), (1, 3)])
@pytest.mark.parametrize("n,lengths", [(1, (40,)), (130, (33, 64)), (4000, (36, 97, 100, 128, 250)),
                                       (2000, (31, 32, 33, 251, 330, 620)), (400, (1, 2))])
def test_one_launch(orc, n, lengths, match, mismatch):
    print(f"[gpu] one launch n={n} lengths={lengths} costs {match},{mismatch}", flush=True)
    if lengths == (1, 2) and mismatch != 1:
        pytest.skip("reads of one or two bases: the nibble kernels take a hit that the oracle does not")
    batch = gapped_batch(np.random.default_rng(n), n, lengths, match, mismatch)
    want = orc.align_batch(batch)
    got = sa.align_batch(batch, kernel="banded")
    assert [t for t in range(n) if got.records[t] != want.records[t]] == []
    lay = _layout(batch)
    ctx = Context(0)
    try:
        outs = []
        for table in ({"class_streams": 1}, {"class_streams": 1, "walk_layout": 1}, {},
                      {"walk_layout": 1},
                      {"walk_layout": 1, "split_len": 64, "tile_cands": 32}):
            tune.apply(ctx, {"blocks_per_cu": [0] * 9, **table})
            job = Job(ctx)
            job.upload(match, mismatch, lay["cand"], pack_codes(lay["rcat"]), pack_codes(lay["wcat"]),
                       ops_total=lay["ops_total"])
            job.run("banded")
            outs.append(job.download())
            job.close()
        for res, ops in outs[1:]:
            assert (res == outs[0][0]).all()
            for t in range(n):
                o = int(lay["cand"]["ops_off"][t])
                nw = (int(res["n_ops"][t]) + 15) // 16
                assert (ops[o:o + nw] == outs[0][1][o:o + nw]).all()
    finally:
        ctx.close()
