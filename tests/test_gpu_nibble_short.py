"""Costs other than 0/1 on reads no longer than their error bound, and next to it: row 0
then lies in the band of every column.  The batch entry and the static one, with the
classes in one launch and one after another, against the oracle's records."""
import numpy as np
import pytest

import saruman_amd as sa
from saruman_amd import tune
from saruman_amd.batch import Context, Job, _layout, format_records, pack_codes
from test_gpu_band_launch import gapped_batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("match,mismatch", [(0, 2), (0, 3), (1, 3), (5, 2)])
@pytest.mark.parametrize("n,lengths", [(400, (1, 2)), (3000, tuple(range(1, 21)))])
def test_short_reads(orc, n, lengths, match, mismatch):
    print(f"[gpu] nibble short n={n} costs {match},{mismatch}", flush=True)
    batch = gapped_batch(np.random.default_rng(n), n, lengths, match, mismatch)
    want = orc.align_batch(batch)
    assert any(want.records)
    for kernel in ("banded", "plain"):
        got = sa.align_batch(batch, kernel=kernel)
        assert [t for t in range(n) if got.records[t] != want.records[t]] == [], kernel
    lay = _layout(batch)
    ctx = Context(0)
    try:
        for streams in (1, 4):
            tune.apply(ctx, {"blocks_per_cu": [0] * 9, "class_streams": streams})
            job = Job(ctx)
            job.upload(match, mismatch, lay["cand"], pack_codes(lay["rcat"]), pack_codes(lay["wcat"]),
                       ops_total=lay["ops_total"])
            job.run("banded")
            res, ops = job.download()
            job.close()
            assert format_records(batch, res, ops, lay) == want.records, streams
    finally:
        ctx.close()
