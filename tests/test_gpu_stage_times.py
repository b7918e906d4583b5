"""What a run reports of its stages: the plain kernels' own time where they run beside the
band's, and each band class's part of the one launch's grid."""
import ctypes as C

import numpy as np
import pytest

from saruman_amd import _lib, tune
from saruman_amd.batch import Context, Job, _layout, pack_codes
from saruman_amd.testing import random_batch

pytestmark = pytest.mark.gpu


def run(ctx, lay, streams):
    tune.apply(ctx, {"blocks_per_cu": [0] * 9, "class_streams": streams})
    job = Job(ctx)
    try:
        job.upload(0, 1, lay["cand"], pack_codes(lay["rcat"]), pack_codes(lay["wcat"]), lay["rcat"],
                   lay["wcat"], ops_total=lay["ops_total"])
        assert job.paths()[0] > 0 and job.paths()[2] > 0
        plain, band = [], []
        for _ in range(5):
            job.run("auto")
            b, p = job.kernel_ms()
            plain.append(p)
            band.append(b)
        info = []
        for nw in range(1, 9):
            blocks, ntiles, ms = C.c_int(), C.c_int(), C.c_float()
            _lib.check(job.lib.srm_job_band_info(job.h, nw, C.byref(blocks), C.byref(ntiles), C.byref(ms)),
                       "srm_job_band_info")
            if ntiles.value:
                info.append((blocks.value, ntiles.value, ms.value))
        return float(np.median(plain)), band, info
    finally:
        job.close()


def test_stage_times():
    print("[gpu] stage times", flush=True)
    # 16,000 banded candidates and eight raw ones, whose chain is shorter than the band's
    batch = random_batch(np.random.default_rng(51), 16_000, L=250, k=12)
    for t in range(8):
        r = bytearray(batch.reads[t])
        r[7] = ord("N")
        batch.reads[t] = bytes(r)
    lay = _layout(batch)
    ctx = Context(0)
    try:
        alone, _, info = run(ctx, lay, 1)
        assert all(b == (n + 3) // 4 for b, n, _ in info)
        beside, band, info = run(ctx, lay, 4)
        # the same kernels: their chain takes as long (a wait of the remainder would not)
        assert beside > 0.5 * alone, (alone, beside, band)
        assert all(b == n for b, n, _ in info)
        assert all(ms == info[0][2] for _, _, ms in info) and info[0][2] > 0
    finally:
        ctx.close()
