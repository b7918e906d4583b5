"""The upload's plan on the device (batches from 16,384 candidates, 4,096 for
srm_align_static) against the host's plan of the same candidates in smaller batches:
equal results and transcripts for every launch shape, with raw-byte candidates, ones
only the plain kernel takes and reads beyond the device plan's lengths among them, and
the same refusals."""
import numpy as np
import pytest

from saruman_amd import _lib, tune
from saruman_amd.batch import Context, Job, _layout, pack_codes
from saruman_amd.testing import random_batch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def laid_out(seed, n, hi=250, base=1500):
    """n candidates over the arrays of `base` random ones."""
    rng = np.random.default_rng(seed)
    batch = random_batch(rng, base, L=(20, hi), k=3, flags=(0, 1, 2, 3, 5, 6, 7),
                         per_cand_k=lambda L: min(14, 1 + L // 25))
    lay = _layout(batch)
    cand = lay["cand"][rng.integers(0, base, n)].copy()
    words = (cand["w"].astype(np.int64) + cand["k"] + 15) // 16
    cand["ops_off"] = np.concatenate([[0], np.cumsum(words)[:-1]])
    return cand, lay, int(words.sum())


def run(ctx, cand, lay, ops_total, kernel="banded", costs=(0, 1)):
    job = Job(ctx)
    try:
        job.upload(*costs, cand, pack_codes(lay["rcat"]), pack_codes(lay["wcat"]), lay["rcat"],
                   lay["wcat"], ops_total=ops_total)
        job.run(kernel)
        return job.download()
    finally:
        job.close()


def same(cand, got, parts):
    res, ops = got
    at = 0
    for pres, pops, pcand in parts:
        for f in ("score", "n_ops", "end_row", "end_col"):
            assert (res[at:at + len(pres)][f] == pres[f]).all(), f
        for t in range(0, len(pres), 7):
            nw = (int(pres["n_ops"][t]) + 15) // 16
            o, p = int(cand["ops_off"][at + t]), int(pcand["ops_off"][t])
            assert (ops[o:o + nw] == pops[p:p + nw]).all()
        at += len(pres)


SHAPES = [{}, {"tile_cands": 32, "walk_layout": 1}, {"split_len": 100, "merge_below": 3},
          {"class_streams": 1}]


@pytest.mark.parametrize("n,hi,raw", [(16_384, 250, False), (16_385, 250, True), (40_001, 511, True),
                                      (20_000, 512, False)])
def test_job_plan(ctx, n, hi, raw):
    print(f"[gpu] device plan n={n} hi={hi} raw={raw}", flush=True)
    cand, lay, total = laid_out(n, n, hi)
    if raw:      # the same bytes by another route
        hit = np.random.default_rng(1).random(n) < 0.02
        cand["bits"][hit] |= _lib.SRM_CAND_BYTES
    k40 = np.random.default_rng(2).random(n) < 0.01      # beyond the band's error bound
    cand["k"][k40] = 16
    words = (cand["w"].astype(np.int64) + cand["k"] + 15) // 16
    cand["ops_off"] = np.concatenate([[0], np.cumsum(words)[:-1]])
    parts = []
    for a in range(0, n, 12_000):
        part = cand[a:a + 12_000].copy()
        part["ops_off"] -= part["ops_off"][0]
        parts.append((*run(ctx, part, lay, int(words[a:a + 12_000].sum())), part))
    for shape in SHAPES:
        tune.apply(ctx, {"blocks_per_cu": [0] * 9, **shape})
        same(cand, run(ctx, cand, lay, int(words.sum())), parts)
    tune.apply(ctx, None)
    plain = run(ctx, cand, lay, int(words.sum()), "plain")[0]["score"].astype(np.int64)
    k1 = cand["k"].astype(np.int64) + 1
    got = run(ctx, cand, lay, int(words.sum()))[0]["score"].astype(np.int64)
    assert (np.minimum(plain, k1) == np.minimum(got, k1)).all()


def test_other_costs_beyond_one_launch(ctx):
    """More tiles than run at once: a launch per class, on streams and one after another."""
    print("[gpu] device plan, other costs", flush=True)
    n = 210_000
    cand, lay, total = laid_out(9, n, 60)
    want = run(ctx, cand, lay, total, costs=(0, 2))
    tune.apply(ctx, {"blocks_per_cu": [0] * 9, "class_streams": 1})
    res, ops = run(ctx, cand, lay, total, costs=(0, 2))
    tune.apply(ctx, None)
    assert (res == want[0]).all()
    parts = []
    for a in (0, 105_000, 205_000):
        part = cand[a:a + 5_000].copy()
        off = int(part["ops_off"][0])
        part["ops_off"] -= off
        words = int((part["ops_off"].astype(np.int64) + (part["w"].astype(np.int64) + part["k"] + 15) // 16).max())
        pres, pops = run(ctx, part, lay, words, costs=(0, 2))
        same(part, (res[a:a + 5_000], ops[off:off + words]), [(pres, pops, part)])


def test_refusals_name_the_first(ctx):
    cand, lay, total = laid_out(5, 20_000)
    for field, value in (("L", 0), ("read_off", 0xFFFFFFF0), ("win_off", 0xFFFFFFF0)):
        messages = []
        for n in (20_000, 9_000):
            bad = cand[:n].copy()
            for t in (8_500, 4_321, 7_000):
                bad[field][t] = value
            with pytest.raises(Exception) as e:
                run(ctx, bad, lay, total)
            messages.append(str(e.value))
        assert "candidate 4321" in messages[0] and messages[0] == messages[1]


@pytest.mark.parametrize("n,hi", [(4_096, 250), (20_000, 250), (9_000, 520)])
def test_static_plan(request, n, hi):
    from test_zz_no_alloc import Hip
    print(f"[gpu] static plan n={n} hi={hi}", flush=True)
    lib = _lib.load()
    cand, lay, total = laid_out(n + 1, n, hi)
    rw, ww = pack_codes(lay["rcat"]), pack_codes(lay["wcat"])
    hip = Hip()
    request.addfinalizer(hip.free)
    d_rw, d_ww = hip.put(rw), hip.put(ww)

    def call(c, words):
        d_res, d_ops = hip.zeros(len(c) * 8), hip.zeros(words * 4)
        rc = lib.srm_align_static(0, None, 0, 1, c.ctypes.data, len(c), d_rw, rw.size, d_ww, ww.size,
                                  d_res, d_ops, words)
        return (rc, hip.get(d_res, np.zeros(len(c), _lib.RES_DTYPE)),
                hip.get(d_ops, np.zeros(max(words, 1), np.uint32)))

    rc, res, ops = call(cand, total)
    assert rc == 0, lib.srm_last_error()
    parts = []
    for a in range(0, n, 4_000):
        c = cand[a:a + 4_000].copy()
        c["ops_off"] -= c["ops_off"][0]
        rc, r, o = call(c, int(((c["w"].astype(np.int64) + c["k"] + 15) // 16).sum()))
        assert rc == 0, lib.srm_last_error()
        parts.append((r, o, c))
    same(cand, (res, ops), parts)
    cand["w"][n - 5] = 0          # shorter than the band takes
    cand["k"][100] = 40
    assert call(cand, total)[0] < 0
    assert b"candidate 100 " in lib.srm_last_error()
