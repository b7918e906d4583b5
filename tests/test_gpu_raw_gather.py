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
