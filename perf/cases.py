"""The work a user has this library do, as timed cases over its public entry points.

Every case starts from reads drawn from a synthetic genome with the error model of
the benchmark's workloads (k = ceil(5% of the read length) throughout); the genome,
its q-gram index and the handles a program keeps between calls (context, device
filter, server, job) are made once per genome and length range, the reads from
the case's seed.  Kinds:

  filter    both strands of a read set through the device q-gram filter: reads in
            host memory in, candidates and perfect hits in host arrays out
  static    srm_align_static: descriptors on the host, codes, results and transcripts
            in device tensors (callers that cannot allocate)
  align     the resident step without records: graph replay of the band kernels,
            then every candidate's score and end cell to page-locked memory
  records   the resident step with the record stage, then the TSV text to page-locked
            memory
  fresh     one new batch through a kept job: upload, run, records; some of the reads
            hold an N, as sequencer output does (those candidates run on raw bytes)
  bulk      one new batch from page-locked memory through a kept job with the record
            stage, its text back to page-locked memory (one lane of bulk mapping)
  request   requests to the continuous-batching server, filter and records on the
            device: reads in, all records of every request out
"""
import ctypes as C
import math
from collections import OrderedDict

import numpy as np
import torch

import saruman_amd as sa
from saruman_amd import _lib, serve, tune
from saruman_amd import workload as wl
from saruman_amd.batch import Job
from saruman_amd.pipeline import PinnedBatch

CHUNK = 1_000_000          # the reference's -s


def _case(kind, reads, lmin, lmax, genome, **more):
    return {"kind": kind, "reads": reads, "lmin": lmin, "lmax": lmax, "genome": genome, **more}


def listed():
    return [
        # the smallest serving request's filter: latency, launches and host passes
        dict(name="filter 1k 36-250bp", **_case("filter", 1_000, 36, 250, 5_000_000)),
        # short reads of one length (the 36 bp workload, whole)
        dict(name="filter 100k 36bp", **_case("filter", 100_000, 36, 36, 1_000_000)),
        # the benchmark's default read set, whole
        dict(name="filter 2M 50-250bp", **_case("filter", 2_000_000, 50, 250, 4_000_000, repeats=True)),
        # a small call from a tight loop, short reads
        dict(name="static 500 36bp", **_case("static", 500, 36, 36, 1_000_000, match=0, mismatch=1)),
        # the largest call the entry point's descriptor limit admits, mixed lengths
        dict(name="static 60k 50-250bp", **_case("static", 60_000, 50, 250, 5_000_000, match=0, mismatch=1)),
        # other costs (the nibble band)
        dict(name="static 20k 100bp cost 2", **_case("static", 20_000, 100, 100, 5_000_000, match=0, mismatch=2)),
        # the benchmark's default step without its record stage: scores and end cells
        dict(name="align 2M 50-250bp", **_case("align", 2_000_000, 50, 250, 4_000_000, repeats=True)),
        # the 100 bp workload's step, names from a table as files give them
        dict(name="records 1M 100bp names", **_case("records", 1_000_000, 100, 100, 5_000_000, table=True)),
        # an ordinary batch of sequencer reads: 3% of the reads hold an N
        dict(name="fresh 50k 36-250bp with N", **_case("fresh", 50_000, 36, 250, 5_000_000, n_rate=0.03)),
        # bulk mapping: a 1,000,000-read batch of 150 bp, host to host, two contigs
        dict(name="bulk 1M 150bp", **_case("bulk", 1_000_000, 150, 150, 12_000_000, contigs=2)),
        # the smallest and a large burst of the serving workload
        dict(name="request 1k 36-250bp", **_case("request", 1_000, 36, 250, 5_000_000, requests=1)),
        dict(name="request 4x50k 36-250bp", **_case("request", 50_000, 36, 250, 5_000_000, requests=4)),
    ]


def draw(rng):
    def logu(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["filter", "static", "align", "records", "fresh", "bulk", "request"])
    if rng.random() < 0.5:
        lmin = lmax = rng.randint(36, 250)
    else:
        lmin = rng.randint(36, 120)
        lmax = rng.randint(lmin + 1, 250)
    genome = logu(1_000_000, 6_000_000)
    if kind == "filter":
        return _case(kind, logu(500, 1_500_000), lmin, lmax, genome, repeats=rng.random() < 0.5)
    if kind == "static":
        mm = rng.choice([1, 1, 2, 3])
        return _case(kind, logu(100, 55_000 if mm == 1 else 18_000), lmin, lmax, genome,
                     match=0, mismatch=mm)
    if kind == "align":
        return _case(kind, logu(1_000, 1_500_000), lmin, lmax, genome, repeats=rng.random() < 0.5)
    if kind == "records":
        return _case(kind, logu(1_000, 800_000), lmin, lmax, genome, table=rng.random() < 0.5)
    if kind == "fresh":
        return _case(kind, logu(1_000, 100_000), lmin, lmax, genome,
                     n_rate=rng.choice([0.0, 0.005, 0.03]))
    if kind == "bulk":
        return _case(kind, logu(20_000, 900_000), lmin, lmax, genome, contigs=rng.choice([1, 2]))
    requests = rng.choice([1, 1, 2, 4])
    return _case(kind, logu(1_000, 150_000 // requests), lmin, lmax, genome, requests=requests)


# ---------------------------------------------------------------------------
# what a program keeps: per genome and read lengths, the last few
# ---------------------------------------------------------------------------
class _Resident:
    """A genome, its index and the handles made from it on first use."""

    def __init__(self, case):
        n, parts = case["genome"], case.get("contigs", 1)
        lens = [n] if parts == 1 else [n - n // 3, n // 3]
        repeats = (20, 1000, 5000, 200, 0.02, 0.005) if case.get("repeats") else None
        self.genome = wl.synth_genome(0x5A2_0003, lens, 0.5, repeats)
        self.qs = serve.qs_for_lengths(case["lmin"], case["lmax"])
        self.index = wl.Index(self.genome, self.qs)
        self.ctx = sa.Context(0)
        tune.apply_cached(self.ctx)
        self.words = wl.genome_words(self.genome)
        self.ctx.set_genome(self.words)
        self.filter = wl.DeviceFilter(self.ctx, self.index, self.genome)
        self._server = self._job = None

    def server(self):
        if self._server is None:
            self._server = serve.Server(self.genome, self.qs, n_slots=4, chunk_value=200_000,
                                        gpu_filter=True, gpu_records=True)
        return self._server

    def kept_job(self):
        if self._job is None:
            self._job = Job(self.ctx)
        return self._job


_RESIDENT: "OrderedDict" = OrderedDict()


def _resident(case):
    key = tuple(case.get(f, 0) for f in ("genome", "contigs", "repeats", "lmin", "lmax"))
    if key not in _RESIDENT:
        while len(_RESIDENT) >= 4:
            _RESIDENT.popitem(last=False)
        _RESIDENT[key] = _Resident(case)
    _RESIDENT.move_to_end(key)
    return _RESIDENT[key]


def _reads(case, genome, n, seed):
    lo, hi = case["lmin"], case["lmax"]
    if hi <= 40:      # up to two errors a read, 80% substitutions
        return wl.synth_reads(seed, genome, n, lo, hi, 0, max_err=2, p_sub=0.8, p_ins=0.1,
                              k_rate=0.05)
    return wl.synth_reads(seed, genome, n, lo, hi, 1, p_sub=0.01, p_ins=0.001, indel_max=3,
                          p_random=0.05 if lo == hi else 0.0, k_rate=0.05)


def _with_n(reads, rate, seed):
    """The reads with one base of a share of them replaced by N, and which."""
    rng = np.random.default_rng(seed)
    seq = np.frombuffer(reads.seq, np.uint8).copy()
    hit = rng.random(reads.n) < rate
    at = reads.off[hit].astype(np.int64) + (rng.random(int(hit.sum())) *
                                            reads.length[hit]).astype(np.int64)
    seq[at] = ord("N")
    return wl.Reads(seq.tobytes(), reads.off, reads.length, reads.true_pos, reads.strand,
                    reads.k), hit


_CODE = np.zeros(256, np.uint8)
_CODE[[ord(c) for c in "ACGT"]] = range(4)
_COMP = np.arange(256, dtype=np.uint8)
_COMP[[ord(c) for c in "ACGT"]] = [ord(c) for c in "TGCA"]


def _both_strands(reads):
    """Bytes and packed codes of every read, then of every reverse complement."""
    dev = torch.device("cuda", 0)
    fwd = torch.from_numpy(np.frombuffer(reads.seq, np.uint8).copy()).to(dev)
    ln = torch.from_numpy(reads.length.astype(np.int64)).to(dev)
    off = torch.from_numpy(reads.off.astype(np.int64)).to(dev)
    src = torch.repeat_interleave(2 * off + ln - 1, ln) - torch.arange(fwd.numel(), device=dev)
    both = torch.cat([fwd, torch.from_numpy(_COMP).to(dev)[fwd[src].long()]])
    del src
    pad = _lib.SRM_CODE_PAD
    total = (2 * pad + both.numel() + 15) // 16 * 16 + 16
    codes = torch.zeros(total, dtype=torch.int32, device=dev)
    table = torch.from_numpy(_CODE).to(dev).int()
    for a in range(0, both.numel(), 1 << 26):
        part = both[a:a + (1 << 26)]
        codes[pad + a:pad + a + part.numel()] = table[part.int()]
    shifts = torch.arange(0, 32, 2, dtype=torch.int32, device=dev)
    words = (codes.view(-1, 16) << shifts).sum(1, dtype=torch.int32)
    return both, words


def _batch(R, reads):
    """The candidates of both strands as the filter finds them, and the read bytes."""
    strands = R.filter.run_both(reads, CHUNK)
    both, words = _both_strands(reads)
    return wl.device_batch(reads, strands, words.cpu().numpy().view(np.uint32)), both


class _State:
    def __init__(self, case, R, **kw):
        self.case, self.R = case, R
        self.job = None
        self.__dict__.update(kw)

    def __del__(self):
        if self.job is not None:
            self.job.close()


def _page_locked(nbytes):
    return torch.zeros(int(nbytes), dtype=torch.uint8).pin_memory().numpy()


# outputs go to buffers whose sizes follow from the case: what its read count yields
# with a quarter to spare, the rest stays zero
def _room(case):
    return case["reads"] * (5 if case.get("repeats") else 4) // 3 + 256


def _text_room(case):
    return int(case["reads"] * 1.3 * (case["lmin"] + case["lmax"] + 60)) + 65536


def prepare(case, seed):
    R = _resident(case)
    kind = case["kind"]
    n = case["reads"] * case.get("requests", 1)
    reads = _reads(case, R.genome, n, 0x5A2_0100 + 7 * seed)
    if kind == "filter":
        pinned, buf = wl.pinned_reads(reads)
        m = _room(case)
        out = [[np.zeros(m, t) for t in (np.int32, np.int64, np.uint8, np.uint16, np.uint64,
                                         np.int32, np.int64)] for _ in range(2)]
        return _State(case, R, reads=pinned, buf=buf, out=out)
    if kind == "request":
        return _State(case, R, reads=reads, server=R.server(),
                      out=[np.zeros(_text_room(case), np.uint8) for _ in range(case["requests"])])
    if kind == "fresh":
        reads, has_n = _with_n(reads, case["n_rate"], seed)
        db, both = _batch(R, reads)
        raw = has_n[db.read_id]
        db.cand["bits"][raw] = _lib.SRM_CAND_BYTES
        db.cand["win_off"][raw] = db.pos[raw]
        return _State(case, R, db=db, read_bytes=both.cpu().numpy().tobytes() if raw.any() else None,
                      ids=db.read_id.astype(np.int32), kept=R.kept_job(),
                      out=_page_locked(_text_room(case)))
    db = _batch(R, reads)[0]
    if kind == "bulk":
        return _State(case, R, batch=PinnedBatch.of(db), kept=R.kept_job(),
                      out=_page_locked(_text_room(case)))
    if kind == "static":
        room = min(_room(case), 65536)
        m = min(db.n, room)
        k = math.ceil(0.05 * case["lmax"])
        words = room * ((case["lmax"] + 3 * k + 15) // 16)
        gw = torch.from_numpy(R.words.view(np.int32)).cuda()
        rw = torch.from_numpy(db.read_words.view(np.int32)).cuda()
        cand = np.ascontiguousarray(db.cand[:m])
        cand["win_off"] -= _lib.SRM_CODE_PAD      # this entry point counts from the first code
        return _State(case, R, n=m, cand=cand, gw=gw, rw=rw, words=words,
                      res=torch.zeros((room, 4), dtype=torch.int16, device="cuda"),
                      ops=torch.zeros(words, dtype=torch.int32, device="cuda"))
    job = Job(R.ctx)
    job.upload(0, 1, db.cand, db.read_words, None, ops_total=db.ops_total)
    if kind == "align":
        out = _page_locked(8 * _room(case))
    else:
        names, stride = None, 60
        if case["table"]:
            tab = np.zeros((n, stride), np.uint8)
            digits = np.char.zfill(np.arange(n).astype("U9"), 9)
            tab[:, :5] = np.frombuffer(b"read/", np.uint8)
            tab[:, 5:14] = digits.view(np.uint32).reshape(n, 9).astype(np.uint8)
            names = tab.tobytes()
        job.set_records(db.pos, read_id=db.read_id.astype(np.int32), names=names,
                        name_stride=stride, prefix="r")
        out = _page_locked(_text_room(case))
    job.use_graph(True)
    return _State(case, R, job=job, out=out, n=db.n)


def _whole(text, got):
    if got > text.size:
        raise RuntimeError(f"{got} bytes of records, room for {text.size}")
    return text


def run(state):
    lib, kind = state.R.ctx.lib, state.case["kind"]
    if kind == "filter":
        f, r, both = state.R.filter, state.reads, (C.c_void_p(), C.c_void_p())
        genome = state.R.genome
        _lib.check(lib.srm_dfilter_run2(
            f.h, _lib.ptr(genome.blocked), r.seq.ctypes.data, r.off.ctypes.data,
            r.length.ctypes.data, r.k.ctypes.data, r.n, CHUNK, C.byref(both[0]),
            C.byref(both[1])), "srm_dfilter_run2")
        sizes = []
        for h, out in zip(both, state.out):
            n = (C.c_uint64 * 3)()
            lib.srm_filter_sizes(h, C.byref(n, 0), C.byref(n, 8), C.byref(n, 16))
            if max(n) > out[0].size:
                raise RuntimeError(f"more filter output than room for it: {list(n)}")
            lib.srm_filter_copy(h, *(a.ctypes.data for a in out))
            lib.srm_filter_destroy(h)
            sizes += list(n)
        return [state.out, np.array(sizes, np.int64)]
    if kind == "static":
        _lib.check(lib.srm_align_static(
            0, None, state.case["match"], state.case["mismatch"], state.cand.ctypes.data, state.n,
            state.rw.data_ptr(), state.rw.numel(), state.gw.data_ptr(), state.gw.numel(),
            state.res.data_ptr(), state.ops.data_ptr(), state.words), "srm_align_static")
        return [state.res, state.ops]
    if kind == "align":
        state.job.run("banded")
        _lib.check(lib.srm_job_download(state.job.h, state.out.ctypes.data, None, 0), "srm_job_download")
        return state.out.view(np.int16).reshape(-1, 4)
    if kind == "records":
        state.job.run("banded")
        got, hits = state.job.records_text(out=state.out, copy=False)
        return [_whole(state.out, got), got, hits]
    if kind == "fresh":
        db, job = state.db, state.kept
        raw = state.read_bytes
        job.upload(0, 1, db.cand, db.read_words, None, raw,
                   state.R.genome.seq if raw is not None else None, ops_total=db.ops_total)
        job.run("auto")
        got, hits = job.records(db.pos, read_id=state.ids, prefix="r", out=state.out,
                                copy=False)
        return [_whole(state.out, got), got, hits]
    if kind == "bulk":
        b, job = state.batch, state.kept
        job.upload(0, 1, b.cand, b.read_words, None, ops_total=b.ops_total)
        job.set_records(b.pos, read_id=b.read_id, prefix="r")
        job.run("banded")
        got, hits = job.records_text(out=state.out, copy=False)
        return [_whole(state.out, got), got, hits]
    S, m = state.server, state.case["reads"]
    ids = [S.submit(state.reads, i * m, (i + 1) * m) for i in range(state.case["requests"])]
    out = []
    for text, rid in zip(state.out, ids):
        S.wait(rid)
        st = serve.RequestStats()
        got = int(lib.srm_server_result(S.h, rid, text.ctypes.data, text.size, C.byref(st), 1))
        if got < 0 or st.status != 0:
            raise RuntimeError(f"request failed: {st.message.decode(errors='replace')}")
        out.append([_whole(text, got), got, st.n_candidates, st.n_hits, st.n_perfect, st.n_mapped])
    return out


def exact(case, seed):
    """Every output is a whole number or a byte of text."""
    return None


def work(case):
    """Host or HBM bytes of one pass: every input once, every output once; about
    0.89 candidates, 0.83 aligned hits and 0.23 perfect hits per read.  No floating
    operations."""
    kind = case["kind"]
    reads = case["reads"] * case.get("requests", 1)
    L = (case["lmin"] + case["lmax"]) / 2
    w = 1.1 * L
    codes = L / 4 + w / 4 + 20          # a candidate's read, window and descriptor
    ops = w / 4                         # its transcript
    text = 2 * L + 40                   # its record
    per = {"filter": L + 11 + 0.89 * 15 + 0.23 * 12,
           "static": 0.89 * (codes + ops + 8),
           "align": 0.89 * (codes + ops + 8),
           "records": 0.89 * (codes + ops + 20) + 0.83 * text,
           "fresh": 0.89 * (codes + 20) + 0.83 * text,
           "bulk": 0.89 * (codes + 20) + 0.83 * text,
           "request": L + 11 + 1.06 * text}[kind]
    return {"bytes": float(reads * per), "flops": 0.0}
