// filter_batch.h -- the batch pass (filter_internal.h: batch_pass) for the device
// filter, as host/device code: what each read yields by itself, counted and written
// by the kernels of filter_gpu.hip, and the few places where one read's outcome
// depends on an earlier one's, settled on the host.
//
// An entry with pos > 0 becomes a candidate when its read's batch is flushed, with
// w = L + s + e, unless its window leaves the genome or meets a separator: then it
// is skipped, keeps its s and e for the next entry in the walk, and its read is
// walked again at every later flush (Q10).  A larger w only skips more, so
//   - an entry that its own flag's w skips is never a candidate;
//   - what enters a read is its predecessor's last entry's s and e if that was
//     skipped, in whichever flush it is walked: a skipped entry's predecessor by
//     which it was skipped is walked again beside it, with the same outcome.  So an
//     entry skipped once stays skipped, and one walk over the reads in order gives
//     every flush's candidates;
//   - only the reads holding an entry that some w could skip (at most L + 2 kmax:
//     "unsafe"; those near a genome end or separator) and the read after one that
//     ends on such an entry need that walk.  Every other entry is a candidate at
//     its place in read order.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <vector>

#include "filter_pair.h"

namespace srm_batch {

// one read's share of the output; summed over the reads before it, its place there
struct Counts {
    uint32_t cand = 0;     // entries that are candidates by their own flag
    uint32_t perf = 0;     // perfect hits
    uint32_t queued = 0;   // entries with pos > 0
    uint32_t with = 0;     // 1: the read has entries
};

struct CountsSum {
    SRM_HD Counts operator()(const Counts &x, const Counts &y) const
    {
        Counts r;
        r.cand = x.cand + y.cand;
        r.perf = x.perf + y.perf;
        r.queued = x.queued + y.queued;
        r.with = x.with + y.with;
        return r;
    }
};

// what the flag adds to the window length (hash.c:938-979)
SRM_HD inline bool has_start(int flag) { return flag == 2 || flag == 3 || flag == 6 || flag == 7; }
SRM_HD inline bool has_end(int flag) { return flag == 1 || flag == 3 || flag == 5 || flag == 7; }
SRM_HD inline int64_t own_window(int L, int flag, int k) { return (int64_t)L + (has_start(flag) ? k : 0) + (has_end(flag) ? k : 0); }

// the window of w bases at pos leaves the genome or meets a separator (hash.c:982)
SRM_HD inline bool outside(const uint8_t *blocked, uint64_t glen, int32_t pos, int64_t w)
{
    if ((uint64_t)pos + (uint64_t)w > glen) return true;
    if (!blocked) return false;
    int64_t j = 0;
    for (; j + 8 <= w; j += 8) {
        uint64_t x;
        __builtin_memcpy(&x, blocked + pos + j, 8);
        if (x) return true;
    }
    for (; j < w; ++j)
        if (blocked[pos + j]) return true;
    return false;
}

// entries of a read that outgrew its slots are not there yet
SRM_HD inline uint32_t entries_of(uint32_t word) { return word == srm_pair::OVERFLOW_MARK ? 0u : word & 0xFFFFu; }
SRM_HD inline uint32_t perfects_of(uint32_t word) { return word == srm_pair::OVERFLOW_MARK ? 0u : word >> 16; }

// a read's counts over its ne entries; unsafe: one of them could be skipped, leaky:
// the last one could
SRM_HD inline Counts count_entries(const int32_t *pos, const int8_t *flag, uint32_t ne, int L, int k,
                                   int kmax, uint64_t glen, const uint8_t *blocked, bool &unsafe,
                                   bool &leaky)
{
    Counts c;
    unsafe = leaky = false;
    for (uint32_t i = 0; i < ne; ++i) {
        leaky = false;
        if (pos[i] <= 0) continue;
        ++c.queued;
        if (!outside(blocked, glen, pos[i], own_window(L, flag[i], k))) ++c.cand;
        leaky = outside(blocked, glen, pos[i], (int64_t)L + 2 * kmax);
        unsafe |= leaky;
    }
    c.with = ne != 0;
    return c;
}

// a read the host walks
struct Walked {
    uint32_t read, rank, cand_start;   // rank: among the reads with entries
    std::vector<int32_t> pos;
    std::vector<int8_t> flag;
};

// a flush: the reads before `hi` that no earlier one took, and the dense candidates
// before hi
struct Flush {
    uint32_t hi, cand;
};

// the flushes over the dense candidates with the walked reads' changes: window
// lengths set in place, skipped candidates left out
inline void finish(srm_filter_impl::Pieces &R, std::vector<uint64_t> &batch_end,
                   const std::vector<Flush> &flushes, std::vector<Walked> &walked,
                   const uint16_t *read_len, const uint8_t *read_k, uint64_t glen,
                   const uint8_t *blocked)
{
    std::sort(walked.begin(), walked.end(),
              [](const Walked &x, const Walked &y) { return x.read < y.read; });
    walked.erase(std::unique(walked.begin(), walked.end(),
                             [](const Walked &x, const Walked &y) { return x.read == y.read; }),
                 walked.end());
    std::vector<uint64_t> left_out;   // dense candidates, ascending
    int s = 0, e = 0;
    uint32_t next_rank = 0;
    for (const Walked &W : walked) {
        if (W.rank != next_rank) s = e = 0;   // another read's entry between
        next_rank = W.rank + 1;
        const int L = read_len[W.read], k = read_k[W.read];
        uint64_t at = W.cand_start;
        for (size_t i = 0; i < W.pos.size(); ++i) {
            const int32_t pos = W.pos[i];
            const int flag = W.flag[i];
            if (pos > 0) {
                if (has_end(flag)) e = k;
                if (has_start(flag)) s = k;
                const int64_t w = (int64_t)L + s + e;
                const bool skip = outside(blocked, glen, pos, w);
                if (!outside(blocked, glen, pos, own_window(L, flag, k))) {   // dense candidate `at`
                    if (skip) left_out.push_back(at);
                    else R.c_w[at] = (uint16_t)w;
                    ++at;
                }
                if (skip) continue;
            }
            s = e = 0;
        }
    }
    uint64_t dense = 0, total = 0;
    size_t x = 0;
    for (const Flush &f : flushes) {
        const uint64_t before = total;
        for (; x < left_out.size() && left_out[x] < f.cand; ++x) {
            R.add(dense, left_out[x] - dense);
            total += left_out[x] - dense;
            dense = left_out[x] + 1;
        }
        R.add(dense, f.cand - dense);
        total += f.cand - dense;
        dense = f.cand;
        if (total > before) batch_end.push_back(total);
    }
    R.n_cand = total;
}

}  // namespace srm_batch
