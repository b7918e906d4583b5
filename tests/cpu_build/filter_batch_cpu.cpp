// Checks the device filter's batch pass (saruman_amd/csrc/filter_batch.h: counts per
// read, dense output, the host's walk of the few reads that depend on others) against
// the host's pass (filter_internal.h: batch_pass) over random filter entries.  The
// kernels' parts run here as plain loops.  TEST INFRASTRUCTURE ONLY.
//
// usage: filter_batch_cpu seed cases [plant] -> one line, exit status 1 on a difference;
// "plant" gives the expected pass another chunk value, which the comparison must report
#include <stdio.h>
#include <stdlib.h>

#include "filter_batch.h"

using namespace srm_batch;
using namespace srm_filter_impl;

int main(int argc, char **argv)
{
    uint64_t x = strtoull(argv[1], nullptr, 0) * 0x9E3779B97F4A7C15ull + 1;
    const int cases = atoi(argv[2]);
    const bool plant = argc > 3;
    auto next = [&] {
        x ^= x << 13;
        x ^= x >> 7;
        x ^= x << 17;
        return x >> 11;
    };
    long cands = 0, left_out = 0, bad = 0;
    for (int t = 0; t < cases; ++t) {
        const size_t n = 1 + next() % 60, glen = 300 + next() % 3000;
        const int cv = 1 + (int)(next() % (1 + next() % 40)), kset = (int)(next() % 3);
        std::vector<uint8_t> sep(glen, 0);
        const bool with_sep = next() % 2;
        if (with_sep)
            for (int i = 0; i < 3; ++i) sep[next() % glen] = 1;
        const uint8_t *blocked = with_sep ? sep.data() : nullptr;
        std::vector<uint16_t> L(n);
        std::vector<uint8_t> k(n);
        std::vector<uint32_t> meta;
        std::vector<int32_t> pos, perf;
        std::vector<int8_t> flag;
        int kmax = 0;
        const int ends = 1 + (int)(next() % 8);   // one entry in so many lies near the end
        for (size_t r = 0; r < n; ++r) {
            L[r] = (uint16_t)(20 + next() % 60);
            k[r] = (uint8_t)(kset == 0 ? 3 : next() % (kset == 1 ? 6 : 30));
            kmax = std::max<int>(kmax, k[r]);
            const uint32_t ne = next() % 3 == 0 ? 0 : (uint32_t)(next() % 5), np = (uint32_t)(next() % 2);
            meta.push_back((uint32_t)pos.size());
            meta.push_back((uint32_t)perf.size());
            meta.push_back(ne | (np << 16));
            for (uint32_t e = 0; e < ne; ++e) {
                int64_t p = next() % ends == 0 ? (int64_t)glen - L[r] - 40 + (int64_t)(next() % 60)
                                               : 1 + (int64_t)(next() % glen);
                p = std::min<int64_t>(std::max<int64_t>(p, 1), (int64_t)glen);
                const bool perfect = next() % 5 == 0;
                pos.push_back((int32_t)(perfect ? -p : p));
                flag.push_back(perfect ? 0 : (int8_t)(next() % 8));
            }
            for (uint32_t e = 0; e < np; ++e) perf.push_back((int32_t)(next() % glen));
        }
        srm_filter *W = batch_pass(MetaAcc{meta, pos, flag, perf}, n, L.data(), k.data(), glen, blocked,
                                   plant ? cv + 1 : cv);
        // the kernels: counts, their sums, the dense output, the flushes, the walked reads
        std::vector<Counts> start(n + 1);
        std::vector<uint32_t> by_rank;
        std::vector<std::pair<uint32_t, bool>> unsafe_reads;
        std::vector<int64_t> c_pos, p_pos;
        std::vector<int32_t> c_read, p_read;
        std::vector<uint16_t> c_w;
        std::vector<uint8_t> c_flag;
        for (size_t r = 0; r < n; ++r) {
            const uint32_t ne = entries_of(meta[3 * r + 2]), np = perfects_of(meta[3 * r + 2]);
            bool uns, leaky;
            Counts c = count_entries(pos.data() + meta[3 * r], flag.data() + meta[3 * r], ne, L[r], k[r],
                                     kmax, glen, blocked, uns, leaky);
            c.perf = np;
            if (uns) unsafe_reads.push_back({(uint32_t)r, leaky});
            start[r + 1] = CountsSum()(start[r], c);
            if (ne) by_rank.push_back((uint32_t)r);
            for (uint32_t e = 0; e < ne; ++e) {
                const int32_t p = pos[meta[3 * r] + e];
                const int f = flag[meta[3 * r] + e];
                const int64_t w = own_window(L[r], f, k[r]);
                if (p <= 0 || outside(blocked, glen, p, w)) continue;
                c_pos.push_back(p);
                c_read.push_back((int32_t)r);
                c_w.push_back((uint16_t)w);
                c_flag.push_back((uint8_t)f);
            }
            for (uint32_t e = 0; e < np; ++e) {
                p_pos.push_back(perf[meta[3 * r + 1] + e]);
                p_read.push_back((int32_t)r);
            }
        }
        std::vector<Flush> flushes;
        for (size_t lo = 0; lo < n;) {
            size_t r = lo;
            while (r < n && start[r + 1].queued - start[lo].queued <= (uint32_t)cv) ++r;
            if (r >= n && start[n].queued == start[lo].queued) break;
            lo = r >= n ? n : r + 1;
            flushes.push_back({(uint32_t)lo, start[lo].cand});
        }
        std::vector<Walked> walked;
        auto put = [&](uint32_t r) {
            Walked w;
            w.read = r;
            w.rank = start[r].with;
            w.cand_start = start[r].cand;
            w.pos.assign(pos.begin() + meta[3 * r], pos.begin() + meta[3 * r] + entries_of(meta[3 * r + 2]));
            w.flag.assign(flag.begin() + meta[3 * r], flag.begin() + meta[3 * r] + entries_of(meta[3 * r + 2]));
            walked.push_back(w);
        };
        for (size_t u = unsafe_reads.size(); u-- > 0;) {   // the kernel lists them in any order
            put(unsafe_reads[u].first);
            const uint32_t rank = start[unsafe_reads[u].first].with + 1;
            if (unsafe_reads[u].second && rank < start[n].with) put(by_rank[rank]);
        }
        srm_filter D;
        D.dense = std::make_unique<Pieces>();
        Pieces &R = *D.dense;
        R.c_pos = c_pos.data();
        R.c_read = c_read.data();
        R.c_w = c_w.data();
        R.c_flag = c_flag.data();
        R.p_pos = p_pos.data();
        R.p_read = p_read.data();
        R.n_perf = p_pos.size();
        finish(R, D.batch_end, flushes, walked, L.data(), k.data(), glen, blocked);
        uint64_t nc, nb, np;
        srm_filter_sizes(&D, &nc, &nb, &np);
        srm_filter G;
        G.c_read.resize(nc);
        G.c_pos.resize(nc);
        G.c_flag.resize(nc);
        G.c_w.resize(nc);
        G.batch_end.resize(nb);
        G.p_read.resize(np);
        G.p_pos.resize(np);
        srm_filter_copy(&D, G.c_read.data(), G.c_pos.data(), G.c_flag.data(), G.c_w.data(),
                        G.batch_end.data(), G.p_read.data(), G.p_pos.data());
        const bool ok = G.c_read == W->c_read && G.c_pos == W->c_pos && G.c_flag == W->c_flag &&
                        G.c_w == W->c_w && G.batch_end == W->batch_end && G.p_read == W->p_read &&
                        G.p_pos == W->p_pos;
        bad += !ok;
        cands += (long)nc;
        left_out += (long)(c_read.size() - nc);
        delete W;
    }
    printf("%s cases=%d candidates=%ld left_out=%ld bad=%ld\n", bad ? "MISMATCH" : "OK", cases,
           cands, left_out, bad);
    return bad ? 1 : 0;
}
