// Runs the band kernels for costs other than 0/1 (saruman_amd/csrc/nw_kernels.hip:
// nibble_band_tile and nibble_trace_tile) on the CPU, every lane of every wave in turn
// (through tests/emu/hip/hip_runtime.h), over random candidates, and compares each score,
// transcript and end cell with the oracle (oracle/nw_oracle.c: oracle_fill,
// oracle_traceback).  TEST INFRASTRUCTURE ONLY.
//
// usage: nibble_emu N seed match mismatch maxL [plant] -> a summary line, exit status 1 on
// a mismatch.  "plant" reads the oracle's gap rows the wrong way round (top for left), a
// mistake planted in the checker, which the comparison must report.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <stdio.h>
#include <stdlib.h>
#include <vector>

// names of nw_kernels.hip that the kernels run here do not reach
inline uint64_t __ballot(bool x) { return x; }
inline int __builtin_amdgcn_readlane(int x, int) { return x; }
inline int __builtin_amdgcn_update_dpp(int, int x, int, int, int, bool) { return x; }
inline void __threadfence_block() {}
inline uint32_t atomicAdd(uint32_t *p, uint32_t v) { return (*p += v) - v; }
extern EmuIdx gridDim;

#include "nw_kernels.hip"

thread_local EmuIdx threadIdx, blockIdx, blockDim;
EmuIdx gridDim;
namespace srm {
uint32_t trace_lds[64 * 64];    // one wave's staged codes
hipError_t launch_bits_band(const BandArgs &, int, int, int, hipStream_t) { return 0; }
hipError_t launch_bits_trace(const BandArgs &, int, int, hipStream_t) { return 0; }
hipError_t launch_bits_all(const BandArgs &, const BitsSpans &, hipStream_t) { return 0; }
int bits_band_occupancy(int) { return 1; }
}

extern "C" int oracle_fill(int ma, int mm, int k, const char *win, int w, const char *read, int L,
                           int flag, int16_t *M);
extern "C" int oracle_traceback(int ma, int mm, int k, const char *win, int w, const char *read,
                                int L, int flag, int stop_at_row0, const int16_t *M, char *R,
                                char *G, int cap, int *end_row, int *end_col);

namespace {

uint64_t rng;
int ma, mm;
bool plant = false;
uint32_t rnd()
{
    rng ^= rng << 13;
    rng ^= rng >> 7;
    rng ^= rng << 17;
    return (uint32_t)(rng >> 11);
}

struct Case {
    std::vector<uint8_t> r, g;
    int L, w, k, flag, stop;
};
long hits = 0, bad = 0, steps[3] = {0, 0, 0};

std::vector<uint32_t> packed(std::vector<uint8_t> c)
{
    for (int i = 0; i < SRM_CODE_PAD + 64; ++i) c.push_back(rnd() & 3);
    std::vector<uint32_t> w(c.size() / 16 + 2, 0u);
    for (size_t i = 0; i < c.size(); ++i) w[i / 16] |= (uint32_t)c[i] << (2 * (i % 16));
    return w;
}

template <int NW>
void run_class(std::vector<Case> &cs)
{
    const int n = (int)cs.size();
    if (!n) return;
    std::stable_sort(cs.begin(), cs.end(), [](const Case &x, const Case &y) { return x.L > y.L; });
    std::vector<uint8_t> rc, wc;
    for (int i = 0; i < SRM_CODE_PAD; ++i) {
        rc.push_back(rnd() & 3);
        wc.push_back(rnd() & 3);
    }
    std::vector<srm_cand> cand(n);
    std::vector<uint32_t> perm(n);
    uint32_t ops_end = 0;
    for (int t = 0; t < n; ++t) {
        srm_cand &cd = cand[t];
        perm[t] = (uint32_t)t;
        cd.read_off = (uint32_t)(rc.size() - SRM_CODE_PAD);
        cd.win_off = (uint32_t)(wc.size() - SRM_CODE_PAD);
        rc.insert(rc.end(), cs[t].r.begin(), cs[t].r.end());
        wc.insert(wc.end(), cs[t].g.begin(), cs[t].g.end());
        cd.L = (uint16_t)cs[t].L;
        cd.w = (uint16_t)cs[t].w;
        cd.k = (uint8_t)cs[t].k;
        cd.flag = (uint8_t)cs[t].flag;
        cd.bits = cs[t].stop ? SRM_CAND_STOP_ROW0 : 0;
        cd.pad = 0;
        cd.ops_off = ops_end;
        ops_end += (cs[t].w + cs[t].k + 15) / 16;
    }
    const std::vector<uint32_t> rw = packed(rc), ww = packed(wc);
    std::vector<uint4> tiles;
    std::vector<uint64_t> off;
    size_t words = 0;
    for (int b = 0; b < n; b += 64) {
        tiles.push_back(uint4{(uint32_t)b, (uint32_t)std::min(64, n - b), (uint32_t)cs[b].L, 0u});
        off.push_back(words);
        words += srm::tile_scratch_words(NW, cs[b].L);
    }
    std::vector<uint32_t> scratch(words, 0xDEADBEEFu), ops(ops_end + 1, 0u);
    std::vector<srm_result> res(n);
    srm::BandArgs a{};
    a.ma = ma;
    a.mm = mm;
    a.cand = cand.data();
    a.perm = perm.data();
    a.tiles = tiles.data();
    a.ntiles = (uint32_t)tiles.size();
    a.read_words = rw.data() + SRM_CODE_PAD / 16;
    a.win_words = ww.data() + SRM_CODE_PAD / 16;
    a.scratch = scratch.data();
    a.tile_scratch = off.data();
    a.res = res.data();
    a.ops = ops.data();
    for (uint32_t tile = 0; tile < a.ntiles; ++tile) {
        a.code_words = srm::trace_code_words((int)tiles[tile].z);
        for (uint32_t lane = 0; lane < 64; ++lane) {
            threadIdx.x = lane;
            srm::nibble_band_tile<NW>(a, tile);
        }
        for (uint32_t lane = 0; lane < 64; ++lane) {
            threadIdx.x = lane;
            srm::nibble_trace_tile<NW>(a, tile);
        }
    }
    for (int t = 0; t < n; ++t) {
        const Case &c = cs[t];
        std::vector<char> rch(c.L + 1), wch(c.w + 1), R(c.w + c.k + 1), G(c.w + c.k + 1);
        for (int i = 0; i < c.L; ++i) rch[i] = "ACGT"[c.r[i]];
        for (int i = 0; i < c.w; ++i) wch[i] = "ACGT"[c.g[i]];
        std::vector<int16_t> M((size_t)(c.w + 1) * (c.L + 1));
        const int sc = oracle_fill(ma, mm, c.k, wch.data(), c.w, rch.data(), c.L, c.flag, M.data());
        bool ok = res[t].score == std::min(sc, c.k + 1);
        int nn = 0, row = c.w, col = c.L;
        if (sc <= c.k) {
            ++hits;
            nn = oracle_traceback(ma, mm, c.k, wch.data(), c.w, rch.data(), c.L, c.flag, c.stop, M.data(),
                                  R.data(), G.data(), c.w + c.k, &row, &col);
        }
        ok = ok && res[t].n_ops == nn && res[t].end_row == row && res[t].end_col == col;
        for (int u = 0; u < nn; ++u) {
            int op = R[nn - 1 - u] == '_' ? 1 : G[nn - 1 - u] == '_' ? 2 : 0;
            ++steps[op];
            if (plant && op) op = 3 - op;
            ok = ok && ((ops[cand[t].ops_off + u / 16] >> (2 * (u % 16))) & 3u) == (uint32_t)op;
        }
        if (!ok && bad++ < 5)
            fprintf(stderr, "mismatch NW%d L=%d w=%d k=%d flag=%d stop=%d: score %d ops %d end %d,%d "
                    "(oracle %d, %d, %d,%d)\n", NW, c.L, c.w, c.k, c.flag, c.stop, res[t].score,
                    res[t].n_ops, res[t].end_row, res[t].end_col, sc, nn, row, col);
    }
}

}  // namespace

int main(int argc, char **argv)
{
    if (argc < 6) return 2;
    const int N = atoi(argv[1]), maxL = atoi(argv[5]);
    rng = strtoull(argv[2], nullptr, 0) * 2 + 1;
    ma = atoi(argv[3]);
    mm = atoi(argv[4]);
    plant = argc > 6;
    std::vector<Case> by[9];
    for (int t = 0; t < N; ++t) {
        Case c;
        const int k = (int)(rnd() % 15), flag = (int)(rnd() % 9);
        const int L = 1 + (int)(rnd() % (unsigned)maxL);
        const int s = srm::flag_s(flag, k), e = srm::flag_e(flag, k);
        // the filter's windows, or any that the band takes
        const int w = rnd() % 2 ? L + s + e : std::max(0, L - k + (int)(rnd() % (unsigned)(2 * k + 2 * s + 1)));
        srm_cand b{};
        b.L = (uint16_t)L;
        b.w = (uint16_t)w;
        b.k = (uint8_t)k;
        b.flag = (uint8_t)flag;
        if (srm::band_cells(b) > SRM_BAND_MAX || w < L - k) continue;
        const int nw = (srm::band_cells(b) + 7) / 8;
        c.g.resize((size_t)w);
        c.r.resize((size_t)L);
        for (auto &x : c.g) x = rnd() & 3;
        // random reads; otherwise copies from a place of the window with substitutions
        // and gaps
        const int mode = (int)(rnd() % 4);
        int p = mode < 2 || w == 0 ? 0 : (int)(rnd() % (unsigned)(2 * s + 1));
        for (int i = 0; i < L; ++i, ++p) {
            if (mode == 3 && rnd() % 24 == 0) ++p;
            else if (mode == 3 && rnd() % 24 == 0 && p > 0) --p;
            c.r[i] = mode && p < w && rnd() % 12 ? c.g[p] : (uint8_t)(rnd() & 3);
        }
        c.L = L;
        c.w = w;
        c.k = k;
        c.flag = flag;
        c.stop = rnd() % 5 == 0;
        by[nw].push_back(c);
    }
    run_class<1>(by[1]);
    run_class<2>(by[2]);
    run_class<3>(by[3]);
    run_class<4>(by[4]);
    run_class<5>(by[5]);
    run_class<6>(by[6]);
    run_class<7>(by[7]);
    run_class<8>(by[8]);
    printf("cases %d hits %ld bad %ld diag %ld top %ld left %ld\n", N, hits, bad, steps[0], steps[1], steps[2]);
    return bad != 0;
}
