// static_align.hip -- the banded alignment of a candidate batch without any
// allocation: srm_job_upload + srm_job_run(SRM_KERNEL_BANDED) + the results, for
// callers that cannot allocate device memory (code that a hipGraph capture
// surrounds, tight serving loops, harnesses that forbid allocation).
//
// Everything the band kernels need besides the caller's inputs and outputs -- the
// descriptors in candidate and tile order, the tile table, the per-tile offsets,
// the scores handed from the forward pass to the walk, the class counters and the
// band scratch of every tile -- lives in one file-scope device array, `scratch`,
// of SRM_STATIC_SCRATCH_BYTES.  Each GPU holds its own copy until the process
// ends; its address is taken once per device with hipGetSymbolAddress and used
// for every kernel argument and copy.  The plan (the order by band class, L mod 8 and
// L, and the tiles) is made on the device, or by small calls in fixed host arrays, so
// the call
// allocates nothing on the host either.  Calls are serialised by a mutex: a call
// returns when its results are in the caller's buffers, and the scratch then
// holds that call's contents.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <mutex>

#include "nw_device.h"
#include "plan.h"
#include "saruman_hip.h"

namespace {

// what a call may fill, then the device plan's own arrays and the room by which arrays laid
// out for the most tiles there can be exceed those for the tiles there are
constexpr size_t PLAN_ROOM = (size_t)256 << 10;
static __device__ __align__(256) unsigned char scratch[SRM_STATIC_SCRATCH_BYTES + PLAN_ROOM];
static_assert(PLAN_ROOM / 2 >= srm::PLAN_SCRATCH, "the plan's arrays");

constexpr int MAX_DEVICES = 64;
constexpr size_t MAX_TILES = SRM_STATIC_MAX_CAND / 64 + 8 * 8;
constexpr int MAX_L = SRM_MAX_L;

std::mutex g_mu;
unsigned char *g_scratch[MAX_DEVICES] = {};   // the array's address on each device

// the host plan, rebuilt by each call (under g_mu)
uint32_t h_perm[SRM_STATIC_MAX_CAND];
uint32_t h_tmp[SRM_STATIC_MAX_CAND];
uint8_t h_cls[SRM_STATIC_MAX_CAND];
uint32_t h_tiles[4 * MAX_TILES];
uint64_t h_tile_off[MAX_TILES];
size_t h_lcount[MAX_L + 2];
srm::PlanSums h_sums;
// what one copy sends: the plan's arrays as they lie in the scratch, from the descriptors
// (candidate order, then tile order) to the tile offsets.  Five copies of a few KB were 25
// of the 47 us of 500 candidates of 36 bp
__attribute__((aligned(256))) unsigned char h_image[SRM_STATIC_MAX_CAND * (2 * sizeof(srm_cand) + 4) +
                                                    MAX_TILES * 24 + 5 * 256];

struct Class {
    int nw = 0, maxL = 0;
    uint32_t tile_begin = 0, ntiles = 0;
};

// From this many candidates on the plan is made on the device (plan_gpu.hip), which
// costs launches and a wait and then little per candidate.  Whole calls, host's plan and
// device's, 50-250 bp: 3,317 candidates 140 and 146 us, 4,946 162 and 151, 16,408 246 and
// 162, 49,055 554 and 203
constexpr int PLAN_DEVICE_MIN = 4096;

// why candidate t was refused
int refused(const srm_cand &c, int t, int why)
{
    using srm::set_error;
    switch (why) {
    case srm::E_RANGE:
        return set_error(SRM_EINVAL, "candidate %d: L=%d w=%d outside 1..%d / 0..%d", t, c.L, c.w,
                         SRM_MAX_L, SRM_MAX_W);
    case srm::E_BYTES: return set_error(SRM_EINVAL, "candidate %d: raw bytes need the plain kernel", t);
    case srm::E_READ: return set_error(SRM_EINVAL, "candidate %d: read codes out of bounds", t);
    case srm::E_WIN: return set_error(SRM_EINVAL, "candidate %d: window codes out of bounds", t);
    case srm::E_OPS: return set_error(SRM_EINVAL, "candidate %d: transcript slot out of bounds", t);
    default:
        return set_error(SRM_EINVAL, "candidate %d needs the plain kernel (k=%d, band %d)", t, c.k,
                         srm::band_cells(c));
    }
}

using srm::align256;

}  // namespace

extern "C" int srm_align_static(int device, void *stream, int match, int mismatch,
                                const srm_cand *cand, int n, const uint32_t *d_read_words,
                                size_t n_read_words, const uint32_t *d_win_words,
                                size_t n_win_words, srm_result *d_res, uint32_t *d_ops,
                                size_t n_ops_words)
{
    using srm::set_error;
    std::lock_guard<std::mutex> lk(g_mu);
    if (device < 0 || device >= MAX_DEVICES) return set_error(SRM_EINVAL, "device %d", device);
    if (n < 0 || n > SRM_STATIC_MAX_CAND)
        return set_error(SRM_EINVAL, "srm_align_static takes at most %d candidates, got %d",
                         SRM_STATIC_MAX_CAND, n);
    if (match < 0 || mismatch < 1)
        return set_error(SRM_EINVAL, "srm_align_static needs match >= 0 and mismatch >= 1 "
                                     "(the exact band)");
    if (n > 0 && (!cand || !d_read_words || !d_win_words || !d_res || !d_ops))
        return set_error(SRM_EINVAL, "srm_align_static: null argument");
    if (n == 0) return SRM_OK;

    const bool unit = match == 0 && mismatch == 1;
    // every candidate must fit the exact band and its arrays, as srm_job_upload checks
    // them (the code arrays carry SRM_CODE_PAD codes of padding at both ends; offsets
    // count from the first code after it)
    srm::PlanIn in{};
    in.read_codes = (uint64_t)n_read_words * 16;
    in.win_codes = (uint64_t)n_win_words * 16;
    in.ops_words = n_ops_words;
    in.band_ok = in.only_band = true;
    in.merge_below = 1;

    // the scratch: counters, descriptors in candidate and tile order, perm, then (below)
    // tiles, tile offsets, scores and the band scratch
    size_t at = 0;
    const size_t o_queue = at;
    at = align256(at + 64 * sizeof(uint32_t));
    const size_t o_cand = at;
    at = align256(at + (size_t)n * sizeof(srm_cand));
    const size_t o_cand_tile = at;
    at = align256(at + (size_t)n * sizeof(srm_cand));
    const size_t o_perm = at;
    at = align256(at + (size_t)n * 4);
    unsigned char *base = nullptr;
    hipStream_t st = (hipStream_t)stream;
#define SA_TRY(expr)                                                                          \
    do {                                                                                      \
        hipError_t e_ = (expr);                                                               \
        if (e_ != hipSuccess)                                                                 \
            return set_error(SRM_EDEVICE, "%s failed: %s", #expr, hipGetErrorString(e_));     \
    } while (0)

    auto on_device = [&]() -> int {
        SA_TRY(hipSetDevice(device));
        if (!g_scratch[device]) {   // once per device, with the device current
            void *p = nullptr;
            const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
            if (e != hipSuccess || !p)
                return set_error(SRM_EDEVICE, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
            g_scratch[device] = (unsigned char *)p;
        }
        base = g_scratch[device];
        return SRM_OK;
    };

    Class cls[9];
    int ncls = 0;
    size_t ntiles = 0, words = 0;
    auto add_tile = [&](Class &bc, uint32_t first, uint32_t count, uint32_t lmax) {
        h_tiles[4 * ntiles + 0] = first;
        h_tiles[4 * ntiles + 1] = count;
        h_tiles[4 * ntiles + 2] = lmax;
        h_tiles[4 * ntiles + 3] = 0;
        h_tile_off[ntiles] = words;
        words += unit ? srm::bits_tile_words(bc.nw, (int)lmax, false)
                      : srm::tile_scratch_words(bc.nw, (int)lmax);
        bc.maxL = std::max(bc.maxL, (int)lmax);
        ++bc.ntiles;
        ++ntiles;
    };
    // ---- on the device: checked, counted and put in tile order there; the tiles follow
    // from the counts
    bool planned = false;
    int num_cus = 0;
    if (!unit) SA_TRY(hipDeviceGetAttribute(&num_cus, hipDeviceAttributeMultiprocessorCount, device));
    srm::BandArgs a{};
    a.ma = match;
    a.mm = mismatch;
    a.read_words = d_read_words + SRM_CODE_PAD / 16;
    a.win_words = d_win_words + SRM_CODE_PAD / 16;
    a.res = d_res;
    a.ops = d_ops;
    auto arrays = [&](size_t o_score, size_t o_band) {
        a.cand = (const srm_cand *)(base + o_cand);
        a.perm = (const uint32_t *)(base + o_perm);
        a.cand_tile = (const srm_cand *)(base + o_cand_tile);
        a.tile_score = (int32_t *)(base + o_score);
        a.scratch = (uint32_t *)(base + o_band);
    };
    auto too_large = [&](size_t need) {
        return set_error(SRM_ENOMEM, "srm_align_static: the batch needs %zu bytes of scratch, the "
                                     "static scratch holds %zu; split the batch",
                         need, (size_t)SRM_STATIC_SCRATCH_BYTES);
    };
    if (n >= PLAN_DEVICE_MIN) {
        if (const int rc = on_device()) return rc;
        unsigned char *sums = base + SRM_STATIC_SCRATCH_BYTES + PLAN_ROOM / 2;
        SA_TRY(hipMemcpyAsync(base + o_cand, cand, (size_t)n * sizeof(srm_cand), hipMemcpyHostToDevice, st));
        // while the most tiles there can be fit one launch, the tiles are made there as well
        // and run, or do not, without a wait: 49,055 candidates 206 -> 189 us
        const uint32_t most = srm::most_tiles((uint32_t)n);
        const bool through = srm::all_classes_fit(unit, most, num_cus);
        const size_t o_toff = align256(at + most * 16), o_score = align256(o_toff + most * 8),
                     o_band = align256(o_score + (size_t)n * 4);
        srm::PlanTiles t{unit, (uint4 *)(base + at), (uint64_t *)(base + o_toff), at,
                         SRM_STATIC_SCRATCH_BYTES};
        SA_TRY(srm::launch_plan(in, (const srm_cand *)(base + o_cand), (uint32_t)n, sums,
                                (uint32_t *)(base + o_perm), (srm_cand *)(base + o_cand_tile), nullptr,
                                nullptr, st, through ? &t : nullptr));
        if (through) {
            arrays(o_score, o_band);
            a.tiles = t.tiles;
            a.tile_scratch = t.off;
            srm::BitsSpans sp;
            sp.blocks = most;
            sp.tiles = &((const srm::PlanSums *)sums)->run;
            sp.max_len[0] = srm::PLAN_MAX_L;
            SA_TRY(srm::launch_all(a, sp, unit, st));
        }
        SA_TRY(hipMemcpyAsync(&h_sums, sums, through ? offsetof(srm::PlanSums, bin) : sizeof h_sums,
                              hipMemcpyDeviceToHost, st));
        SA_TRY(hipStreamSynchronize(st));
        if (h_sums.first_bad != ~0u)
            return refused(cand[h_sums.first_bad], (int)h_sums.first_bad,
                           srm::classify(in, cand[h_sums.first_bad]));
        planned = h_sums.too_long == 0;
        if (planned && through)
            return h_sums.run ? SRM_OK
                              : too_large(srm::static_end(at, h_sums.n_tiles, (uint64_t)n, h_sums.words));
        if (planned)
            srm::plan_tiles(h_sums.bin, 64,
                            [&](int cl) {
                                cls[ncls].nw = cl / 2 + 1;
                                cls[ncls].tile_begin = (uint32_t)ntiles;
                            },
                            [&](uint32_t first, uint32_t count, int lmax) {
                                add_tile(cls[ncls], first, count, (uint32_t)lmax);
                            },
                            [&] { ++ncls; });
    }
    // ---- on the host: order by (class, L mod 8, L descending), a counting pass by L,
    // then a stable one by (class, L mod 8); tiles of up to 64 candidates of one class
    // and one L mod 8
    if (!planned) {
        int maxL = 0;
        for (int t = 0; t < n; ++t) {
            const int why = srm::classify(in, cand[t]);
            if (why != srm::K_BAND) return refused(cand[t], t, why);
            h_cls[t] = (uint8_t)((srm::band_cells(cand[t]) + 7) / 8);
            maxL = std::max(maxL, (int)cand[t].L);
        }
        std::fill(h_lcount, h_lcount + maxL + 2, (size_t)0);
        for (int t = 0; t < n; ++t) ++h_lcount[(size_t)(maxL - cand[t].L) + 1];
        for (int x = 1; x <= maxL + 1; ++x) h_lcount[x] += h_lcount[x - 1];
        for (int t = 0; t < n; ++t) h_tmp[h_lcount[maxL - cand[t].L]++] = (uint32_t)t;
        size_t bk[9 * 8 + 1] = {};
        auto key = [&](uint32_t t) { return (size_t)h_cls[t] * 8 + (cand[t].L & 7); };
        for (int i = 0; i < n; ++i) ++bk[key(h_tmp[i]) + 1];
        for (size_t x = 1; x < 9 * 8 + 1; ++x) bk[x] += bk[x - 1];
        for (int i = 0; i < n; ++i) h_perm[bk[key(h_tmp[i])]++] = h_tmp[i];
        for (int i = 0; i < n;) {
            Class &bc = cls[ncls++];
            bc.nw = h_cls[h_perm[i]];
            bc.tile_begin = (uint32_t)ntiles;
            int e2 = i;
            while (e2 < n && h_cls[h_perm[e2]] == bc.nw) ++e2;
            for (int g = i; g < e2;) {
                int ge = g;
                while (ge < e2 && (cand[h_perm[ge]].L & 7) == (cand[h_perm[g]].L & 7)) ++ge;
                for (int s = g; s < ge; s += 64) {
                    const int cnt = std::min(64, ge - s);
                    uint32_t lmax = 0;
                    for (int u = s; u < s + cnt; ++u) lmax = std::max<uint32_t>(lmax, cand[h_perm[u]].L);
                    add_tile(bc, (uint32_t)s, (uint32_t)cnt, lmax);
                }
                g = ge;
            }
            i = e2;
        }
    }

    const size_t o_tiles = at;
    at = align256(at + ntiles * 16);
    const size_t o_toff = at;
    at = align256(at + ntiles * 8);
    const size_t o_score = at;
    at = align256(at + (size_t)n * 4);
    const size_t o_band = at;
    at += words * 4;
    if (at > SRM_STATIC_SCRATCH_BYTES) return too_large(at);

    // the arrays that the host made, in one copy
    const size_t o_first = planned ? o_tiles : o_cand;
    auto image = [&](size_t o) { return h_image + (o - o_first); };
    if (!planned) {
        if (const int rc = on_device()) return rc;
        std::memcpy(image(o_cand), cand, (size_t)n * sizeof(srm_cand));
        auto *in_order = (srm_cand *)image(o_cand_tile);
        for (int p = 0; p < n; ++p) in_order[p] = cand[h_perm[p]];
        std::memcpy(image(o_perm), h_perm, (size_t)n * 4);
    }
    std::memcpy(image(o_tiles), h_tiles, ntiles * 16);
    std::memcpy(image(o_toff), h_tile_off, ntiles * 8);
    SA_TRY(hipMemcpyAsync(base + o_first, h_image, o_toff + ntiles * 8 - o_first, hipMemcpyHostToDevice, st));
    arrays(o_score, o_band);
    if (srm::all_classes_fit(unit, ntiles, num_cus)) {   // one launch, the widest band first
        srm::BitsSpans sp;
        for (int c = ncls; c-- > 0;) sp.add(cls[c].nw, cls[c].tile_begin, cls[c].ntiles, cls[c].maxL);
        a.tiles = (const uint4 *)(base + o_tiles);
        a.tile_scratch = (const uint64_t *)(base + o_toff);
        SA_TRY(srm::launch_all(a, sp, unit, st));
    } else {
        // the class counters of the persistent kernel start at zero
        SA_TRY(srm::launch_reset((uint32_t *)(base + o_queue), ncls, st));
        for (int c = 0; c < ncls; ++c) {
            const Class &bc = cls[c];
            a.tiles = (const uint4 *)(base + o_tiles) + bc.tile_begin;
            a.ntiles = bc.ntiles;
            a.queue = (uint32_t *)(base + o_queue) + c;
            a.tile_scratch = (const uint64_t *)(base + o_toff) + bc.tile_begin;
            // persistent grid: the blocks that stay resident, at most a wave per tile
            const int blocks = std::min((int)((bc.ntiles + 3) / 4),
                                        std::max(1, num_cus * srm::band_occupancy(bc.nw, false)));
            SA_TRY(srm::launch_band(a, bc.nw, unit, blocks, bc.maxL, st));
            SA_TRY(srm::launch_trace(a, bc.nw, unit, bc.maxL, st));
        }
    }
    // the host arrays and the scratch are reused by the next call
    SA_TRY(hipStreamSynchronize(st));
#undef SA_TRY
    return SRM_OK;
}
