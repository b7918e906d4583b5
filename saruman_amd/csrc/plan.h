// plan.h -- what srm_job_upload and srm_align_static decide about each candidate
// before a launch, as host/device code: whether it is valid, which kernel takes it,
// and for the unit-cost band kernels its place among the tiles.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "nw_device.h"

namespace srm {

// srm_ops_words, for both sides
__host__ __device__ inline uint32_t slot_words(uint32_t w, uint32_t k) { return (w + k + 15u) / 16u; }

// a candidate's route, or (from E_RANGE on) why it is refused
enum { K_BAND, K_REST, K_BYTES, E_RANGE, E_BYTES, E_READ, E_GENOME, E_WIN, E_OPS, E_PLAIN };

// the arrays behind the candidates, and the launch tuning
struct PlanIn {
    uint64_t read_codes, win_codes;       // codes in the arrays, padding included
    uint64_t read_bytes, win_bytes;       // raw bytes
    uint64_t ops_words;                   // room for transcripts (static)
    bool resident_genome;                 // windows are offsets into a padded genome
    bool band_ok;                         // costs the band takes
    bool only_band;                       // static: anything else is refused
    int merge_below, split_len;
};

__host__ __device__ inline int classify(const PlanIn &in, const srm_cand &c)
{
    const uint64_t pad = SRM_CODE_PAD;
    if (c.L < 1 || c.L > SRM_MAX_L || c.w > SRM_MAX_W) return E_RANGE;
    if (c.bits & SRM_CAND_BYTES) {
        if (in.only_band || (uint64_t)c.read_off + c.L > in.read_bytes ||
            (uint64_t)c.win_off + c.w > in.win_bytes)
            return E_BYTES;
        return K_BYTES;
    }
    // code arrays: pad codes readable before 0 and after the end (the caller's
    // arrays start with SRM_CODE_PAD pad codes for uploaded arrays, and offsets
    // count from the first code after them).  Written without subtraction: an
    // array shorter than the padding must fail, not wrap.
    if ((uint64_t)c.read_off + c.L + 2 * pad > in.read_codes) return E_READ;
    if (in.resident_genome) {
        // the genome carries SRM_CODE_PAD codes of padding at both ends
        if ((uint64_t)c.win_off < pad || (uint64_t)c.win_off + c.w + pad > in.win_codes) return E_GENOME;
    } else if ((uint64_t)c.win_off + c.w + 2 * pad > in.win_codes) {
        return E_WIN;
    }
    if (in.only_band && (uint64_t)c.ops_off + slot_words(c.w, c.k) > in.ops_words) return E_OPS;
    // banded: exact-band conditions, and w >= L - k (a shorter window can never
    // hold a hit; the window code stream reads up to L + 93 codes past win_off)
    if (in.band_ok && c.k <= SRM_BAND_KMAX && band_cells(c) <= SRM_BAND_MAX &&
        (int)c.w >= (int)c.L - (int)c.k)
        return K_BAND;
    return in.only_band ? E_PLAIN : K_REST;
}

// the class of a banded candidate: 2 x (band words - 1), + 1 from split_len codes on
// (a class split by read length runs as two launches)
constexpr int PLAN_CLASSES = 16;
__host__ __device__ inline int band_class(const PlanIn &in, const srm_cand &c)
{
    int nw = (band_cells(c) + 7) / 8;
    if (nw < in.merge_below) nw = in.merge_below;
    return 2 * (nw - 1) + (in.split_len > 0 && (int)c.L >= in.split_len ? 1 : 0);
}

// Tiles hold candidates of one class and one L mod 8, longest reads first.  With
// reads of at most PLAN_MAX_L codes that order is the order of these bins, and a
// counting sort's counts give the tiles.
constexpr int PLAN_MAX_L = 511;
constexpr int PLAN_BINS = PLAN_CLASSES * 8 * 64;
__host__ __device__ inline int plan_bin(const PlanIn &in, const srm_cand &c)
{
    return (band_class(in, c) * 8 + (c.L & 7)) * 64 + 63 - (c.L >> 3);
}
__host__ __device__ inline int bin_len(int bin) { return 8 * (63 - (bin & 63)) + ((bin >> 6) & 7); }

// the tiles of the bins' counts: begin(class), tile(first place, candidates, longest
// read) for each of its tiles, end() -- for every class that has candidates
template <class Begin, class Tile, class End>
void plan_tiles(const uint32_t *bin, uint32_t tile_cands, Begin begin, Tile tile, End end)
{
    uint32_t at = 0;   // place in tile order
    for (int cl = 0; cl < PLAN_CLASSES; ++cl) {
        bool any = false;
        for (int lm = 0; lm < 8; ++lm) {
            const uint32_t *run = bin + (cl * 8 + lm) * 64;
            uint32_t stop = at, next = at;   // the run's end; where its next tile starts
            for (int b = 0; b < 64; ++b) stop += run[b];
            for (int b = 0; b < 64; ++b) {
                at += run[b];
                for (; next < at; next += tile_cands) {
                    if (!any) begin(cl);
                    any = true;
                    tile(next, stop - next < tile_cands ? stop - next : tile_cands,
                         bin_len((cl * 8 + lm) * 64 + b));
                }
            }
        }
        if (any) end();
    }
}

// the sums over the candidates, then the bins' counts
struct PlanSums {
    unsigned long long ops_end;   // the longest extent of a transcript slot, words
    unsigned long long rows;      // 2 (w + k)
    uint32_t first_bad;           // the first refused candidate (~0: none)
    uint32_t n_band, n_rest, n_bytes;
    uint32_t too_long;            // banded reads of more than PLAN_MAX_L codes
    uint32_t run;                 // tiles to run, 0 when something forbids it (PlanTiles)
    unsigned long long words;     // of the tiles' scratch (PlanTiles)
    uint32_t n_tiles, pad;        // likewise
    uint32_t bin[PLAN_BINS];
};
// what the plan kernels need besides their inputs and lists
constexpr size_t PLAN_SCRATCH = sizeof(PlanSums) + 2 * PLAN_BINS * sizeof(uint32_t);

// The tiles made on the device too, for srm_align_static: in the order they run, the
// widest band first, w the band; off: where each one's scratch starts.  They run if every
// candidate is banded, no read is longer than PLAN_MAX_L and the call's arrays end within
// `room` (static_end)
struct PlanTiles {
    bool unit;
    uint4 *tiles;
    uint64_t *off;
    uint64_t o_tiles, room;
};
// tiles of n candidates, at most
__host__ __device__ inline uint32_t most_tiles(uint32_t n) { return n / 64 + PLAN_CLASSES / 2 * 8; }
__host__ __device__ inline uint64_t align256(uint64_t x) { return (x + 255) & ~(uint64_t)255; }
// where the arrays of srm_align_static end: tiles (from o_tiles), their offsets, a score a
// candidate, the tiles' scratch
__host__ __device__ inline uint64_t static_end(uint64_t o_tiles, uint64_t n_tiles, uint64_t n, uint64_t words)
{
    return align256(align256(align256(o_tiles + n_tiles * 16) + n_tiles * 8) + n * 4) + words * 4;
}

// counts the candidates into scratch (a PlanSums at its start) and writes the banded
// ones in tile order (perm, cand_tile) and the indexes of the others to rest and
// bytes (null: none can come), in no order
hipError_t launch_plan(const PlanIn &in, const srm_cand *cand, uint32_t n, void *scratch,
                       uint32_t *perm, srm_cand *cand_tile, uint32_t *rest, uint32_t *bytes,
                       hipStream_t st, const PlanTiles *tiles = nullptr);

}  // namespace srm
