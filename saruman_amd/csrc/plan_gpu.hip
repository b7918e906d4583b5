// plan_gpu.hip -- the upload's plan on the device: every candidate's checks and
// route, and the unit-cost band kernels' tile order by a counting sort over the bins
// of plan.h.  The order inside a bin is any: a candidate's result depends on no other.
//
// 810,000 candidates: 17 + 12 us and two small launches of 5; 53,000: 12 + 14 and those.
// Bound by the descriptors' bytes (20 read twice, 24 written per candidate) and, for
// few, by the launches.  A block sorts its own candidates' bins in LDS and takes a
// range of each with one atomic, so that equal reads (every one of a class may fall
// into one bin) do not queue at one address.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "plan.h"

namespace {

using namespace srm;

constexpr int PT = 1024;          // threads per block
constexpr int PER = 4;            // candidates per thread
constexpr int PB = PT * PER;      // per block

__global__ void __launch_bounds__(PT) plan_zero(PlanSums *s)
{
    uint32_t *w = (uint32_t *)s;
    for (uint32_t i = threadIdx.x; i < sizeof(PlanSums) / 4; i += PT) w[i] = 0;
    __syncthreads();
    if (threadIdx.x == 0) s->first_bad = ~0u;
}

__global__ void __launch_bounds__(PT) plan_count(PlanIn in, const srm_cand *__restrict__ cand,
                                                 uint32_t n, PlanSums *s)
{
    __shared__ uint32_t bin[PLAN_BINS];
    __shared__ unsigned long long ops_end, rows;
    __shared__ uint32_t count[4], bad;
    for (int i = threadIdx.x; i < PLAN_BINS; i += PT) bin[i] = 0;
    if (threadIdx.x < 4) count[threadIdx.x] = 0;
    if (threadIdx.x == 0) {
        ops_end = rows = 0;
        bad = ~0u;
    }
    __syncthreads();
    unsigned long long my_ops = 0, my_rows = 0;
    uint32_t my_bad = ~0u, my[4] = {0, 0, 0, 0};
    for (int u = 0; u < PER; ++u) {
        const uint32_t t = blockIdx.x * PB + u * PT + threadIdx.x;
        if (t >= n) break;
        const srm_cand c = cand[t];
        const int r = classify(in, c);
        if (r >= E_RANGE) {
            if (my_bad == ~0u) my_bad = t;
            continue;
        }
        const unsigned long long end = (unsigned long long)c.ops_off + slot_words(c.w, c.k);
        if (end > my_ops) my_ops = end;
        my_rows += 2 * ((unsigned)c.w + c.k);
        if (r != K_BAND) ++my[r];
        else if (c.L > PLAN_MAX_L) ++my[3];
        else {
            ++my[0];
            atomicAdd(&bin[plan_bin(in, c)], 1u);
        }
    }
    for (int d = 32; d; d >>= 1) {
        const unsigned long long o = __shfl_xor(my_ops, d, 64);
        if (o > my_ops) my_ops = o;
        my_rows += __shfl_xor(my_rows, d, 64);
        const uint32_t b = (uint32_t)__shfl_xor((int)my_bad, d, 64);
        if (b < my_bad) my_bad = b;
        for (int i = 0; i < 4; ++i) my[i] += (uint32_t)__shfl_xor((int)my[i], d, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        atomicMax(&ops_end, my_ops);
        atomicAdd(&rows, my_rows);
        atomicMin(&bad, my_bad);
        for (int i = 0; i < 4; ++i)
            if (my[i]) atomicAdd(&count[i], my[i]);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < PLAN_BINS; i += PT)
        if (bin[i]) atomicAdd(&s->bin[i], bin[i]);
    if (threadIdx.x == 0) {
        atomicMax(&s->ops_end, ops_end);
        atomicAdd(&s->rows, rows);
        if (bad != ~0u) atomicMin(&s->first_bad, bad);
        if (count[0]) atomicAdd(&s->n_band, count[0]);
        if (count[1]) atomicAdd(&s->n_rest, count[1]);
        if (count[2]) atomicAdd(&s->n_bytes, count[2]);
        if (count[3]) atomicAdd(&s->too_long, count[3]);
    }
}

// the sum over the threads before this one; total: over all
__device__ __forceinline__ uint32_t excl_sum(uint32_t v, uint32_t &total)
{
    __shared__ uint32_t wave[PT / 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    uint32_t incl = v;
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)incl, d, 64);
        if (lane >= d) incl += o;
    }
    __syncthreads();   // the sums before have been read
    if (lane == 63) wave[wv] = incl;
    __syncthreads();
    uint32_t at = incl - v;
    total = 0;
    for (int w = 0; w < PT / 64; ++w) {
        if (w < wv) at += wave[w];
        total += wave[w];
    }
    return at;
}

// The tiles of the bins whose first places are in place[] (PLAN_BINS + 1 of them): a run is
// one class and one L mod 8, 64 bins; tile j of a run starts at its place 64 j, and the bin
// that holds it has its longest reads.
__device__ __forceinline__ void make_tiles(PlanSums *s, uint32_t n, const uint32_t *place, const PlanTiles &t)
{
    constexpr int RUNS = PLAN_CLASSES * 8;
    __shared__ uint32_t first[RUNS + 1];
    auto run_of = [](int x) { return (PLAN_CLASSES - 1 - x / 8) * 8 + x % 8; };   // widest first
    uint32_t mine = 0, n_tiles;
    if (threadIdx.x < RUNS) {
        const uint32_t *p = place + 64 * run_of((int)threadIdx.x);
        mine = (p[64] - p[0] + 63) / 64;
    }
    const uint32_t f = excl_sum(mine, n_tiles);
    if (threadIdx.x < RUNS) first[threadIdx.x] = f;
    if (threadIdx.x == 0) first[RUNS] = n_tiles;
    __syncthreads();
    uint32_t words = 0;
    for (uint32_t x0 = 0; x0 < n_tiles; x0 += PT) {
        const uint32_t x = x0 + threadIdx.x;
        uint32_t w = 0, all;
        if (x < n_tiles) {
            int lo = 0;   // the last run that starts at or before tile x
            for (int m = RUNS; m > 1;) {
                const int h = m >> 1;
                if (first[lo + h] <= x) lo += h;
                m -= h;
            }
            const int r = run_of(lo);
            const uint32_t *p = place + 64 * r;
            const uint32_t at = p[0] + 64 * (x - first[lo]), left = p[64] - at;
            int b = 0;    // the last bin that starts at or before it
            for (int m = 64; m > 1; m >>= 1)
                if (p[b + (m >> 1)] <= at) b += m >> 1;
            const int nw = r / 16 + 1, len = bin_len(64 * r + b);
            w = (uint32_t)(t.unit ? (size_t)bits_rows(nw, len) * 64 : tile_scratch_words(nw, len));
            t.tiles[x] = make_uint4(at, left < 64 ? left : 64, (uint32_t)len, (uint32_t)nw);
        }
        const uint32_t o = excl_sum(w, all);
        if (x < n_tiles) t.off[x] = (uint64_t)words + o;
        words += all;
    }
    if (threadIdx.x == 0) {
        s->n_tiles = n_tiles;
        s->words = words;
        const bool run = s->first_bad == ~0u && s->too_long == 0 &&
                         static_end(t.o_tiles, n_tiles, n, words) <= t.room;
        s->run = run ? n_tiles : 0;
    }
}

// next[i]: the first place of bin i; the two list lengths start at 0.  TILES: and the tiles
template <bool TILES>
__global__ void __launch_bounds__(PT) plan_starts(PlanSums *s, uint32_t n, uint32_t *next, uint32_t *lists,
                                                  PlanTiles t)
{
    constexpr int E = PLAN_BINS / PT;
    __shared__ uint32_t place[TILES ? PLAN_BINS + 1 : 1];
    uint32_t v[E], sum = 0, total;
    for (int e = 0; e < E; ++e) {
        v[e] = s->bin[threadIdx.x * E + e];
        sum += v[e];
    }
    uint32_t at = excl_sum(sum, total);
    for (int e = 0; e < E; ++e) {
        next[threadIdx.x * E + e] = at;
        if (TILES) place[threadIdx.x * E + e] = at;
        at += v[e];
    }
    if (threadIdx.x < 2) lists[threadIdx.x] = 0;
    if (!TILES) return;
    if (threadIdx.x == 0) place[PLAN_BINS] = total;
    __syncthreads();
    make_tiles(s, n, place, t);
}

__global__ void __launch_bounds__(PT) plan_scatter(PlanIn in, const srm_cand *__restrict__ cand,
                                                   uint32_t n, uint32_t *next, uint32_t *lists,
                                                   uint32_t *__restrict__ perm,
                                                   srm_cand *__restrict__ cand_tile,
                                                   uint32_t *__restrict__ rest,
                                                   uint32_t *__restrict__ bytes)
{
    __shared__ uint32_t bin[PLAN_BINS];
    for (int i = threadIdx.x; i < PLAN_BINS; i += PT) bin[i] = 0;
    __syncthreads();
    int where[PER];
    uint32_t rank[PER];
    srm_cand c[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const uint32_t t = blockIdx.x * PB + u * PT + threadIdx.x;
        where[u] = -1;
        if (t >= n) continue;
        c[u] = cand[t];
        const int r = classify(in, c[u]);
        if (r == K_BAND && c[u].L <= PLAN_MAX_L) {
            where[u] = plan_bin(in, c[u]);
            rank[u] = atomicAdd(&bin[where[u]], 1u);
        } else if (r == K_REST && rest) {
            rest[atomicAdd(&lists[0], 1u)] = t;
        } else if (r == K_BYTES && bytes) {
            bytes[atomicAdd(&lists[1], 1u)] = t;
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < PLAN_BINS; i += PT)
        if (bin[i]) bin[i] = atomicAdd(&next[i], bin[i]);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        if (where[u] < 0) continue;
        const uint32_t p = bin[where[u]] + rank[u];
        perm[p] = blockIdx.x * PB + u * PT + threadIdx.x;
        cand_tile[p] = c[u];
    }
}

}  // namespace

namespace srm {

hipError_t launch_plan(const PlanIn &in, const srm_cand *cand, uint32_t n, void *scratch,
                       uint32_t *perm, srm_cand *cand_tile, uint32_t *rest, uint32_t *bytes,
                       hipStream_t st, const PlanTiles *tiles)
{
    auto *s = (PlanSums *)scratch;
    uint32_t *next = (uint32_t *)(s + 1), *lists = next + PLAN_BINS;
    const dim3 grid((n + PB - 1) / PB);
    hipLaunchKernelGGL(plan_zero, dim3(1), dim3(PT), 0, st, s);
    hipLaunchKernelGGL(plan_count, grid, dim3(PT), 0, st, in, cand, n, s);
    if (tiles) hipLaunchKernelGGL(plan_starts<true>, dim3(1), dim3(PT), 0, st, s, n, next, lists, *tiles);
    else hipLaunchKernelGGL(plan_starts<false>, dim3(1), dim3(PT), 0, st, s, n, next, lists, PlanTiles{});
    hipLaunchKernelGGL(plan_scatter, grid, dim3(PT), 0, st, in, cand, n, next, lists, perm, cand_tile,
                       rest, bytes);
    return hipGetLastError();
}

}  // namespace srm
