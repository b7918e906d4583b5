// filter_gpu.hip -- the q-gram filter ("SEASHORE") on the GPU.
//
// Same candidates, flags, perfect hits and batch boundaries as the host filter
// (filter.cpp); only the per-read work moves to the device:
//   0. pack    the reads' bytes as 2-bit codes and a mask of other bytes;
//   1. count   a lane per q-gram list looks it up in the device copy of the q-gram
//              index and writes the list length + 1 and the index of the list's
//              first key;
//   2. sum     of the lengths = the offset of every 0-terminated list in one flat
//              array, reads in order (the reference's data_array,
//              hash.c:396-461, for all chunks at once): a scan, or for small calls
//              the blocks' sums;
//   3. fill    the same threads write the lists: a copy of the key run the
//              count found, or the hash-table lookup again for a q-gram
//              holding a byte other than ACGT;
//   4. pair    a group of lanes per read runs run_seashore (hash.c:502-834) and
//              add_start_position (hash.c:40-178) over the flat array.  A list
//              index beyond the list runs on into the following lists and the
//              following reads' lists up to the end of the read's chunk of
//              chunk_value reads (Q12), exactly as a walk of data_array does.
//              The read's result-hash entries live in LDS (16 entries, 4 perfect
//              hits per read) and go to places of its own; a read that needs
//              more is marked and run again with slots in HBM (1024, then
//              65534 entries);
//   5. batch   the sequential batch pass (Q10 leak, flush boundaries) in parallel:
//              counts per read, their sum, candidates and perfect hits in read
//              order in one block for the host, which settles the few reads
//              whose outcome depends on others (filter_batch.h).
// blockIdx.y is the strand: a call of both runs each kernel once.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <array>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "alloc.h"
#include "filter_batch.h"
#include "filter_internal.h"
#include "filter_pair.h"
#include "nw_device.h"

using namespace srm_filter_impl;
using namespace srm_pair;
using namespace srm_batch;

namespace {

constexpr int FB = 256;      // threads per block
constexpr int ECAP = 16;     // result-hash entries per read kept in LDS
constexpr int PCAP = 4;      // perfect hits per read kept in LDS
constexpr int PB = 64;       // threads per block of the pairing pass (one wave: pair_list)
// reads per block of it with G lanes a read: half as many again as it takes at a time,
// since about half are dropped; one each where a read may take long
constexpr int pair_reads(int G) { return G == 8 ? PB / G * 3 / 2 : PB / G; }
constexpr int NSTARTS = 33;  // list starts per read kept in LDS (odd: the groups of a
constexpr int NVALS = 64;    // wave read from different banks), and list elements

// the reads' (or the genome's) bytes as codes and as a mask of other bytes: 16 bytes
// a thread; src holds n16 * 16 readable bytes
__global__ void __launch_bounds__(FB) fl_pack(const uint4 *__restrict__ src, uint32_t *__restrict__ pk,
                                              uint16_t *__restrict__ odd, size_t n16)
{
    const size_t i = (size_t)blockIdx.x * FB + threadIdx.x;
    if (i >= n16) return;
    const uint4 v = src[i];
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    uint32_t o;
    pk[i] = pack16(w, o);
    odd[i] = (uint16_t)o;
}

// A small call's inputs from page-locked host memory to dst, and the reads among them
// (from 16-byte word `first` on) packed as by fl_pack: a copy before it takes 9 us for
// 160 KB and starts and ends with a wait of 13
__global__ void __launch_bounds__(FB) fl_take(const uint4 *__restrict__ src, uint4 *__restrict__ dst,
                                              size_t first, uint32_t *__restrict__ pk,
                                              uint16_t *__restrict__ odd, size_t n16)
{
    const size_t i = (size_t)blockIdx.x * FB + threadIdx.x;
    if (i >= n16) return;
    const uint4 v = src[i];
    dst[i] = v;
    if (i < first) return;
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    uint32_t o;
    pk[i - first] = pack16(w, o);
    odd[i - first] = (uint16_t)o;
}

constexpr size_t OVER_ROOM = (size_t)1 << 19;   // entries
// The reads' codes as the alignment kernels take them (16 per word, the first lowest, other
// bytes 0), `pad` codes of zero before them, every read's reverse complement after them:
// a thread per word.  The reads lie one after another from byte 0, `total` in all; off: n.
//
// HBM-bound and small beside the lookups (7 MB of reads: 12 us); on the host a request's
// reverse complements and packing took 1 ms of 7 MB, 0.2 ms of 140 KB.
__global__ void __launch_bounds__(FB) fl_read_words(const uint32_t *__restrict__ pk,
                                                    const uint16_t *__restrict__ odd,
                                                    const uint64_t *__restrict__ off, uint32_t n,
                                                    uint64_t total, uint32_t pad, uint32_t *__restrict__ out,
                                                    size_t n_words)
{
    const size_t w = (size_t)blockIdx.x * FB + threadIdx.x;
    if (w >= n_words) return;
    const int64_t p = (int64_t)(16 * w) - (int64_t)pad;   // the word's first code
    uint32_t v = 0;
    uint32_t r = 0;      // the read of the reverse complements' code at hand
    uint64_t lo = 0, hi = 0;
    for (int j = 0; j < 16; ++j) {
        const int64_t c = p + j;
        if (c < 0 || (uint64_t)c >= 2 * total) continue;
        uint64_t at = (uint64_t)c;
        const bool rev = at >= total;
        if (rev) {
            at -= total;
            if (at >= hi) {
                if (hi == 0) {   // the last read that starts at or before it
                    uint32_t b = 0;
                    for (uint32_t m = n; m > 1;) {
                        const uint32_t h = m >> 1;
                        if (off[b + h] <= at) b += h;
                        m -= h;
                    }
                    r = b;
                } else {
                    ++r;         // (no read is empty)
                }
                lo = off[r];
                hi = r + 1 < n ? off[r + 1] : total;
            }
            at = lo + hi - 1 - at;
        }
        const uint32_t code = (pk[at >> 4] >> (30 - 2 * (int)(at & 15))) & 3u;
        if ((odd[at >> 4] >> (at & 15)) & 1u) continue;
        v |= (rev ? 3u - code : code) << (2 * j);
    }
    out[w] = v;
}

constexpr uint32_t MAX_FLUSH = 256;      // flushes the device lists
constexpr uint32_t MAX_UNSAFE = 1 << 16; // reads it lists for the host's walk
constexpr uint32_t MAX_WALK = 1 << 16;   // words of their entries

// one strand's counters and flushes
struct Header {
    uint32_t counters[3];    // entries, perfect hits, reads that outgrew their slots
    uint32_t n_unsafe, walk_words;
    uint32_t n_flush;        // MAX_FLUSH + 1: more
    uint32_t flat;           // list entries (terminators included; TOO_MANY)
    uint32_t blob_ok;        // the output fitted
    Counts total;
    Flush flush[MAX_FLUSH];
};

static_assert(sizeof(Header) % 16 == 0, "the output behind it is read 16 bytes at a time");

struct Strand {
    FArgs f;
    Header *hdr;
    uint64_t flat_cap;       // entries that flat holds, MAX_FLAT at most
    Counts *cnt, *start;     // [n_reads + 1] per read; summed over the reads before
    uint32_t *list_sum;      // small calls: the sums of fl_count's and fl_batch_count's
    Counts *cnt_sum;         // blocks
    uint32_t *by_rank;       // the reads with entries
    uint32_t *unsafe;        // read | leaky << 31
    uint32_t *walk;
};

// one call's strands, in the order the kernels' blockIdx.y takes them
struct Call {
    Strand s[2];
    int n;
    uint64_t n_lists;        // per strand
    bool sums;               // block sums in place of scans (SUM_READS)
    uint64_t list_stride;    // words from a strand's list arrays to the other's
    int kmax;
    const uint8_t *blocked;
    unsigned char *blob;     // the strands' candidates and perfect hits, arrays packed
    uint64_t blob_cap;
    unsigned char *back;     // page-locked host memory for the headers and, if it fits
    uint64_t back_cap;       // back_cap bytes, the blob
};

// the total in place of one that 32 bits do not hold: no room has as much
constexpr uint32_t TOO_MANY = ~0u;
static_assert(TOO_MANY > MAX_FLAT, "");

// a strand's arguments; false when its lists do not fit (the host makes room and
// runs the call again, or refuses it)
__device__ __forceinline__ bool strand_of(const Call &c, FArgs &a)
{
    const Strand &s = c.s[blockIdx.y];
    a = s.f;
    a.list_org = a.list_start[0];
    return (uint64_t)list_at(a, c.n_lists) <= s.flat_cap;
}

// One thread per q-gram list; a block takes the lists of `per` consecutive reads,
// whose offsets, lengths and first lists it holds in LDS.
//
// Bound by HBM lines: a lookup reads a prefix-table line and, when the prefix
// occurs, a line of keys, both at random.  A thread per read (walking the read's
// lists in turn, a byte load per base) fetched ten lines per lookup: neighbouring
// lanes' read bytes and list words lie hundreds of bytes apart.  A lane per list
// has neighbours on the same read, stores its list words side by side and takes the
// q-gram from three packed words.  2M reads of 50-250 bp (36M lists), one strand:
// 7.10 -> 1.46 ms, the fill 1.98 -> 0.37 ms; 1,000 reads, where a read took its
// lookups one after another: 262 -> 6 us.
constexpr int CREADS = 64;

// the block's reads in LDS, and the read a list of the block belongs to
struct BlockReads {
    uint32_t base[CREADS + 1];
    uint64_t off[CREADS];
    int L[CREADS], q[CREADS];
    __device__ uint32_t load(const FArgs &a, uint32_t per, uint32_t lo, uint32_t hi)
    {
        const uint32_t r0 = lo + blockIdx.x * per;
        const uint32_t nr = hi - r0 < per ? hi - r0 : per;
        for (uint32_t t = threadIdx.x; t <= nr; t += FB) {
            base[t] = a.list_base[r0 + t];
            if (t < nr) {
                const DParam P = a.par[a.pid[r0 + t]];
                off[t] = a.roff[r0 + t];
                L[t] = P.L;
                q[t] = P.q;
            }
        }
        __syncthreads();
        return nr;
    }
    __device__ uint32_t read_of(uint32_t i, uint32_t nr) const
    {
        uint32_t t = 0;
        while (nr > 1) {
            const uint32_t h = nr >> 1;
            if (base[t + h] <= i) t += h;
            nr -= h;
        }
        return t;
    }
};

// list i of the block: its length with the terminator, which it writes with the first key
__device__ __forceinline__ uint32_t count_list(const FArgs &a, const BlockReads &s, uint32_t nr, uint32_t i)
{
    const uint32_t t = s.read_of(i, nr);
    const int L = s.L[t], q = s.q[t], g = gram_offset(L, q, (int)(i - s.base[t]));
    const DQ X = a.qix[q];
    uint64_t code;
    uint32_t first, c;
    if (gram_code(a.read_pk, a.read_odd, s.off[t], L, a.dr, q, g, code))
        c = lookup_code(X, code, first);
    else
        c = lookup<false>(X, a.genome, a.reads + s.off[t], L, a.dr, g, nullptr, &first);
    a.list_cnt[i] = c + 1;
    a.list_lo[i] = first;
    return c + 1;
}

// Sums over a block's threads, and over the blocks of a small call.  Up to SUM_READS reads
// a kernel adds up its own blocks' parts and the next one adds the blocks before: a scan
// kernel and its start-up between them cost 8 us and two launches, as much as the work of
// 1,000 reads on either side (its whole call 142 -> 132 us).  Beyond, every block of
// hundreds would read every block's sum, and the scan is the smaller part.
constexpr size_t SUM_READS = 32768;
constexpr size_t SUM_BLOCKS = 1024;   // blocks of either kernel, at most

// the sum over the threads before this one; total: over all
template <int N>
__device__ __forceinline__ void block_excl(uint32_t (&v)[N], uint32_t (&total)[N])
{
    __shared__ uint32_t s[FB / 64][N];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    __syncthreads();   // the sums before have been read
#pragma unroll
    for (int e = 0; e < N; ++e) {
        uint32_t x = v[e];
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = (uint32_t)__shfl_up((int)x, d, 64);
            if (lane >= d) x += o;
        }
        if (lane == 63) s[wv][e] = x;
        v[e] = x - v[e];
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < N; ++e) {
        total[e] = 0;
#pragma unroll
        for (int w = 0; w < FB / 64; ++w) {
            if (w == wv) v[e] += total[e];
            total[e] += s[w][e];
        }
    }
}

// of `blocks` blocks' sums of N words each: the sum over those before this block, over all
template <int N>
__device__ __forceinline__ void sums_before(const uint32_t *sum, uint32_t blocks, uint32_t (&before)[N],
                                            uint32_t (&total)[N])
{
    uint32_t v[2 * N] = {}, t[2 * N];
    for (uint32_t b = threadIdx.x; b < blocks; b += FB)
#pragma unroll
        for (int e = 0; e < N; ++e) {
            const uint32_t x = sum[(size_t)b * N + e];
            v[N + e] += x;
            if (b < blockIdx.x) v[e] += x;
        }
    block_excl<2 * N>(v, t);
#pragma unroll
    for (int e = 0; e < N; ++e) {
        before[e] = t[e];
        total[e] = t[N + e];
    }
}

// the lists of reads [lo, hi); SUMS: with their starts in the block, and the block's sum
template <bool SUMS>
__global__ void __launch_bounds__(FB) fl_count(Call c_, uint32_t per, uint32_t lo, uint32_t hi)
{
    __shared__ BlockReads s;
    const FArgs &a = c_.s[blockIdx.y].f;
    if (blockIdx.x == 0 && hi == a.n_reads) {   // what later kernels of the call add to
        // (the entries and perfect hits of reads that are run again follow all slots')
        if (threadIdx.x < 6)
            ((uint32_t *)c_.s[blockIdx.y].hdr)[threadIdx.x] =
                threadIdx.x > 1 || a.packed ? 0 : threadIdx.x == 0 ? a.n_reads * ECAP : a.n_reads * PCAP;
        if (threadIdx.x == 0) {
            a.list_cnt[c_.n_lists] = 0;
            if (SUMS) ((uint32_t *)a.list_start)[c_.n_lists] = 0;   // (fl_fill's maximum)
        }
    }
    const uint32_t nr = s.load(a, per, lo, hi);
    uint32_t carry = 0;
    for (uint32_t i0 = s.base[0]; i0 < s.base[nr]; i0 += FB) {
        const uint32_t i = i0 + threadIdx.x;
        const bool in = i < s.base[nr];
        uint32_t len[1] = {0}, all[1];
        if (in) len[0] = count_list(a, s, nr, i);
        if (!SUMS) continue;
        block_excl<1>(len, all);
        if (in) ((uint32_t *)a.list_start)[i] = carry + len[0];
        carry += all[0];
    }
    if (SUMS && threadIdx.x == 0) c_.s[blockIdx.y].list_sum[blockIdx.x] = carry;
}
// the lists themselves, blocks and threads as in fl_count: the positions are the
// keys it found, or, for a q-gram holding another byte, the hash table's
template <bool SUMS>
__global__ void __launch_bounds__(FB) fl_fill(Call c_, uint32_t per)
{
    __shared__ BlockReads s;
    FArgs a;
    uint32_t before[1] = {0}, total[1];
    bool fits = true;
    const Strand &st = c_.s[blockIdx.y];
    if (SUMS) {
        a = st.f;
        a.list_org = 0;
        sums_before<1>(st.list_sum, gridDim.x, before, total);
        fits = total[0] <= st.flat_cap;
        if (threadIdx.x == 0 && blockIdx.x == gridDim.x - 1)
            atomicMax((uint32_t *)a.list_start + c_.n_lists, total[0]);
    } else if (!strand_of(c_, a)) {
        return;
    }
    const uint32_t nr = s.load(a, per, 0, a.n_reads);
    for (uint32_t i = s.base[0] + threadIdx.x; i < s.base[nr]; i += FB) {
        const uint32_t c = a.list_cnt[i] - 1, at = list_at(a, i) + before[0];
        if (SUMS) ((uint32_t *)a.list_start)[i] = at;
        if (!fits) continue;
        if (!list_fits(at, c + 1, st.flat_cap)) {
            if (SUMS) atomicMax((uint32_t *)a.list_start + c_.n_lists, TOO_MANY);
            else ((uint32_t *)a.list_start)[c_.n_lists] = a.list_org + TOO_MANY;
            continue;
        }
        uint32_t *dst = a.flat + at;
        if (c) {
            const uint32_t lo = a.list_lo[i], t = s.read_of(i, nr);
            const int q = s.q[t];
            const DQ X = a.qix[q];
            if (lo != NO_RANGE) {
                const uint64_t mask = ((uint64_t)1 << X.pos_bits) - 1;
                for (uint32_t x = 0; x < c; ++x) dst[x] = (uint32_t)(X.keys[lo + x] & mask);
            } else {
                lookup<true>(X, a.genome, a.reads + s.off[t], s.L[t], a.dr,
                             gram_offset(s.L[t], q, (int)(i - s.base[t])), dst);
            }
        }
        dst[c] = 0;
    }
}

// one lane's stores to its read's slots before the group's later loads of them
template <bool GLOBAL>
__device__ __forceinline__ void slots_written()
{
    if (GLOBAL) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// add_start by a group's G lanes alike (gl: this lane's place, gb: the group's first
// lane in the wave): the entries in steps of G, the first one that decides decides
template <int G, bool GLOBAL>
__device__ __forceinline__ int group_add(Store &s, int32_t pos, int flag, int k, int gl, int gb)
{
    constexpr uint64_t GM = G == 64 ? ~0ull : (1ull << (G & 63)) - 1;
    for (uint32_t e0 = 0; e0 < s.n; e0 += G) {
        const uint32_t e = e0 + (uint32_t)gl;
        const int rule = e < s.n ? entry_rule(s.P(e), s.F(e), pos, flag, k) : 0;
        const uint64_t m = (__ballot(rule != 0) >> gb) & GM;
        if (m) {
            const int first = (int)__builtin_ctzll(m);
            const int decided = __shfl(rule, gb + first, 64);
            if (decided == 2 && gl == first) s.F(e) = (int8_t)flag;
            slots_written<GLOBAL>();
            return decided;
        }
    }
    if (s.n == s.cap) {
        s.ovf = true;
        return 2;
    }
    if (gl == 0) {
        s.P(s.n) = pos;
        s.F(s.n) = (int8_t)flag;
    }
    slots_written<GLOBAL>();
    ++s.n;
    return 2;
}

// a read of the pairing pass: what its loads depend on, found for all of a block's reads
// at once
struct PairRead {
    uint64_t off;            // its first byte
    uint32_t r, at;          // the read, its place among the launch's
    uint32_t lb, n;          // its first list, its lists
    uint32_t i0, i1, end;    // flat indices: its first list, its second half, its end
    uint32_t flat_end;
    uint32_t pid;
};

// the reads of a block (`per` <= PB) that have a position to start from; nothing comes of
// the others, half of the reads on either strand
__device__ __forceinline__ uint32_t pair_list(const FArgs &a, PairRead *list, uint32_t per)
{
    const uint32_t at = blockIdx.x * per + threadIdx.x;
    PairRead R;
    bool some = false;
    if (threadIdx.x < per && at < a.n_todo) {
        R.at = at;
        R.r = a.todo ? a.todo[at] : at;
        R.lb = a.list_base[R.r];
        R.off = a.roff[R.r];
        R.pid = a.pid[R.r];
        R.flat_end = chunk_end(a, R.r);
        const uint32_t half = (uint32_t)a.par[R.pid].half;
        R.n = (uint32_t)a.par[R.pid].n;
        R.i0 = list_at(a, R.lb);
        R.i1 = list_at(a, R.lb + half);
        R.end = list_at(a, R.lb + R.n);
        some = R.i1 - R.i0 != half;   // (an empty list is its terminator)
        if (!some) {
            a.meta[3 * (size_t)R.r + 0] = 0;
            a.meta[3 * (size_t)R.r + 1] = 0;
            a.meta[3 * (size_t)R.r + 2] = 0;
        }
    }
    const uint64_t m = __ballot(some);
    if (some) list[__popcll(m & ((1ull << threadIdx.x) - 1))] = R;
    __syncthreads();
    return (uint32_t)__popcll(m);
}

// run_seashore (hash.c:502-834) by G lanes per read: each lane takes a start
// position (an element of the first half of the read's lists, which lie one after
// another in the flat array) and finds what it would insert -- that depends on the
// lists alone -- and the group then adds the results in the reference's order.
//
// Latency-bound: a start position is a chain of dependent list loads and the perfect
// check.  With the lists in HBM a wave waited 100 times in turn, and where a block's
// waves had to meet for one reservation of output, all waited for the slowest.  So a
// read's lists come to LDS in one step, its loads' addresses are found for all of a
// block's reads at once (without those that nothing comes of), starts that fail at
// the read's ends are dropped before the group's compare, a start is added once, the
// slots' entries have places of their own, and a block is one wave.  Both strands: 2M
// reads of 50-250 bp 4.78 -> 2.60 ms, 100,000 of 36 bp 162 -> 79 us, 1,000 of
// 36-250 bp 46 -> 22 us (by a thread per read: 21 ms, 1.7 ms for the 1,000).
template <int G, bool GLOBAL>
__global__ void __launch_bounds__(PB) fl_pair(Call c_)
{
    FArgs a;
    if (!strand_of(c_, a)) return;
    constexpr int NG = PB / G, LIST = pair_reads(G);   // reads at a time, reads in all
    constexpr uint64_t GM = G == 64 ? ~0ull : (1ull << (G & 63)) - 1;
    __shared__ int32_t s_pos[GLOBAL ? 1 : ECAP * NG];
    __shared__ int8_t s_flag[GLOBAL ? 1 : ECAP * NG];
    __shared__ int32_t s_perf[GLOBAL ? 1 : PCAP * NG];
    __shared__ uint32_t s_starts[NG][NSTARTS], s_vals[NG][NVALS + 1];
    __shared__ PairRead s_list[LIST];
    const int gl = threadIdx.x & (G - 1);
    const int gb = threadIdx.x & 63 & ~(G - 1);
    const uint32_t slot = threadIdx.x / G;
    const uint32_t n_list = pair_list(a, s_list, (uint32_t)LIST);
    for (uint32_t j = slot; j < n_list; j += NG) {
        const PairRead R = s_list[j];
        const uint32_t r = R.r;
        Store s;
        if (GLOBAL) {
            s.pos = a.slot_pos + (size_t)R.at * a.cap;
            s.flag = a.slot_flag + (size_t)R.at * a.cap;
            s.perf = a.slot_perf + (size_t)R.at * a.pcap;
            s.stride = 1;
            s.cap = a.cap;
            s.pcap = a.pcap;
        } else {
            s.pos = s_pos + slot;
            s.flag = s_flag + slot;
            s.perf = s_perf + slot;
            s.stride = NG;
            s.cap = ECAP;
            s.pcap = PCAP;
        }
        const DParam P = a.par[R.pid];
        const uint32_t n_starts = R.n < NSTARTS ? R.n + 1 : NSTARTS;
        const uint32_t n_vals = R.end - R.i0 < NVALS ? R.end - R.i0 : NVALS;
        for (uint32_t x = gl; x < n_starts; x += G) s_starts[slot][x] = list_at(a, R.lb + x);
#pragma unroll 4
        for (uint32_t x = gl; x < n_vals; x += G) s_vals[slot][x] = a.flat[R.i0 + x];
        slots_written<false>();
        const ReadLists ls{a, R.lb, s_starts[slot], n_starts, s_vals[slot], R.i0, n_vals};
        const uint64_t at = R.off;
        for (uint32_t p0 = R.i0; p0 < R.i1 && !s.ovf; p0 += G) {
            const uint32_t p = p0 + (uint32_t)gl;
            const uint32_t Pa = p < R.i1 ? ls.val(p) : 0u;
            int aa = 0;
            uint32_t off = 0;
            bool valid = Pa != 0;
            if (valid) {
                for (int n = P.half; n > 1;) {   // the list holding p
                    const int h = n >> 1;
                    if (ls.start(aa + h) <= p) aa += h;
                    n -= h;
                }
                const uint32_t first = ls.start(aa);
                off = p - first;
                // a list that starts with offset 0 reads as empty (Q14)
                valid = off == 0 || ls.val(first) != 0;
            }
            const int64_t gs = (int64_t)Pa - ((int64_t)aa * P.q + 1);
            valid = valid && gs + 1 > 0;
            const uint32_t S = (uint32_t)(gs + 1);
            // perfect check (strncpy + strcmp, hash.c:550-583), each genome start once, the
            // group's lanes 16 bases each.  Most starts of a chance hit fail at the read's
            // ends, which each lane looks at for its own: the starts of the loop below wait
            // for memory one after another
            const bool check = valid && (uint64_t)S + (uint64_t)P.L <= a.glen &&
                               (same16(a, at, P.L, a.dr, S, 0) &
                                same16(a, at, P.L, a.dr, S, (P.L - 1) >> 4));
            bool perfect = false;
            uint64_t todo = (__ballot(check) >> gb) & GM;
            while (todo) {
                const uint32_t S0 = (uint32_t)__shfl((int)S, gb + (int)__builtin_ctzll(todo), 64);
                bool ok = true;
                for (int x = gl + 1; 16 * x < P.L && ok; x += G) ok = same16(a, at, P.L, a.dr, S0, x);
                const bool all = ((__ballot(!ok) >> gb) & GM) == 0;
                const bool mine = check && S == S0;
                if (mine) perfect = all;
                todo &= ~((__ballot(mine) >> gb) & GM);
            }
            int32_t hpos = 0;
            int hflag = 0;
            const bool found = valid && pair_matches(ls, P, R.flat_end, aa, off, Pa, gs, hpos, hflag);
            const int what = (perfect ? 1 : 0) | (found ? 2 : 0) | (hflag << 2);
            uint64_t add = (__ballot((what & 3) != 0) >> gb) & GM;
            while (add && !s.ovf) {
                const int src = gb + (int)__builtin_ctzll(add);
                const int w = __shfl(what, src, 64);
                const uint32_t S0 = (uint32_t)__shfl((int)S, src, 64);
                const int32_t hpos0 = __shfl(hpos, src, 64);
                if (w & 1) {
                    if (group_add<G, GLOBAL>(s, -(int32_t)S0, 0, P.k, gl, gb) != 1 && !s.ovf) {
                        if (s.np == s.pcap) {
                            s.ovf = true;
                        } else {
                            if (gl == 0) s.Q(s.np) = (int32_t)S0;
                            ++s.np;
                        }
                    }
                }
                if ((w & 2) && !s.ovf) group_add<G, GLOBAL>(s, hpos0, w >> 2, P.k, gl, gb);
                // a start added again is rejected: its entry, or the one that rejected it,
                // still decides (an entry's flag is only ever lowered)
                add &= ~((__ballot(what == w && S == S0 && hpos == hpos0) >> gb) & GM);
            }
        }
        // the group's first lane speaks for its read.  The slots' entries go to the read's
        // own places; those of a read run again follow them all
        if (gl == 0) {
            const uint32_t ne = s.ovf ? 0 : s.n, np = s.ovf ? 0 : s.np;
            const uint32_t be = !GLOBAL && !a.packed ? r * ECAP : ne ? atomicAdd(&a.counters[0], ne) : 0;
            const uint32_t bp = !GLOBAL && !a.packed ? r * PCAP : np ? atomicAdd(&a.counters[1], np) : 0;
            for (uint32_t e = 0; e < ne; ++e) {
                a.out_pos[be + e] = s.P(e);
                a.out_flag[be + e] = s.F(e);
            }
            for (uint32_t e = 0; e < np; ++e) a.out_perf[bp + e] = s.Q(e);
            a.meta[3 * (size_t)r + 0] = be;
            a.meta[3 * (size_t)r + 1] = bp;
            a.meta[3 * (size_t)r + 2] = s.ovf ? OVERFLOW_MARK : (ne | (np << 16));
            if (s.ovf) a.over[atomicAdd(&a.counters[2], 1u)] = r;
        }
        slots_written<GLOBAL>();   // before the next read's
    }
}

__device__ __forceinline__ Counts counts_of(const uint32_t (&v)[4])
{
    Counts n;
    n.cand = v[0];
    n.perf = v[1];
    n.queued = v[2];
    n.with = v[3];
    return n;
}

// ---- the batch pass (filter_batch.h), a thread per read: counts, and after their
// sum the candidates and perfect hits at their places in read order.  HBM-bound
// (12 bytes of meta per read, 5 per entry, 15 out per candidate); the host's pass
// over the same data and its download took 80 of the 96 ms of a call of 2M reads.
// With both strands in each launch and two waits in a call (one, while the output fits
// the first copy) instead of eight, the whole call: 2M reads 96.2 -> 20.8 ms, 100,000 of
// 36 bp 3.14 -> 0.74 ms, 1,000 0.47 -> 0.22 ms
template <bool SUMS>
__global__ void __launch_bounds__(FB) fl_batch_count(Call c)
{
    FArgs a;
    if (!strand_of(c, a)) return;
    const Strand &s = c.s[blockIdx.y];
    const uint32_t r = blockIdx.x * FB + threadIdx.x;
    if (!SUMS && r > a.n_reads) return;
    Counts n;
    if (r < a.n_reads) {
        const uint32_t m0 = a.meta[3 * (size_t)r], m2 = a.meta[3 * (size_t)r + 2];
        const DParam P = a.par[a.pid[r]];
        bool unsafe, leaky;
        n = count_entries(a.out_pos + m0, a.out_flag + m0, entries_of(m2), P.L, P.k, c.kmax, a.glen,
                          c.blocked, unsafe, leaky);
        n.perf = perfects_of(m2);
        if (unsafe) {
            const uint32_t u = atomicAdd(&s.hdr->n_unsafe, 1u);
            if (u < MAX_UNSAFE) s.unsafe[u] = r | (leaky ? 1u << 31 : 0u);
        }
    }
    if (!SUMS) {
        s.cnt[r] = n;
        return;
    }
    uint32_t v[4] = {n.cand, n.perf, n.queued, n.with}, all[4];
    block_excl<4>(v, all);
    if (r <= a.n_reads) s.start[r] = counts_of(v);
    if (threadIdx.x == 0) s.cnt_sum[blockIdx.x] = counts_of(all);
}

// the sum over a strand's reads before r
__device__ __forceinline__ Counts counts_before(const Strand &s, uint32_t r)
{
    const Counts x = s.start[r], o = s.start[0];
    Counts n;
    n.cand = x.cand - o.cand;
    n.perf = x.perf - o.perf;
    n.queued = x.queued - o.queued;
    n.with = x.with - o.with;
    return n;
}

// the byte offsets of the strands' arrays in the blob, widest elements first
struct BlobAt {
    uint64_t c_pos[2], p_pos[2], c_read[2], p_read[2], c_w[2], c_flag[2], bytes;
};

__host__ __device__ inline BlobAt blob_at(const Counts &t0, const Counts &t1)
{
    const uint64_t c[2] = {t0.cand, t1.cand}, p[2] = {t0.perf, t1.perf};
    BlobAt b;
    uint64_t at = 0;
    for (int s = 0; s < 2; ++s) {
        b.c_pos[s] = at;
        b.p_pos[s] = b.c_pos[s] + 8 * c[s];
        at = b.p_pos[s] + 8 * p[s];
    }
    for (int s = 0; s < 2; ++s) {
        b.c_read[s] = at;
        b.p_read[s] = b.c_read[s] + 4 * c[s];
        at = b.p_read[s] + 4 * p[s];
    }
    for (int s = 0; s < 2; ++s) {
        b.c_w[s] = at;
        at += 2 * c[s];
    }
    for (int s = 0; s < 2; ++s) {
        b.c_flag[s] = at;
        at += c[s];
    }
    b.bytes = at;
    return b;
}

template <bool SUMS>
__global__ void __launch_bounds__(FB) fl_batch_write(Call c)
{
    FArgs a;
    if (!strand_of(c, a)) return;
    const int y = blockIdx.y;
    const Strand &s = c.s[y];
    const uint32_t r = blockIdx.x * FB + threadIdx.x;
    Counts total[2], at;
    if (SUMS) {   // the other strand's sums are there too: it counted in the same launch
        uint32_t before[4] = {}, x[4], all[4];
        for (int z = 0; z < c.n; ++z) {
            sums_before<4>((const uint32_t *)c.s[z].cnt_sum, gridDim.x, x, all);
            total[z] = counts_of(all);
            if (z == y)
                for (int e = 0; e < 4; ++e) before[e] = x[e];
        }
        if (r <= a.n_reads) {
            at = CountsSum()(s.start[r], counts_of(before));
            s.start[r] = at;
        }
    } else {
        total[0] = counts_before(c.s[0], a.n_reads);
        if (c.n > 1) total[1] = counts_before(c.s[1], a.n_reads);
        if (r < a.n_reads) at = counts_before(s, r);
    }
    const BlobAt b = blob_at(total[0], total[1]);
    const bool fits = b.bytes <= c.blob_cap;
    if (r == 0) s.hdr->blob_ok = fits;
    if (r >= a.n_reads) return;
    const uint32_t m0 = a.meta[3 * (size_t)r], m1 = a.meta[3 * (size_t)r + 1], m2 = a.meta[3 * (size_t)r + 2];
    const uint32_t ne = entries_of(m2), np = perfects_of(m2);
    if (ne) s.by_rank[at.with] = r;
    if (!fits) return;
    const DParam P = a.par[a.pid[r]];
    int64_t *c_pos = (int64_t *)(c.blob + (y ? b.c_pos[1] : b.c_pos[0])), *p_pos = (int64_t *)(c.blob + (y ? b.p_pos[1] : b.p_pos[0]));
    int32_t *c_read = (int32_t *)(c.blob + (y ? b.c_read[1] : b.c_read[0])), *p_read = (int32_t *)(c.blob + (y ? b.p_read[1] : b.p_read[0]));
    uint16_t *c_w = (uint16_t *)(c.blob + (y ? b.c_w[1] : b.c_w[0]));
    uint8_t *c_flag = c.blob + (y ? b.c_flag[1] : b.c_flag[0]);
    uint32_t o = at.cand;
    for (uint32_t e = 0; e < ne; ++e) {
        const int32_t pos = a.out_pos[m0 + e];
        const int flag = a.out_flag[m0 + e];
        const int64_t w = own_window(P.L, flag, P.k);
        if (pos <= 0 || outside(c.blocked, a.glen, pos, w)) continue;
        c_pos[o] = pos;
        c_read[o] = (int32_t)r;
        c_w[o] = (uint16_t)w;
        c_flag[o] = (uint8_t)flag;
        ++o;
    }
    for (uint32_t e = 0; e < np; ++e) {
        p_pos[at.perf + e] = a.out_perf[m1 + e];
        p_read[at.perf + e] = (int32_t)r;
    }
}

// where fl_batch_end does not run: the lists' total
__global__ void fl_totals(Call c)
{
    FArgs a;
    (void)strand_of(c, a);
    if (threadIdx.x == 0) c.s[blockIdx.y].hdr->flat = list_at(a, c.n_lists);
}

// the strand's header and its share of the output to the host (by one block per strand),
// as the call's last stores: a copy in their place would wait 13 us for this kernel's end
// and take 7 more
__device__ __forceinline__ void send_back(const Call &c, uint64_t bytes)
{
    __threadfence();
    __syncthreads();
    const uint32_t y = blockIdx.y;
    const auto *h = (const uint32_t *)c.s[y].hdr;
    auto *to = (uint32_t *)(c.back + y * sizeof(Header));
    // (the atomics' words among them do not pass this CU's cache)
    for (uint32_t i = threadIdx.x; i < sizeof(Header) / 4; i += FB)
        to[i] = __hip_atomic_load(h + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (bytes > c.back_cap) return;
    const auto *b = (const uint4 *)c.blob;
    auto *out = (uint4 *)(c.back + c.n * sizeof(Header));
    const uint64_t n16 = (bytes + 15) / 16;
    for (uint64_t i = (uint64_t)threadIdx.x * c.n + y; i < n16; i += (uint64_t)FB * c.n) out[i] = b[i];
}

// one block per strand: the flushes (a flush ends with the first read that takes the
// queue past chunk_value; found by a wave's 64-way search of the queued sums), and
// the entries of the reads the host walks
__global__ void __launch_bounds__(FB) fl_batch_end(Call c)
{
    FArgs a;
    if (!strand_of(c, a)) {
        if (threadIdx.x == 0) c.s[blockIdx.y].hdr->flat = list_at(a, c.n_lists);
        send_back(c, ~0ull);
        return;
    }
    const Strand &s = c.s[blockIdx.y];
    const uint32_t n = a.n_reads;
    const Counts total = counts_before(s, n);
    if (threadIdx.x < 64) {
        const uint32_t lane = threadIdx.x;
        uint32_t lo = 0, nf = 0;
        for (;;) {
            const uint32_t q0 = counts_before(s, lo).queued;
            uint32_t x = lo, y = n;          // the read is in [x, y], n: none
            while (x < y) {
                const uint32_t step = (y - x + 63) / 64;
                const uint64_t e = (uint64_t)x + (uint64_t)(lane + 1) * step;
                const uint32_t r = (uint32_t)(e < y ? e : y) - 1;
                const uint64_t m = __ballot(counts_before(s, r + 1).queued - q0 > a.cv);
                if (m == 0) {
                    x = y;
                    break;
                }
                const uint32_t f = (uint32_t)__builtin_ctzll(m);
                y = (uint32_t)__shfl((int)r, (int)f, 64);
                x += f * step;
            }
            const bool last = x >= n;
            if (last && total.queued == q0) break;
            if (nf == MAX_FLUSH) {
                nf = MAX_FLUSH + 1;
                break;
            }
            lo = last ? n : x + 1;
            if (lane == 0) s.hdr->flush[nf] = {lo, counts_before(s, lo).cand};
            ++nf;
            if (last) break;
        }
        if (lane == 0) {
            s.hdr->n_flush = nf;
            s.hdr->flat = list_at(a, c.n_lists);
            s.hdr->total = total;
        }
    }
    auto put = [&](uint32_t r) {
        const uint32_t m0 = a.meta[3 * (size_t)r], ne = entries_of(a.meta[3 * (size_t)r + 2]);
        const Counts at = counts_before(s, r);
        if (4 + 2 * ne > MAX_WALK / 4) {   // (kept out of the sum, which must not wrap)
            atomicMax(&s.hdr->walk_words, MAX_WALK + 1);
            return;
        }
        const uint32_t w = atomicAdd(&s.hdr->walk_words, 4 + 2 * ne);
        if (w + 4 + 2 * ne > MAX_WALK) return;
        s.walk[w] = r;
        s.walk[w + 1] = at.with;
        s.walk[w + 2] = at.cand;
        s.walk[w + 3] = ne;
        for (uint32_t e = 0; e < ne; ++e) {
            s.walk[w + 4 + e] = (uint32_t)a.out_pos[m0 + e];
            s.walk[w + 4 + ne + e] = (uint32_t)(int32_t)a.out_flag[m0 + e];
        }
    };
    const uint32_t nu = s.hdr->n_unsafe < MAX_UNSAFE ? s.hdr->n_unsafe : MAX_UNSAFE;
    for (uint32_t u = threadIdx.x; u < nu; u += FB) {
        const uint32_t r = s.unsafe[u] & 0x7FFFFFFFu;
        put(r);
        const uint32_t next = counts_before(s, r).with + 1;
        if ((s.unsafe[u] >> 31) && next < total.with) put(s.by_rank[next]);
    }
    const BlobAt b = blob_at(counts_before(c.s[0], n), c.n > 1 ? counts_before(c.s[1], n) : Counts());
    send_back(c, b.bytes <= c.blob_cap ? b.bytes : ~0ull);
}

// GBuf::ensure's SRM_ENOMEM, as which it leaves this file: a call that needs less may
// still do
constexpr int NO_ROOM = -1000;

struct GBuf {
    void *p = nullptr;
    size_t cap = 0;
    int ensure(size_t bytes)
    {
        if (bytes <= cap) return SRM_OK;
        if (p) (void)hipFree(p);
        p = nullptr;
        cap = 0;
        size_t want = (std::max(bytes, (size_t)256) + 4095) & ~(size_t)4095;
        const hipError_t e = srm::device_alloc(&p, srm::filter_alloc_fails() ? srm::NO_DEVICE_HAS : want);
        if (e != hipSuccess)
            return srm::set_error(NO_ROOM, "hipMalloc(%zu) failed: %s", want, hipGetErrorString(e));
        cap = want;
        return SRM_OK;
    }
    void release()
    {
        if (p) (void)hipFree(p);
        p = nullptr;
        cap = 0;
    }
    template <class T> T *as() const { return (T *)p; }
};

#define FL_TRY(expr)                                                                        \
    do {                                                                                    \
        hipError_t e_ = (expr);                                                             \
        if (e_ != hipSuccess)                                                               \
            return srm::set_error(SRM_EDEVICE, "%s failed: %s (%s:%d)", #expr,              \
                                  hipGetErrorString(e_), __FILE__, __LINE__);               \
    } while (0)

#define FL_RC(expr)                      \
    do {                                 \
        int rc_ = (expr);                \
        if (rc_ != SRM_OK) return rc_;   \
    } while (0)

// page-locked blocks for results: at most MAX_BLOCKS exist at a time (a caller that
// holds more results gets ordinary memory), two of them kept for the next calls.
// The results hold the pool too, so it outlives the filter for as long as they do.
class BlockPool : public std::enable_shared_from_this<BlockPool> {
public:
    ~BlockPool()
    {
        for (auto &b : kept_) (void)hipHostFree(b.p);
    }
    // `bytes` of memory, given back when the last owner lets go; null: none to be had
    std::shared_ptr<void> take(size_t bytes)
    {
        Block b;
        bool make = false;
        {
            std::lock_guard<std::mutex> lk(mu_);
            for (size_t i = 0; i < kept_.size() && !b.p; ++i)
                if (kept_[i].bytes >= bytes) {
                    b = kept_[i];
                    kept_.erase(kept_.begin() + (std::ptrdiff_t)i);
                }
            if (!b.p && !kept_.empty()) {   // too small: make room for this size
                (void)hipHostFree(kept_.back().p);
                kept_.pop_back();
                --made_;
            }
            if (!b.p && made_ < MAX_BLOCKS) {
                make = true;
                ++made_;
            }
        }
        if (make) {
            b.bytes = bytes + bytes / 4 + 4096;
            if (srm::host_alloc(&b.p, b.bytes) != hipSuccess) {
                std::lock_guard<std::mutex> lk(mu_);
                --made_;
            }
        }
        if (!b.p) {
            void *p = std::malloc(bytes);
            return p ? std::shared_ptr<void>(p, std::free) : std::shared_ptr<void>();
        }
        auto self = shared_from_this();
        return std::shared_ptr<void>(b.p, [self, b](void *) { self->give(b); });
    }

private:
    static constexpr size_t MAX_BLOCKS = 4, KEEP = 2;
    struct Block {
        void *p = nullptr;
        size_t bytes = 0;
    };
    void give(Block b)
    {
        std::lock_guard<std::mutex> lk(mu_);
        if (kept_.size() < KEEP) {
            kept_.push_back(b);
            return;
        }
        (void)hipHostFree(b.p);
        --made_;
    }
    std::mutex mu_;
    std::vector<Block> kept_;
    size_t made_ = 0;
};

// inputs up to this size are put together in page-locked memory, from which a kernel takes
// them (a copy of a few KB takes 10-30 us of calls and waits, whatever its size)
constexpr size_t STAGE_IN = (size_t)1 << 20;
// and this much of the output comes back with the headers, by the last kernel's stores:
// 1,000 reads 132 -> 115 us with both
constexpr size_t STAGE_OUT = (size_t)128 << 10;
// reads of one piece of a large upload, at most, and its plan in page-locked memory
constexpr size_t PIECE = 131072, PIECE_BYTES = (PIECE + 2) * (8 + 4 + 2);
constexpr size_t MAX_SETS = 16384;   // parameter sets (length, k) of a call in pieces

}  // namespace

struct srm_dfilter {
    srm_ctx *ctx = nullptr;
    int device = 0;
    hipStream_t st = nullptr;
    const srm_index *ix = nullptr;
    size_t glen = 0;
    GBuf genome, gen_pk, gen_odd, dq;
    std::vector<GBuf> keys, pre, odd_hash, odd_pos;
    GBuf in, read_pk, read_odd, words, sums, blocked, list_cnt, list_lo, list_start, cub_tmp, cnt, start, by_rank,
        unsafe, walk, out;
    GBuf flat[2], out_pos[2], out_flag[2], out_perf[2], meta[2], over[2][2];
    GBuf slot_pos, slot_flag, slot_perf;
    void *stage_in = nullptr, *stage_out = nullptr;   // page-locked
    std::shared_ptr<BlockPool> pool = std::make_shared<BlockPool>();
    void *stage_plan = nullptr;                       // two pieces' plans, likewise
    hipStream_t copy_st = nullptr, plan_st = nullptr; // the pieces' copies
    hipEvent_t plan_ev[2] = {nullptr, nullptr};
    hipEvent_t ev[2] = {nullptr, nullptr}, piece_ev[2] = {nullptr, nullptr}, words_ev = nullptr;
    float last_ms = 0.f;
    size_t last_lists = 0, last_flat = 0, last_overflow = 0;

    // the buffers of a call beside its inputs
    void release_strands()
    {
        for (GBuf *b : {&sums, &blocked, &list_cnt, &list_lo, &list_start, &cub_tmp, &cnt, &start, &by_rank,
                        &unsafe, &walk, &out, &slot_pos, &slot_flag, &slot_perf})
            b->release();
        for (int s = 0; s < 2; ++s)
            for (GBuf *b : {&flat[s], &out_pos[s], &out_flag[s], &out_perf[s], &meta[s], &over[s][0],
                            &over[s][1]})
                b->release();
        last_flat = last_overflow = 0;
    }

    ~srm_dfilter()
    {
        release_strands();
        for (GBuf *b : {&genome, &gen_pk, &gen_odd, &dq, &in, &read_pk, &read_odd, &words}) b->release();
        for (auto *v : {&keys, &pre, &odd_hash, &odd_pos})
            for (auto &b : *v) b.release();
        if (stage_in) (void)hipHostFree(stage_in);
        if (stage_out) (void)hipHostFree(stage_out);
        if (stage_plan) (void)hipHostFree(stage_plan);
        if (copy_st) (void)hipStreamDestroy(copy_st);
        if (plan_st) (void)hipStreamDestroy(plan_st);
        for (auto &e : plan_ev)
            if (e) (void)hipEventDestroy(e);
        for (auto &e : ev)
            if (e) (void)hipEventDestroy(e);
        for (auto &e : piece_ev)
            if (e) (void)hipEventDestroy(e);
        if (words_ev) (void)hipEventDestroy(words_ev);
    }

    int upload(GBuf &b, const void *src, size_t bytes)
    {
        FL_RC(b.ensure(bytes + 64));   // slack: whole 16-byte words are read
        if (bytes) FL_TRY(hipMemcpyAsync(b.p, src, bytes, hipMemcpyHostToDevice, st));
        return SRM_OK;
    }

    // the codes and the mask of other bytes of the bytes [from, to) at src, of which there
    // will be `bytes` (two code words and one mask word past the last are read beside them)
    int pack(const void *src, size_t bytes, GBuf &pk, GBuf &odd, size_t from, size_t to)
    {
        const size_t n16 = (bytes + 15) / 16, b = from / 16, e = (to + 15) / 16;
        FL_RC(pk.ensure((n16 + 4) * 4));
        FL_RC(odd.ensure((n16 + 4) * 2 + 4));
        if (e <= b) return SRM_OK;
        hipLaunchKernelGGL(fl_pack, dim3((unsigned)((e - b + FB - 1) / FB)), dim3(FB), 0, st,
                           (const uint4 *)src + b, pk.as<uint32_t>() + b, odd.as<uint16_t>() + b, e - b);
        FL_TRY(hipGetLastError());
        return SRM_OK;
    }
    int pack(const void *src, size_t bytes, GBuf &pk, GBuf &odd) { return pack(src, bytes, pk, odd, 0, bytes); }

    // b with room for `bytes`, its first `used` bytes kept
    int grow(GBuf &b, size_t bytes, size_t used)
    {
        if (bytes <= b.cap) return SRM_OK;
        GBuf n;
        FL_RC(n.ensure(bytes));
        hipError_t e = used ? hipMemcpyAsync(n.p, b.p, used, hipMemcpyDeviceToDevice, st) : hipSuccess;
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e != hipSuccess) {
            n.release();
            return srm::set_error(SRM_EDEVICE, "copy to a larger buffer failed: %s", hipGetErrorString(e));
        }
        b.release();
        b = n;
        return SRM_OK;
    }

    template <class T> int get(std::vector<T> &h, const GBuf &b, size_t n)
    {
        h.resize(n);
        if (n) FL_TRY(hipMemcpyAsync(h.data(), b.p, n * sizeof(T), hipMemcpyDeviceToHost, st));
        return SRM_OK;
    }
};

namespace {

// reads per block of the lookups and the fill: CREADS while that fills the chip twice
// over, fewer below
uint32_t list_reads(size_t n)
{
    return (uint32_t)std::min<size_t>(CREADS, std::max<size_t>(4, n / 512));
}

// the lookups of reads [lo, hi)
int launch_count(srm_dfilter *G, const Call &c, uint32_t lo, uint32_t hi)
{
    const uint32_t per = list_reads(hi - lo);
    const dim3 grid((hi - lo + per - 1) / per, (unsigned)c.n);
    if (c.sums) hipLaunchKernelGGL(fl_count<true>, grid, dim3(FB), 0, G->st, c, per, lo, hi);
    else hipLaunchKernelGGL(fl_count<false>, grid, dim3(FB), 0, G->st, c, per, lo, hi);
    FL_TRY(hipGetLastError());
    return SRM_OK;
}

// lists and pairing of the call's strands
int launch_search(srm_dfilter *G, const Call &c)
{
    const uint32_t n = c.s[0].f.n_reads;
    const uint64_t nl = c.n_lists;
    const uint32_t per = list_reads(n);
    const dim3 grid((n + per - 1) / per, (unsigned)c.n);
    // both strands' lengths in one sum where they lie together: the second strand's
    // offsets count from its first (list_org), modulo 2^32
    const bool one = c.list_stride == nl + 1;
    const int items = (int)((nl + 1) * (uint64_t)(one ? c.n : 1));
    for (int x = 0; x < (c.sums ? 0 : one ? 1 : c.n); ++x) {
        size_t tmp = 0;
        const uint32_t *from = c.s[x].f.list_cnt;
        uint32_t *to = G->list_start.as<uint32_t>() + (size_t)x * c.list_stride;
        FL_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, from, to, items, G->st));
        FL_RC(G->cub_tmp.ensure(tmp));
        FL_TRY(hipcub::DeviceScan::ExclusiveSum(G->cub_tmp.p, tmp, from, to, items, G->st));
    }
    if (c.sums) hipLaunchKernelGGL(fl_fill<true>, grid, dim3(FB), 0, G->st, c, per);
    else hipLaunchKernelGGL(fl_fill<false>, grid, dim3(FB), 0, G->st, c, per);
    FL_TRY(hipGetLastError());
    // lanes per read: a wave for the reads of hundreds of entries (run_overflow); 8, about
    // the start positions of a read that maps once, for many reads (2M reads, both
    // strands: 2.82 ms with 8, 3.04 with 16); 32 for the few thousand that leave the chip
    // idle either way, where one step covers a read's lists (1,000 reads, the whole
    // filter's kernels with a thread's chain of loads: 0.373 ms with 32, 0.414 with 8)
    auto pgrid = [&](uint32_t reads) { return dim3((n + reads - 1) / reads, (unsigned)c.n); };
    if (n < 4096)
        hipLaunchKernelGGL((fl_pair<32, false>), pgrid(pair_reads(32)), dim3(PB), 0, G->st, c);
    else
        hipLaunchKernelGGL((fl_pair<8, false>), pgrid(pair_reads(8)), dim3(PB), 0, G->st, c);
    FL_TRY(hipGetLastError());
    return SRM_OK;
}

int launch_batch(srm_dfilter *G, const Call &c)
{
    const uint32_t n = c.s[0].f.n_reads;
    const dim3 grid(n / FB + 1, (unsigned)c.n);
    if (c.sums) {
        hipLaunchKernelGGL(fl_batch_count<true>, grid, dim3(FB), 0, G->st, c);
        FL_TRY(hipGetLastError());
        hipLaunchKernelGGL(fl_batch_write<true>, grid, dim3(FB), 0, G->st, c);
        FL_TRY(hipGetLastError());
    } else {
        hipLaunchKernelGGL(fl_batch_count<false>, grid, dim3(FB), 0, G->st, c);
        FL_TRY(hipGetLastError());
        size_t tmp = 0;
        const int items = (int)(((uint64_t)n + 1) * (uint64_t)c.n);
        FL_TRY(hipcub::DeviceScan::ExclusiveScan(nullptr, tmp, G->cnt.as<Counts>(), G->start.as<Counts>(),
                                                 CountsSum(), Counts(), items, G->st));
        FL_RC(G->cub_tmp.ensure(tmp));
        FL_TRY(hipcub::DeviceScan::ExclusiveScan(G->cub_tmp.p, tmp, G->cnt.as<Counts>(),
                                                 G->start.as<Counts>(), CountsSum(), Counts(), items,
                                                 G->st));
        hipLaunchKernelGGL(fl_batch_write<false>, grid, dim3(FB), 0, G->st, c);
        FL_TRY(hipGetLastError());
    }
    hipLaunchKernelGGL(fl_batch_end, dim3(1, (unsigned)c.n), dim3(FB), 0, G->st, c);
    FL_TRY(hipGetLastError());
    return SRM_OK;
}

// strand x's reads that outgrew the LDS slots, run again with slots in HBM (1024, then
// 65534 entries); their entries follow the others'
int run_overflow(srm_dfilter *G, const Call &call, int x, Header &h)
{
    Call c = call;
    c.s[0] = call.s[x];
    c.n = 1;
    FArgs &a = c.s[0].f;
    int from = 0;
    uint32_t left = h.counters[2];
    // (65534: a count word of 0xFFFF | 0xFFFF << 16 would read as the overflow mark)
    for (uint32_t cap : {1024u, 65534u}) {
        if (!left) break;
        const uint32_t per = (uint32_t)std::max<size_t>(1, ((size_t)256 << 20) / ((size_t)cap * 9));
        FL_RC(G->over[x][1 - from].ensure((size_t)left * 4));
        FL_TRY(srm::launch_reset(a.counters + 2, 1, G->st));
        for (uint32_t b = 0, m; b < left; b += m) {
            // (the entries' offsets are 32 bits)
            m = (uint32_t)std::min<uint64_t>(std::min(per, left - b),
                                             (~0u - std::max(h.counters[0], h.counters[1])) / cap);
            if (m == 0) return srm::set_error(SRM_ENOMEM, "too many filter entries; split the call");
            FL_RC(G->slot_pos.ensure((size_t)m * cap * 4));
            FL_RC(G->slot_flag.ensure((size_t)m * cap));
            FL_RC(G->slot_perf.ensure((size_t)m * cap * 4));
            const size_t ne = h.counters[0], np = h.counters[1];
            FL_RC(G->grow(G->out_pos[x], (ne + (size_t)m * cap) * 4, ne * 4));
            FL_RC(G->grow(G->out_flag[x], ne + (size_t)m * cap, ne));
            FL_RC(G->grow(G->out_perf[x], (np + (size_t)m * cap) * 4, np * 4));
            a.slot_pos = G->slot_pos.as<int32_t>();
            a.slot_flag = G->slot_flag.as<int8_t>();
            a.slot_perf = G->slot_perf.as<int32_t>();
            a.out_pos = G->out_pos[x].as<int32_t>();
            a.out_flag = G->out_flag[x].as<int8_t>();
            a.out_perf = G->out_perf[x].as<int32_t>();
            a.todo = G->over[x][from].as<uint32_t>() + b;
            a.n_todo = m;
            a.over = G->over[x][1 - from].as<uint32_t>();
            a.cap = a.pcap = cap;
            const uint32_t pr = pair_reads(64);
            hipLaunchKernelGGL((fl_pair<64, true>), dim3((m + pr - 1) / pr), dim3(PB), 0, G->st, c);
            FL_TRY(hipGetLastError());
            FL_TRY(hipMemcpyAsync(h.counters, a.counters, 12, hipMemcpyDeviceToHost, G->st));
            FL_TRY(hipStreamSynchronize(G->st));
        }
        left = h.counters[2];
        from = 1 - from;
    }
    if (left) {
        uint32_t r = 0;
        FL_TRY(hipMemcpy(&r, G->over[x][from].p, 4, hipMemcpyDeviceToHost));
        return srm::set_error(SRM_ENOMEM, "read %u holds more than 65534 filter entries", r);
    }
    return SRM_OK;
}

// the buffers that the lookups write: lists of c.n strands, list_stride words each, and
// the headers with the output behind them
int ensure_lists(srm_dfilter *G, const Call &c)
{
    const size_t words = c.list_stride * (size_t)c.n, n = c.s[0].f.n_reads;
    FL_RC(G->list_cnt.ensure(words * 4));
    FL_RC(G->list_lo.ensure(words * 4));
    FL_RC(G->list_start.ensure(words * 4));
    FL_RC(G->sums.ensure(2 * SUM_BLOCKS * (4 + sizeof(Counts))));
    // candidates and perfect hits of both strands are 1-1.2 a read, 16-20 bytes each
    FL_RC(G->out.ensure(sizeof(Header) * (size_t)c.n + std::max<size_t>(STAGE_OUT, 28 * n)));
    return SRM_OK;
}

void bind_lists(const srm_dfilter *G, Call &c)
{
    for (int x = 0; x < c.n; ++x) {
        FArgs &a = c.s[x].f;
        c.s[x].hdr = G->out.as<Header>() + x;
        a.counters = c.s[x].hdr->counters;
        a.list_cnt = G->list_cnt.as<uint32_t>() + (size_t)x * c.list_stride;
        a.list_lo = G->list_lo.as<uint32_t>() + (size_t)x * c.list_stride;
        a.list_start = G->list_start.as<uint32_t>() + (size_t)x * c.list_stride;
        c.s[x].list_sum = (uint32_t *)G->sums.p + (size_t)x * SUM_BLOCKS;
        c.s[x].cnt_sum = (Counts *)((uint32_t *)G->sums.p + 2 * SUM_BLOCKS) + (size_t)x * SUM_BLOCKS;
    }
}

// where the results of a call's strands go, in their order
using Outs = std::array<srm_filter **, 2>;

// The batch pass runs on the device unless separators have to come along that outweigh
// it (a byte a base at 20 GB/s; the host's pass takes tens of nanoseconds a read), or its
// lists of flushes and walked reads run over (run_strands): then the host's pass over the
// downloaded entries, which come down one after another.  (From the reads' own places
// they are 80 bytes a read and strand, empty or not: 100,000 reads over 60 Mbp in two
// contigs 10.4 ms, 7.8 packed; 500,000 over 4 Mbp with a flush at every 100, 34.7 and 18.6)
bool batch_on_device(const srm_dfilter *G, const uint8_t *blocked, size_t n_reads)
{
    return !blocked || G->glen / 512 <= n_reads;
}

// one or both strands over the reads on the device (both while their lists fit one sum);
// counted: their lookups are under way (upload_pieces)
int run_strands(srm_dfilter *G, Call c, bool counted, const uint8_t *blocked, const uint16_t *read_len,
                const uint8_t *read_k, const Outs &out)
{
    const uint64_t nl = c.n_lists;
    const uint32_t n = c.s[0].f.n_reads;
    bool on_device = batch_on_device(G, blocked, n);
    if (on_device && blocked) {
        FL_RC(G->upload(G->blocked, blocked, G->glen));
        c.blocked = G->blocked.as<uint8_t>();
    }
    if (!counted) FL_RC(ensure_lists(G, c));
    FL_RC(G->cnt.ensure(((size_t)n + 1) * sizeof(Counts) * (size_t)c.n));
    FL_RC(G->start.ensure(((size_t)n + 1) * sizeof(Counts) * (size_t)c.n));
    FL_RC(G->by_rank.ensure((size_t)n * 4 * (size_t)c.n));
    FL_RC(G->unsafe.ensure((size_t)MAX_UNSAFE * 4 * (size_t)c.n));
    FL_RC(G->walk.ensure((size_t)MAX_WALK * 4 * (size_t)c.n));
    const size_t head = sizeof(Header) * (size_t)c.n;
    for (int x = 0; x < c.n; ++x) {
        // about one position a list beside its terminator
        FL_RC(G->flat[x].ensure((nl * 2 + 1024) * 4));
        // (behind the slots, room for the first reads that outgrow them)
        FL_RC(G->out_pos[x].ensure(((size_t)n * ECAP + OVER_ROOM) * 4));
        FL_RC(G->out_flag[x].ensure((size_t)n * ECAP + OVER_ROOM));
        FL_RC(G->out_perf[x].ensure(((size_t)n * PCAP + OVER_ROOM) * 4));
        FL_RC(G->meta[x].ensure((size_t)n * 12));
        FL_RC(G->over[x][0].ensure((size_t)n * 4));
    }
    auto bind = [&] {
        bind_lists(G, c);
        for (int x = 0; x < c.n; ++x) {
            Strand &s = c.s[x];
            FArgs &a = s.f;
            s.flat_cap = std::min<uint64_t>(G->flat[x].cap / 4, MAX_FLAT);
            s.cnt = G->cnt.as<Counts>() + (size_t)x * ((size_t)n + 1);
            s.start = G->start.as<Counts>() + (size_t)x * ((size_t)n + 1);
            s.by_rank = G->by_rank.as<uint32_t>() + (size_t)x * n;
            s.unsafe = G->unsafe.as<uint32_t>() + (size_t)x * MAX_UNSAFE;
            s.walk = G->walk.as<uint32_t>() + (size_t)x * MAX_WALK;
            a.flat = G->flat[x].as<uint32_t>();
            a.out_pos = G->out_pos[x].as<int32_t>();
            a.out_flag = G->out_flag[x].as<int8_t>();
            a.out_perf = G->out_perf[x].as<int32_t>();
            a.meta = G->meta[x].as<uint32_t>();
            a.over = G->over[x][0].as<uint32_t>();
            a.todo = nullptr;
            a.n_todo = n;
            a.cap = ECAP;
            a.pcap = PCAP;
        }
        c.blob = G->out.as<unsigned char>() + head;
        c.blob_cap = G->out.cap - head;
        c.back = (unsigned char *)G->stage_out;
        c.back_cap = STAGE_OUT;
    };
    bind();
    if (!counted) FL_RC(launch_count(G, c, 0, n));
    FL_RC(launch_search(G, c));
    if (on_device) FL_RC(launch_batch(G, c));
    // the headers and the first part of the output; what did not fit is made room for
    // and run again
    Header h[2];
    const auto *so = (const unsigned char *)G->stage_out;
    auto fetch = [&]() -> int {
        FL_TRY(hipEventRecord(G->ev[1], G->st));
        if (!on_device)   // (fl_batch_end sends them)
            FL_TRY(hipMemcpyAsync(G->stage_out, G->out.p, head, hipMemcpyDeviceToHost, G->st));
        FL_TRY(hipStreamSynchronize(G->st));
        std::memcpy(h, so, head);
        return SRM_OK;
    };
    if (!on_device) {   // the list total, which fl_batch_end would have left
        hipLaunchKernelGGL(fl_totals, dim3(1, (unsigned)c.n), dim3(64), 0, G->st, c);
        FL_TRY(hipGetLastError());
    }
    FL_RC(fetch());
    auto countable = [&]() -> int {
        for (int x = 0; x < c.n; ++x)
            if (h[x].flat > MAX_FLAT)   // (or TOO_MANY)
                return srm::set_error(SRM_ENOMEM, "the q-gram lists of %u reads hold more than %llu "
                                      "positions; split the call", n, (unsigned long long)MAX_FLAT);
        return SRM_OK;
    };
    FL_RC(countable());
    bool again = false;
    for (int x = 0; x < c.n; ++x)
        if ((uint64_t)h[x].flat > c.s[x].flat_cap) {
            FL_RC(G->flat[x].ensure(((size_t)h[x].flat + h[x].flat / 8) * 4));
            again = true;
        }
    if (again) {
        bind();
        FL_RC(launch_count(G, c, 0, n));   // (the counters start over)
        FL_RC(launch_search(G, c));
        if (on_device) FL_RC(launch_batch(G, c));
        FL_RC(fetch());
        FL_RC(countable());
    }
    again = false;
    auto overflow = [&]() -> int {
        for (int x = 0; x < c.n; ++x)
            if (h[x].counters[2]) {
                FL_RC(run_overflow(G, c, x, h[x]));
                again = true;
            }
        return SRM_OK;
    };
    for (int x = 0; x < c.n; ++x) {
        G->last_flat += h[x].flat;
        G->last_overflow += h[x].counters[2];
    }
    FL_RC(overflow());
    // the counters of the reads the batch pass lists start over
    auto batch_again = [&]() -> int {
        bind();
        for (int x = 0; x < c.n; ++x) FL_TRY(srm::launch_reset(&c.s[x].hdr->n_unsafe, 3, G->st));
        FL_RC(launch_batch(G, c));
        return fetch();
    };
    if (again && on_device) FL_RC(batch_again());
    if (on_device && !h[0].blob_ok) {
        const BlobAt b = blob_at(h[0].total, c.n > 1 ? h[1].total : Counts());
        // (the headers' entry counts stay: the output is made anew behind them)
        FL_RC(G->grow(G->out, head + b.bytes, head));
        FL_RC(batch_again());
    }
    FL_TRY(hipEventElapsedTime(&G->last_ms, G->ev[0], G->ev[1]));
    for (int x = 0; x < c.n; ++x)
        if (h[x].n_flush > MAX_FLUSH || h[x].n_unsafe > MAX_UNSAFE || h[x].walk_words > MAX_WALK)
            on_device = false;
    if (!on_device && !c.s[0].f.packed) {
        for (int x = 0; x < c.n; ++x) c.s[x].f.packed = true;
        bind();
        FL_RC(launch_count(G, c, 0, n));   // (the counters start over)
        FL_RC(launch_search(G, c));
        FL_RC(fetch());
        FL_RC(overflow());
    }
    if (!on_device) {
        std::vector<uint32_t> meta_h[2];
        std::vector<int32_t> pos_h[2], perf_h[2];
        std::vector<int8_t> flag_h[2];
        for (int x = 0; x < c.n; ++x) {
            FL_RC(G->get(meta_h[x], G->meta[x], (size_t)n * 3));
            FL_RC(G->get(pos_h[x], G->out_pos[x], h[x].counters[0]));
            FL_RC(G->get(flag_h[x], G->out_flag[x], h[x].counters[0]));
            FL_RC(G->get(perf_h[x], G->out_perf[x], h[x].counters[1]));
        }
        FL_TRY(hipStreamSynchronize(G->st));
        auto pass = [&](int x) {
            *out[x] = batch_pass(MetaAcc{meta_h[x], pos_h[x], flag_h[x], perf_h[x]}, n, read_len, read_k,
                                G->glen, blocked, (int)c.s[0].f.cv);
        };
        std::thread other;   // the two strands' passes side by side
        if (c.n > 1) {
            try {
                other = std::thread(pass, 1);
            } catch (...) {   // no thread to be had: both passes on this one
                pass(1);
            }
        }
        pass(0);
        if (other.joinable()) other.join();
        return SRM_OK;
    }
    // the output: from the first copy when it is all there, else into page-locked memory
    const BlobAt b = blob_at(h[0].total, c.n > 1 ? h[1].total : Counts());
    std::shared_ptr<void> hold;
    if (b.bytes <= STAGE_OUT) {
        void *p = std::malloc(std::max<size_t>(b.bytes, 1));
        if (p) hold = std::shared_ptr<void>(p, std::free);
    } else {
        hold = G->pool->take(b.bytes);
    }
    if (!hold) return srm::set_error(SRM_ENOMEM, "no memory for %zu bytes of filter results", (size_t)b.bytes);
    auto *m = (unsigned char *)hold.get();
    std::vector<uint32_t> walk_h[2];
    bool wait = false;
    if (b.bytes <= STAGE_OUT) {
        std::memcpy(m, so + head, b.bytes);
    } else {
        FL_TRY(hipMemcpyAsync(m, c.blob, b.bytes, hipMemcpyDeviceToHost, G->st));
        wait = true;
    }
    for (int x = 0; x < c.n; ++x)
        if (h[x].walk_words) {
            walk_h[x].resize(h[x].walk_words);
            FL_TRY(hipMemcpyAsync(walk_h[x].data(), c.s[x].walk, (size_t)h[x].walk_words * 4,
                                  hipMemcpyDeviceToHost, G->st));
            wait = true;
        }
    if (wait) FL_TRY(hipStreamSynchronize(G->st));
    for (int x = 0; x < c.n; ++x) {
        std::vector<Walked> walked;
        for (size_t w = 0; w < walk_h[x].size();) {
            const uint32_t *v = walk_h[x].data() + w;
            Walked k;
            k.read = v[0];
            k.rank = v[1];
            k.cand_start = v[2];
            const uint32_t ne = v[3];
            for (uint32_t e = 0; e < ne; ++e) {
                k.pos.push_back((int32_t)v[4 + e]);
                k.flag.push_back((int8_t)(int32_t)v[4 + ne + e]);
            }
            walked.push_back(std::move(k));
            w += 4 + 2 * (size_t)ne;
        }
        auto F = std::make_unique<srm_filter>();
        F->dense = std::make_unique<Pieces>();
        Pieces &R = *F->dense;
        R.hold = hold;
        R.c_pos = (int64_t *)(m + b.c_pos[x]);
        R.p_pos = (int64_t *)(m + b.p_pos[x]);
        R.c_read = (int32_t *)(m + b.c_read[x]);
        R.p_read = (int32_t *)(m + b.p_read[x]);
        R.c_w = (uint16_t *)(m + b.c_w[x]);
        R.c_flag = m + b.c_flag[x];
        R.n_perf = h[x].total.perf;
        finish(R, F->batch_end, std::vector<Flush>(h[x].flush, h[x].flush + h[x].n_flush), walked,
               read_len, read_k, G->glen, blocked);
        *out[x] = F.release();
    }
    return SRM_OK;
}

// The reads and their plan to the device in pieces, the plan and the lookups of one
// piece made while the next ones are on their way.  c: the strands to look up.  counted
// stays false where the totals guessed from a sample of the reads do not hold: the call
// goes on as a small one.
//
// Bound by the copy of the reads (57 GB/s from page-locked memory).  With the plan made
// before it and the lookups after it, 2M reads of 143 bp took 3.5 + 6.6 + 2.9 ms; in
// pieces 6.5 ms.
int upload_pieces(srm_dfilter *G, Call &c, const char *reads, const uint64_t *read_off,
                  const uint16_t *read_len, const uint8_t *read_k, size_t n, bool &counted)
{
    Planner plan(G->ix, false);
    std::string err;
    // the totals: the end of the last read, and the lists of every so many reads
    const size_t bytes = read_off[n - 1] + read_len[n - 1], step = std::max<size_t>(1, n / 512);
    uint64_t sum = 0, seen = 0;
    for (size_t i = 0; i < n; i += step, ++seen) {
        const int32_t id = plan.set_of(read_len[i], read_k[i], err);
        if (id < 0) return SRM_OK;   // the first bad read's error is the call's
        sum += (uint64_t)plan.params[(size_t)id].n;
    }
    const uint64_t room = (uint64_t)((double)sum / (double)seen * (double)n * 1.125) + 4096;
    if (room >= (uint64_t)1 << 30 || plan.params.size() > MAX_SETS) return SRM_OK;
    size_t at[5] = {MAX_SETS * sizeof(DParam), (n + 1) * 4, n * 2, n * 8, bytes}, all = 0;
    for (size_t &p : at) {
        const size_t b = p;
        p = all;
        all = (all + b + 255) & ~(size_t)255;
    }
    FL_RC(G->in.ensure(all + 64));   // slack: whole 16-byte words of the reads are read
    char *in = G->in.as<char>();
    c.list_stride = room;
    FArgs &a = c.s[0].f;
    a.par = (const DParam *)(in + at[0]);
    a.list_base = (const uint32_t *)(in + at[1]);
    a.pid = (const uint16_t *)(in + at[2]);
    a.roff = (const uint64_t *)(in + at[3]);
    a.reads = in + at[4];
    FL_RC(ensure_lists(G, c));
    FL_RC(G->pack(a.reads, bytes, G->read_pk, G->read_odd, 0, 0));
    a.read_pk = G->read_pk.as<uint32_t>();
    a.read_odd = G->read_odd.as<uint32_t>();
    if (c.n > 1) {
        c.s[1].f = a;
        c.s[1].f.dr = 4;
    }
    bind_lists(G, c);
    size_t sent = 0, sets = 0;
    std::vector<DParam> dpar;
    std::vector<uint16_t> gram;
    // an eighth of the reads, so that little is left to do after the last one's arrival;
    // a piece below 65,536 costs more calls than it hides
    const size_t piece = std::min(PIECE, std::max<size_t>(PIECE / 2, (n + 7) / 8));
    int k = 0;
    for (size_t lo = 0; lo < n; lo += piece, ++k) {
        const size_t hi = std::min(n, lo + piece), m = hi - lo;
        hipEvent_t planned = G->plan_ev[k & 1], sent_ev = G->piece_ev[k & 1];
        if (k >= 2) FL_TRY(hipEventSynchronize(planned));   // its staging is free again
        char *st = (char *)G->stage_plan + (size_t)(k & 1) * PIECE_BYTES;
        auto *off = (uint64_t *)st;
        auto *base = (uint32_t *)(off + PIECE);
        auto *pid = (uint16_t *)(base + PIECE + 2);
        if (int rc = plan.piece(read_off, read_len, read_k, lo, hi, pid, base, err))
            return srm::set_error(rc, "%s", err.c_str());
        if (plan.n_lists + 1 > room || plan.read_bytes > bytes || plan.params.size() > MAX_SETS)
            return SRM_OK;
        if (plan.params.size() > sets) {
            dpar.clear();
            device_params(plan.params, dpar, gram);
            FL_TRY(hipMemcpyAsync(in + at[0] + sets * sizeof(DParam), dpar.data() + sets,
                                  (dpar.size() - sets) * sizeof(DParam), hipMemcpyHostToDevice, G->plan_st));
            FL_TRY(hipStreamSynchronize(G->plan_st));   // (dpar changes with the next sets)
            sets = plan.params.size();
        }
        if (plan.read_bytes > sent)
            FL_TRY(hipMemcpyAsync(in + at[4] + sent, reads + sent, plan.read_bytes - sent,
                                  hipMemcpyHostToDevice, G->copy_st));
        FL_TRY(hipEventRecord(sent_ev, G->copy_st));
        // the plan's arrays on another stream: between two copies of one an engine rests for
        // 25 us, 100 us of a piece's 490 with all four on one stream (2M reads 13.0 -> 12.6 ms)
        std::memcpy(off, read_off + lo, m * 8);
        FL_TRY(hipMemcpyAsync(in + at[1] + lo * 4, base, (m + 1) * 4, hipMemcpyHostToDevice, G->plan_st));
        FL_TRY(hipMemcpyAsync(in + at[2] + lo * 2, pid, m * 2, hipMemcpyHostToDevice, G->plan_st));
        FL_TRY(hipMemcpyAsync(in + at[3] + lo * 8, off, m * 8, hipMemcpyHostToDevice, G->plan_st));
        FL_TRY(hipEventRecord(planned, G->plan_st));
        FL_TRY(hipStreamWaitEvent(G->st, planned, 0));
        FL_TRY(hipStreamWaitEvent(G->st, sent_ev, 0));
        // (the bytes of a word that two pieces share are packed again with the second)
        FL_RC(G->pack(a.reads, bytes, G->read_pk, G->read_odd, sent, plan.read_bytes));
        sent = plan.read_bytes;
        c.n_lists = plan.n_lists;
        FL_RC(launch_count(G, c, (uint32_t)lo, (uint32_t)hi));
    }
    for (const Params &p : plan.params) c.kmax = std::max(c.kmax, p.k);
    counted = true;
    return SRM_OK;
}

// the codes of the call's reads to words (srm::dfilter_run2_words), copied beside the
// kernels that follow
int send_words(srm_dfilter *G, const FArgs &a, uint64_t total, uint32_t *words)
{
    const size_t n_words = (2 * total + 2 * SRM_CODE_PAD + 15) / 16 + 1;
    FL_RC(G->words.ensure(n_words * 4));
    hipLaunchKernelGGL(fl_read_words, dim3((unsigned)((n_words + FB - 1) / FB)), dim3(FB), 0, G->st,
                       a.read_pk, (const uint16_t *)a.read_odd, a.roff, a.n_reads, total,
                       (uint32_t)SRM_CODE_PAD, G->words.as<uint32_t>(), n_words);
    FL_TRY(hipGetLastError());
    FL_TRY(hipEventRecord(G->words_ev, G->st));
    FL_TRY(hipStreamWaitEvent(G->copy_st, G->words_ev, 0));
    FL_TRY(hipMemcpyAsync(words, G->words.p, n_words * 4, hipMemcpyDeviceToHost, G->copy_st));
    return SRM_OK;
}

// one or both strands (strands: bit 0 forward, bit 1 reverse) over one upload of
// the reads
int run_device(srm_dfilter *G, const uint8_t *blocked, const char *reads,
               const uint64_t *read_off, const uint16_t *read_len, const uint8_t *read_k,
               size_t n_reads, int strands, int chunk_value, uint32_t *words,
               srm_filter **out_fwd, srm_filter **out_rev)
{
    G->last_flat = 0;
    G->last_overflow = 0;
    FL_TRY(hipSetDevice(G->device));
    FL_TRY(hipEventRecord(G->ev[0], G->st));
    FArgs a{};
    // (beyond 2^27, the places of all reads leave no 32-bit offsets for the entries behind
    // them; and the host takes the entries alone)
    a.packed = n_reads > ((size_t)1 << 27) || !batch_on_device(G, blocked, n_reads);
    a.qix = G->dq.as<DQ>();
    a.genome = G->genome.as<char>();
    a.glen = G->glen;
    a.gen_pk = G->gen_pk.as<uint32_t>();
    a.gen_odd = G->gen_odd.as<uint32_t>();
    a.n_reads = (uint32_t)n_reads;
    a.cv = (uint32_t)chunk_value;
    const Outs outs = strands == 2 ? Outs{out_rev, nullptr} : Outs{out_fwd, out_rev};
    Call c{};
    c.n = strands == 3 ? 2 : 1;
    c.s[0].f = a;
    c.s[0].f.dr = strands == 2 ? 4 : 0;
    // in pieces of 65,536 reads and more; half a piece's worth is one piece
    if (n_reads > PIECE / 4) {
        bool counted = false;
        int rc = upload_pieces(G, c, reads, read_off, read_len, read_k, n_reads, counted);
        if (rc == SRM_OK && counted) {
            G->last_lists = c.n_lists * (uint64_t)c.n;
            if (words) rc = send_words(G, c.s[0].f, read_off[n_reads - 1] + read_len[n_reads - 1], words);
            if (rc == SRM_OK) rc = run_strands(G, c, true, blocked, read_len, read_k, outs);
        }
        if (rc != NO_ROOM && (rc != SRM_OK || counted)) return rc;
        FL_TRY(hipStreamSynchronize(G->copy_st));
        FL_TRY(hipStreamSynchronize(G->plan_st));
        FL_TRY(hipStreamSynchronize(G->st));
        if (rc == NO_ROOM) {   // for the guessed totals: the exact ones take less
            G->release_strands();
            for (GBuf *b : {&G->in, &G->read_pk, &G->read_odd, &G->words}) b->release();
        }
    }
    ReadPlan plan;
    std::string err;
    if (int rc = plan_reads(G->ix, read_off, read_len, read_k, n_reads, plan, err, false))
        return srm::set_error(rc, "%s", err.c_str());
    std::vector<DParam> dpar;
    std::vector<uint16_t> gram;
    device_params(plan.params, dpar, gram);
    const auto &pid = plan.pid;
    const auto &list_base = plan.list_base;
    const uint64_t nl = list_base[n_reads];
    const uint64_t rbytes = plan.read_bytes;
    G->last_lists = nl * (strands == 3 ? 2 : 1);
    // the inputs, one after another in one buffer
    struct Part {
        const void *src;
        size_t bytes, at;
    };
    Part part[] = {{dpar.data(), dpar.size() * sizeof(DParam), 0},
                   {list_base.data(), (n_reads + 1) * 4, 0},
                   {pid.data(), n_reads * 2, 0},
                   {read_off, n_reads * 8, 0},
                   {reads, rbytes, 0}};
    size_t all = 0;
    for (Part &p : part) {
        p.at = all;
        all = (all + p.bytes + 255) & ~(size_t)255;
    }
    FL_RC(G->in.ensure(all + 64));   // slack: whole 16-byte words of the reads are read
    if (all <= STAGE_IN) {
        for (const Part &p : part) std::memcpy((char *)G->stage_in + p.at, p.src, p.bytes);
        FL_RC(G->pack(nullptr, rbytes, G->read_pk, G->read_odd, 0, 0));   // their room
        const size_t n16 = (part[4].at + rbytes + 15) / 16;
        hipLaunchKernelGGL(fl_take, dim3((unsigned)((n16 + FB - 1) / FB)), dim3(FB), 0, G->st,
                           (const uint4 *)G->stage_in, G->in.as<uint4>(), part[4].at / 16,
                           G->read_pk.as<uint32_t>(), G->read_odd.as<uint16_t>(), n16);
        FL_TRY(hipGetLastError());
    } else {
        for (const Part &p : part)
            if (p.bytes)
                FL_TRY(hipMemcpyAsync(G->in.as<char>() + p.at, p.src, p.bytes, hipMemcpyHostToDevice,
                                      G->st));
        FL_RC(G->pack(G->in.as<char>() + part[4].at, rbytes, G->read_pk, G->read_odd));
    }
    const char *in = G->in.as<char>();
    a.par = (const DParam *)(in + part[0].at);
    a.reads = in + part[4].at;
    a.read_pk = G->read_pk.as<uint32_t>();
    a.read_odd = G->read_odd.as<uint32_t>();
    a.roff = (const uint64_t *)(in + part[3].at);
    a.pid = (const uint16_t *)(in + part[2].at);
    a.list_base = (const uint32_t *)(in + part[1].at);
    if (words) FL_RC(send_words(G, a, rbytes, words));
    c = Call{};
    c.n_lists = nl;
    c.list_stride = nl + 1;
    c.sums = n_reads <= SUM_READS;
    for (const Params &p : plan.params) c.kmax = std::max(c.kmax, p.k);
    // both strands in each launch, while their lists fit one sum
    if (strands == 3 && nl < ((uint64_t)1 << 30) - 1) {
        c.n = 2;
        c.s[0].f = c.s[1].f = a;
        c.s[1].f.dr = 4;
        const int rc = run_strands(G, c, false, blocked, read_len, read_k, outs);
        if (rc != NO_ROOM) return rc;
        // one strand at a time holds half as much
        FL_TRY(hipStreamSynchronize(G->st));
        G->release_strands();
    }
    for (int x = 0; x < 2; ++x) {
        if (!(strands & (1 << x))) continue;
        c.n = 1;
        c.s[0].f = a;
        c.s[0].f.dr = x ? 4 : 0;
        FL_RC(run_strands(G, c, false, blocked, read_len, read_k, {x ? out_rev : out_fwd, nullptr}));
    }
    return SRM_OK;
}

// run_device, its exceptions as error codes; whatever fails, nothing of the call's is
// still being copied when it returns
int run_call(srm_dfilter *G, const uint8_t *blocked, const char *reads, const uint64_t *read_off,
             const uint16_t *read_len, const uint8_t *read_k, size_t n_reads, int strands,
             int chunk_value, uint32_t *words, srm_filter **out_fwd, srm_filter **out_rev)
{
    int rc;
    try {
        rc = run_device(G, blocked, reads, read_off, read_len, read_k, n_reads, strands, chunk_value,
                        words, out_fwd, out_rev);
        if (rc == SRM_OK && words && hipStreamSynchronize(G->copy_st) != hipSuccess)
            rc = srm::set_error(SRM_EDEVICE, "the copy of the reads' codes failed");
    } catch (const std::bad_alloc &) {
        rc = srm::set_error(SRM_ENOMEM, "no memory on the host for %zu reads", n_reads);
    }
    if (rc == NO_ROOM) rc = SRM_ENOMEM;
    if (rc != SRM_OK) {
        (void)hipStreamSynchronize(G->copy_st);
        (void)hipStreamSynchronize(G->plan_st);
        (void)hipStreamSynchronize(G->st);
    }
    return rc;
}

}  // namespace

namespace srm {

int dfilter_run2_words(srm_dfilter *G, const uint8_t *blocked, const char *reads,
                       const uint64_t *read_off, const uint16_t *read_len, const uint8_t *read_k,
                       size_t n_reads, int chunk_value, uint32_t *words, srm_filter **out_fwd,
                       srm_filter **out_rev)
{
    *out_fwd = nullptr;
    *out_rev = nullptr;
    if (!G || chunk_value < 1) return srm::set_error(SRM_EINVAL, "bad filter arguments");
    if (n_reads == 0) {
        *out_fwd = new srm_filter();
        *out_rev = new srm_filter();
        return SRM_OK;
    }
    srm_filter *Ff = nullptr, *Fr = nullptr;
    const int rc = run_call(G, blocked, reads, read_off, read_len, read_k, n_reads, 3, chunk_value,
                            words, &Ff, &Fr);
    if (rc != SRM_OK) {
        delete Ff;
        delete Fr;
        return rc;
    }
    *out_fwd = Ff;
    *out_rev = Fr;
    return SRM_OK;
}

}  // namespace srm

extern "C" {

int srm_dfilter_create(srm_ctx *ctx, const srm_index *ix, const char *genome, size_t glen,
                       srm_dfilter **out)
{
    *out = nullptr;
    if (!ctx || !ix || glen != ix->glen)
        return srm::set_error(SRM_EINVAL, "genome length does not match the index");
    if (ix->base != 0)
        return srm::set_error(SRM_EINVAL, "a -G chunk's index runs on the host filter");
    auto *G = new srm_dfilter();
    G->ctx = ctx;
    G->device = srm::ctx_device(ctx);
    G->st = srm::ctx_stream(ctx);
    G->ix = ix;
    G->glen = glen;
    auto fail = [&](int rc) {
        delete G;
        return rc == NO_ROOM ? SRM_ENOMEM : rc;
    };
    if (hipSetDevice(G->device) != hipSuccess ||
        hipEventCreate(&G->ev[0]) != hipSuccess || hipEventCreate(&G->ev[1]) != hipSuccess ||
        hipEventCreateWithFlags(&G->piece_ev[0], hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&G->piece_ev[1], hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&G->words_ev, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&G->plan_ev[0], hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&G->plan_ev[1], hipEventDisableTiming) != hipSuccess ||
        hipStreamCreateWithFlags(&G->plan_st, hipStreamNonBlocking) != hipSuccess ||
        hipStreamCreateWithFlags(&G->copy_st, hipStreamNonBlocking) != hipSuccess)
        return fail(srm::set_error(SRM_EDEVICE, "event creation failed"));
    if (srm::host_alloc(&G->stage_in, STAGE_IN) != hipSuccess ||
        srm::host_alloc(&G->stage_plan, 2 * PIECE_BYTES) != hipSuccess ||
        srm::host_alloc(&G->stage_out, 2 * sizeof(Header) + STAGE_OUT) != hipSuccess)
        return fail(srm::set_error(SRM_ENOMEM, "no page-locked memory for the filter's staging"));
    int rc = G->upload(G->genome, genome, glen);
    if (!rc) rc = G->pack(G->genome.p, glen, G->gen_pk, G->gen_odd);
    if (rc) return fail(rc);
    std::vector<DQ> dq(32);
    std::memset(dq.data(), 0, dq.size() * sizeof(DQ));
    G->keys.resize(ix->idx.size());
    G->pre.resize(ix->idx.size());
    G->odd_hash.resize(ix->idx.size());
    G->odd_pos.resize(ix->idx.size());
    for (size_t i = 0; i < ix->idx.size(); ++i) {
        const QIndex &X = ix->idx[i];
        std::vector<uint64_t> oh;
        std::vector<uint32_t> op;
        odd_table(X, oh, op);
        if ((rc = G->upload(G->keys[i], X.keys.data(), X.keys.size() * 8)) ||
            (rc = G->upload(G->pre[i], X.pre.data(), X.pre.size() * 4)) ||
            (rc = G->upload(G->odd_hash[i], oh.data(), oh.size() * 8)) ||
            (rc = G->upload(G->odd_pos[i], op.data(), op.size() * 4)))
            return fail(rc);
        DQ &d = dq[(size_t)X.q];
        d.keys = G->keys[i].as<uint64_t>();
        d.pre = G->pre[i].as<uint32_t>();
        d.odd_hash = G->odd_hash[i].as<uint64_t>();
        d.odd_pos = G->odd_pos[i].as<uint32_t>();
        d.n_odd = (uint32_t)oh.size();
        d.q = X.q;
        d.pos_bits = X.pos_bits;
        d.pre_bases = X.pre_bases;
        // the upload above is asynchronous; the host vectors must outlive it
        if (hipStreamSynchronize(G->st) != hipSuccess)
            return fail(srm::set_error(SRM_EDEVICE, "index upload failed"));
    }
    if ((rc = G->upload(G->dq, dq.data(), dq.size() * sizeof(DQ)))) return fail(rc);
    if (hipStreamSynchronize(G->st) != hipSuccess)
        return fail(srm::set_error(SRM_EDEVICE, "index upload failed"));
    *out = G;
    return SRM_OK;
}

int srm_dfilter_run(srm_dfilter *G, const uint8_t *blocked, const char *reads,
                    const uint64_t *read_off, const uint16_t *read_len, const uint8_t *read_k,
                    size_t n_reads, int do_reverse, int chunk_value, srm_filter **out)
{
    *out = nullptr;
    if (!G || chunk_value < 1 || (do_reverse != 0 && do_reverse != 4))
        return srm::set_error(SRM_EINVAL, "bad filter arguments");
    if (n_reads == 0) {
        *out = new srm_filter();
        return SRM_OK;
    }
    srm_filter *F = nullptr;
    const int rc = run_call(G, blocked, reads, read_off, read_len, read_k, n_reads,
                            do_reverse ? 2 : 1, chunk_value, nullptr, &F, &F);
    if (rc != SRM_OK) {
        delete F;
        return rc;
    }
    *out = F;
    return SRM_OK;
}

int srm_dfilter_run2(srm_dfilter *G, const uint8_t *blocked, const char *reads,
                     const uint64_t *read_off, const uint16_t *read_len, const uint8_t *read_k,
                     size_t n_reads, int chunk_value, srm_filter **out_fwd, srm_filter **out_rev)
{
    return srm::dfilter_run2_words(G, blocked, reads, read_off, read_len, read_k, n_reads, chunk_value,
                                   nullptr, out_fwd, out_rev);
}

int srm_dfilter_stats(const srm_dfilter *G, float *device_ms, uint64_t *n_lists,
                      uint64_t *n_list_entries, uint64_t *n_overflow)
{
    if (device_ms) *device_ms = G->last_ms;
    if (n_lists) *n_lists = G->last_lists;
    if (n_list_entries) *n_list_entries = G->last_flat;
    if (n_overflow) *n_overflow = G->last_overflow;
    return SRM_OK;
}

void srm_dfilter_destroy(srm_dfilter *G)
{
    if (!G) return;
    (void)hipSetDevice(G->device);
    (void)hipStreamSynchronize(G->copy_st);
    (void)hipStreamSynchronize(G->plan_st);
    (void)hipStreamSynchronize(G->st);
    delete G;
}

}  // extern "C"
