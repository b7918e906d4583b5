// filter_gpu.hip -- the q-gram filter ("SEASHORE") on the GPU.
//
// Same candidates, flags, perfect hits and batch boundaries as the host filter
// (filter.cpp); only the per-read work moves to the device:
//   0. pack    the reads' bytes as 2-bit codes and a mask of other bytes;
//   1. count   one thread per q-gram of a read looks it up in the device copy of
//              the q-gram index and writes the list length + 1 and the index of
//              the list's first key;
//   2. scan    exclusive sum of the lengths = the offset of every 0-terminated
//              list in one flat array, reads in order (the reference's
//              data_array, hash.c:396-461, for all chunks at once);
//   3. fill    the same threads write the lists: a copy of the key run the
//              count found, or the hash-table lookup again for a q-gram
//              holding a byte other than ACGT;
//   4. pair    a group of lanes per read runs run_seashore (hash.c:502-834) and
//              add_start_position (hash.c:40-178) over the flat array.  A list
//              index beyond the list runs on into the following lists and the
//              following reads' lists up to the end of the read's chunk of
//              chunk_value reads (Q12), exactly as a walk of data_array does.
//              The read's result-hash entries live in LDS (16 entries, 4 perfect
//              hits per read); a read that needs more is marked and run again
//              with slots in HBM (1024, then 65534 entries);
//   5. compact every wave reserves space for its reads' entries with one atomic
//              and writes them contiguously; the host downloads 12 bytes per
//              read plus the entries.
// The sequential batch pass (Q10 leak, flush boundaries) then runs on the host
// over the downloaded entries (filter_internal.h).
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <map>
#include <string>
#include <thread>
#include <vector>

#include "filter_internal.h"
#include "filter_pair.h"
#include "nw_device.h"

using namespace srm_filter_impl;
using namespace srm_pair;

namespace {

constexpr int FB = 256;      // threads per block
constexpr int ECAP = 16;     // result-hash entries per read kept in LDS
constexpr int PCAP = 4;      // perfect hits per read kept in LDS

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
    __device__ uint32_t load(const FArgs &a, uint32_t per)
    {
        const uint32_t r0 = blockIdx.x * per;
        const uint32_t nr = a.n_reads - r0 < per ? a.n_reads - r0 : per;
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

__global__ void __launch_bounds__(FB) fl_count(FArgs a, uint32_t per)
{
    __shared__ BlockReads s;
    const uint32_t nr = s.load(a, per);
    for (uint32_t i = s.base[0] + threadIdx.x; i < s.base[nr]; i += FB) {
        const uint32_t t = s.read_of(i, nr);
        const int L = s.L[t], q = s.q[t], g = gram_offset(L, q, (int)(i - s.base[t]));
        const DQ X = a.qix[q];
        uint64_t code;
        uint32_t lo, c;
        if (gram_code(a.read_pk, a.read_odd, s.off[t], L, a.dr, q, g, code))
            c = lookup_code(X, code, lo);
        else
            c = lookup<false>(X, a.genome, a.reads + s.off[t], L, a.dr, g, nullptr, &lo);
        a.list_cnt[i] = c + 1;
        a.list_lo[i] = lo;
    }
}

// the lists themselves, blocks and threads as in fl_count: the positions are the
// keys it found, or, for a q-gram holding another byte, the hash table's
__global__ void __launch_bounds__(FB) fl_fill(FArgs a, uint32_t per)
{
    __shared__ BlockReads s;
    const uint32_t nr = s.load(a, per);
    for (uint32_t i = s.base[0] + threadIdx.x; i < s.base[nr]; i += FB) {
        const uint32_t c = a.list_cnt[i] - 1;
        uint32_t *dst = a.flat + a.list_start[i];
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

__device__ __forceinline__ uint32_t wave_incl_sum(uint32_t v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(v, d, 64);
        if (lane >= d) v += o;
    }
    return v;
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

// run_seashore (hash.c:502-834) by G lanes per read: each lane takes a start
// position (an element of the first half of the read's lists, which lie one after
// another in the flat array) and finds what it would insert -- that depends on the
// lists alone -- and the group then adds the results in the reference's order.
//
// Latency-bound: a start position is a chain of a few dependent list loads and the
// perfect check.  A thread per read walked its positions one after another and
// compared the read with the genome byte by byte, so a call lasted as long as its
// longest read's chain; here the positions' chains run side by side and the group
// compares 16 bases per lane at once, a genome start that several positions share
// only once.  2M reads of 50-250 bp, one strand: 10.6 -> 2.44 ms, the reads of many
// entries 3.39 -> 0.11 ms; 1,000 reads: 856 -> 45 us.
template <int G, bool GLOBAL>
__global__ void __launch_bounds__(FB) fl_pair(FArgs a)
{
    constexpr int NG = FB / G;           // reads per block
    constexpr uint64_t GM = G == 64 ? ~0ull : (1ull << (G & 63)) - 1;
    __shared__ int32_t s_pos[GLOBAL ? 1 : ECAP * NG];
    __shared__ int8_t s_flag[GLOBAL ? 1 : ECAP * NG];
    __shared__ int32_t s_perf[GLOBAL ? 1 : PCAP * NG];
    const int gl = threadIdx.x & (G - 1);
    const int gb = threadIdx.x & 63 & ~(G - 1);
    const uint32_t slot = threadIdx.x / G;
    const uint32_t j = blockIdx.x * NG + slot;
    const bool active = j < a.n_todo;
    Store s;
    if (GLOBAL) {
        s.pos = a.slot_pos + (size_t)j * a.cap;
        s.flag = a.slot_flag + (size_t)j * a.cap;
        s.perf = a.slot_perf + (size_t)j * a.pcap;
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
    if (active) {
        const uint32_t r = a.todo ? a.todo[j] : j;
        const DParam P = a.par[a.pid[r]];
        const uint32_t lb = a.list_base[r];
        const uint32_t i0 = a.list_start[lb], i1 = a.list_start[lb + P.half];
        // (an empty list is its terminator: nothing to do when all of them are)
        if (i1 - i0 != (uint32_t)P.half) {
            const uint64_t flat_end = chunk_end(a, r), at = a.roff[r];
            for (uint32_t p0 = i0; p0 < i1 && !s.ovf; p0 += G) {
                const uint32_t p = p0 + (uint32_t)gl;
                const uint32_t Pa = p < i1 ? a.flat[p] : 0u;
                int aa = 0;
                uint32_t off = 0;
                bool valid = Pa != 0;
                if (valid) {
                    for (int n = P.half; n > 1;) {   // the list holding p
                        const int h = n >> 1;
                        if (a.list_start[lb + aa + h] <= p) aa += h;
                        n -= h;
                    }
                    const uint32_t first = a.list_start[lb + aa];
                    off = p - first;
                    // a list that starts with offset 0 reads as empty (Q14)
                    valid = off == 0 || a.flat[first] != 0;
                }
                const long gs = (long)Pa - ((long)aa * P.q + 1);
                valid = valid && gs + 1 > 0;
                const uint32_t S = (uint32_t)(gs + 1);
                // perfect check (strncpy + strcmp, hash.c:550-583), each genome start
                // once, the group's lanes 16 bases each
                const bool check = valid && (uint64_t)S + (uint64_t)P.L <= a.glen;
                bool perfect = false;
                uint64_t todo = (__ballot(check) >> gb) & GM;
                while (todo) {
                    const uint32_t S0 = (uint32_t)__shfl((int)S, gb + (int)__builtin_ctzll(todo), 64);
                    bool ok = true;
                    for (int x = gl; 16 * x < P.L && ok; x += G) ok = same16(a, at, P.L, a.dr, S0, x);
                    const bool all = ((__ballot(!ok) >> gb) & GM) == 0;
                    const bool mine = check && S == S0;
                    if (mine) perfect = all;
                    todo &= ~((__ballot(mine) >> gb) & GM);
                }
                int32_t hpos = 0;
                int hflag = 0;
                const bool found = valid && pair_matches(a, P, lb, flat_end, aa, off, Pa, gs, hpos, hflag);
                const int what = (perfect ? 1 : 0) | (found ? 2 : 0) | (hflag << 2);
                uint64_t add = (__ballot((what & 3) != 0) >> gb) & GM;
                while (add && !s.ovf) {
                    const int src = gb + (int)__builtin_ctzll(add);
                    add &= add - 1;
                    const int w = __shfl(what, src, 64);
                    if (w & 1) {
                        const int32_t S0 = __shfl((int)S, src, 64);
                        if (group_add<G, GLOBAL>(s, -S0, 0, P.k, gl, gb) != 1 && !s.ovf) {
                            if (s.np == s.pcap) {
                                s.ovf = true;
                            } else {
                                if (gl == 0) s.Q(s.np) = S0;
                                ++s.np;
                            }
                        }
                    }
                    if ((w & 2) && !s.ovf)
                        group_add<G, GLOBAL>(s, __shfl(hpos, src, 64), w >> 2, P.k, gl, gb);
                }
            }
        }
    }
    // the group's first lane speaks for its read
    const bool lead = active && gl == 0;
    const uint32_t ne = (lead && !s.ovf) ? s.n : 0, np = (lead && !s.ovf) ? s.np : 0;
    // one atomic pair per block reserves the block's output (the two counters are
    // words that every wave would otherwise update); the waves take consecutive
    // parts of it
    __shared__ uint32_t s_sum[FB / 64][2], s_base[2];
    const uint32_t ie = wave_incl_sum(ne), ip = wave_incl_sum(np);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 63) {
        s_sum[wv][0] = ie;
        s_sum[wv][1] = ip;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t te = 0, tp = 0;
        for (int v = 0; v < FB / 64; ++v) {
            te += s_sum[v][0];
            tp += s_sum[v][1];
        }
        s_base[0] = te ? atomicAdd(&a.counters[0], te) : 0u;
        s_base[1] = tp ? atomicAdd(&a.counters[1], tp) : 0u;
    }
    __syncthreads();
    uint32_t be = s_base[0] + ie - ne, bp = s_base[1] + ip - np;
    for (int v = 0; v < wv; ++v) {
        be += s_sum[v][0];
        bp += s_sum[v][1];
    }
    if (!lead) return;
    for (uint32_t e = 0; e < ne; ++e) {
        a.out_pos[be + e] = s.P(e);
        a.out_flag[be + e] = s.F(e);
    }
    for (uint32_t e = 0; e < np; ++e) a.out_perf[bp + e] = s.Q(e);
    a.meta[3 * (size_t)j + 0] = be;
    a.meta[3 * (size_t)j + 1] = bp;
    a.meta[3 * (size_t)j + 2] = s.ovf ? OVERFLOW_MARK : (ne | (np << 16));
}

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
        hipError_t e = hipMalloc(&p, want);
        if (e != hipSuccess) {
            p = nullptr;
            return srm::set_error(SRM_ENOMEM, "hipMalloc(%zu) failed: %s", want,
                                  hipGetErrorString(e));
        }
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

}  // namespace

struct srm_dfilter {
    srm_ctx *ctx = nullptr;
    int device = 0;
    hipStream_t st = nullptr;
    const srm_index *ix = nullptr;
    size_t glen = 0;
    GBuf genome, gen_pk, gen_odd, dq;
    std::vector<GBuf> keys, pre, odd_hash, odd_pos;
    GBuf par, gram, reads, read_pk, read_odd, roff, rlen, pid, list_base, list_cnt, list_lo,
        list_start, flat, cub_tmp;
    GBuf slot_pos, slot_flag, slot_perf, out_pos, out_flag, out_perf, meta, counters, todo;
    hipEvent_t ev[2] = {nullptr, nullptr};
    float last_ms = 0.f;
    size_t last_lists = 0, last_flat = 0, last_overflow = 0;

    ~srm_dfilter()
    {
        for (GBuf *b : {&genome, &gen_pk, &gen_odd, &dq, &par, &gram, &reads, &read_pk, &read_odd, &roff, &rlen, &pid, &list_base,
                        &list_cnt, &list_lo, &list_start, &flat, &cub_tmp, &slot_pos, &slot_flag,
                        &slot_perf, &out_pos, &out_flag, &out_perf, &meta, &counters, &todo})
            b->release();
        for (auto *v : {&keys, &pre, &odd_hash, &odd_pos})
            for (auto &b : *v) b.release();
        for (auto &e : ev)
            if (e) (void)hipEventDestroy(e);
    }

    int upload(GBuf &b, const void *src, size_t bytes)
    {
        FL_RC(b.ensure(bytes + 64));   // slack: whole 16-byte words are read
        if (bytes) FL_TRY(hipMemcpyAsync(b.p, src, bytes, hipMemcpyHostToDevice, st));
        return SRM_OK;
    }

    // the codes and the mask of other bytes of b's bytes (two code words and one mask
    // word past the last are read beside them)
    int pack(const GBuf &b, size_t bytes, GBuf &pk, GBuf &odd)
    {
        const size_t n16 = (bytes + 15) / 16;
        FL_RC(pk.ensure((n16 + 4) * 4));
        FL_RC(odd.ensure((n16 + 4) * 2 + 4));
        if (n16 == 0) return SRM_OK;
        hipLaunchKernelGGL(fl_pack, dim3((unsigned)((n16 + FB - 1) / FB)), dim3(FB), 0, st,
                           b.as<const uint4>(), pk.as<uint32_t>(), odd.as<uint16_t>(), n16);
        FL_TRY(hipGetLastError());
        return SRM_OK;
    }

    // runs the pairing kernel over n reads (todo == null: all reads of the call)
    // and downloads meta and the compact output
    int pair(FArgs a, bool global, const uint32_t *todo_host, uint32_t n, uint32_t cap,
             uint32_t pcap, std::vector<uint32_t> &meta_h, std::vector<int32_t> &pos_h,
             std::vector<int8_t> &flag_h, std::vector<int32_t> &perf_h)
    {
        a.n_todo = n;
        a.todo = nullptr;
        if (todo_host) {
            FL_RC(upload(todo, todo_host, (size_t)n * 4));
            a.todo = todo.as<uint32_t>();
        }
        if (global) {
            FL_RC(slot_pos.ensure((size_t)n * cap * 4));
            FL_RC(slot_flag.ensure((size_t)n * cap));
            FL_RC(slot_perf.ensure((size_t)n * pcap * 4));
            a.slot_pos = slot_pos.as<int32_t>();
            a.slot_flag = slot_flag.as<int8_t>();
            a.slot_perf = slot_perf.as<int32_t>();
        }
        a.cap = cap;
        a.pcap = pcap;
        FL_RC(out_pos.ensure((size_t)n * cap * 4));
        FL_RC(out_flag.ensure((size_t)n * cap));
        FL_RC(out_perf.ensure((size_t)n * pcap * 4));
        FL_RC(meta.ensure((size_t)n * 12));
        FL_RC(counters.ensure(8));
        a.out_pos = out_pos.as<int32_t>();
        a.out_flag = out_flag.as<int8_t>();
        a.out_perf = out_perf.as<int32_t>();
        a.meta = meta.as<uint32_t>();
        a.counters = counters.as<uint32_t>();
        FL_TRY(hipMemsetAsync(a.counters, 0, 8, st));
        // lanes per read: a wave for the reads of hundreds of entries; 8, about the
        // start positions of a read that maps once, for many reads; 32 for the few
        // thousand that leave the chip idle either way, where one step covers a
        // read's lists (1,000 reads, both strands: 0.373 ms on the device with 32,
        // 0.414 with 8; 2M reads: 38.1 and 32.2 ms)
        auto grid = [&](unsigned g) { return dim3((n + FB / g - 1) / (FB / g)); };
        if (global) hipLaunchKernelGGL((fl_pair<64, true>), grid(64), dim3(FB), 0, st, a);
        else if (n < 4096) hipLaunchKernelGGL((fl_pair<32, false>), grid(32), dim3(FB), 0, st, a);
        else hipLaunchKernelGGL((fl_pair<8, false>), grid(8), dim3(FB), 0, st, a);
        FL_TRY(hipGetLastError());
        uint32_t tot[2];
        FL_TRY(hipMemcpyAsync(tot, a.counters, 8, hipMemcpyDeviceToHost, st));
        meta_h.resize((size_t)n * 3);
        FL_TRY(hipMemcpyAsync(meta_h.data(), a.meta, (size_t)n * 12, hipMemcpyDeviceToHost, st));
        FL_TRY(hipStreamSynchronize(st));
        pos_h.resize(tot[0]);
        flag_h.resize(tot[0]);
        perf_h.resize(tot[1]);
        if (tot[0]) {
            FL_TRY(hipMemcpyAsync(pos_h.data(), a.out_pos, (size_t)tot[0] * 4,
                                  hipMemcpyDeviceToHost, st));
            FL_TRY(hipMemcpyAsync(flag_h.data(), a.out_flag, tot[0], hipMemcpyDeviceToHost, st));
        }
        if (tot[1])
            FL_TRY(hipMemcpyAsync(perf_h.data(), a.out_perf, (size_t)tot[1] * 4,
                                  hipMemcpyDeviceToHost, st));
        FL_TRY(hipStreamSynchronize(st));
        return SRM_OK;
    }
};

namespace {

// one or both strands (strands: bit 0 forward, bit 1 reverse) over one upload of
// the reads
int run_device(srm_dfilter *G, const uint8_t *blocked, const char *reads,
               const uint64_t *read_off, const uint16_t *read_len, const uint8_t *read_k,
               size_t n_reads, int strands, int chunk_value, srm_filter **out_fwd,
               srm_filter **out_rev)
{
    ReadPlan plan;
    std::string err;
    if (int rc = plan_reads(G->ix, read_off, read_len, read_k, n_reads, plan, err))
        return srm::set_error(rc, "%s", err.c_str());
    std::vector<DParam> dpar;
    std::vector<uint16_t> gram;
    device_params(plan.params, dpar, gram);
    const auto &pid = plan.pid;
    const auto &list_base = plan.list_base;
    const uint64_t nl = list_base[n_reads];
    const uint64_t rbytes = plan.read_bytes;
    G->last_lists = 0;
    G->last_flat = 0;
    G->last_overflow = 0;
    FL_TRY(hipSetDevice(G->device));
    FL_TRY(hipEventRecord(G->ev[0], G->st));
    FL_RC(G->upload(G->par, dpar.data(), dpar.size() * sizeof(DParam)));
    FL_RC(G->upload(G->gram, gram.data(), gram.size() * 2));
    FL_RC(G->upload(G->reads, reads, rbytes));
    FL_RC(G->pack(G->reads, rbytes, G->read_pk, G->read_odd));
    FL_RC(G->upload(G->roff, read_off, n_reads * 8));
    FL_RC(G->upload(G->rlen, read_len, n_reads * 2));
    FL_RC(G->upload(G->pid, pid.data(), n_reads * 2));
    FL_RC(G->upload(G->list_base, list_base.data(), (n_reads + 1) * 4));
    FL_RC(G->list_cnt.ensure((nl + 1) * 4));
    FL_RC(G->list_lo.ensure((nl + 1) * 4));
    FL_RC(G->list_start.ensure((nl + 1) * 4));
    FArgs a{};
    a.qix = G->dq.as<DQ>();
    a.par = G->par.as<DParam>();
    a.gram = G->gram.as<uint16_t>();
    a.genome = G->genome.as<char>();
    a.glen = G->glen;
    a.reads = G->reads.as<char>();
    a.read_pk = G->read_pk.as<uint32_t>();
    a.read_odd = G->read_odd.as<uint32_t>();
    a.gen_pk = G->gen_pk.as<uint32_t>();
    a.gen_odd = G->gen_odd.as<uint32_t>();
    a.roff = G->roff.as<uint64_t>();
    a.rlen = G->rlen.as<uint16_t>();
    a.pid = G->pid.as<uint16_t>();
    a.n_reads = (uint32_t)n_reads;
    a.cv = (uint32_t)chunk_value;
    a.list_base = G->list_base.as<uint32_t>();
    a.list_cnt = G->list_cnt.as<uint32_t>();
    a.list_lo = G->list_lo.as<uint32_t>();
    a.list_start = G->list_start.as<uint32_t>();
    // per strand: the device's entries and perfect hits for the batch pass, which
    // runs on the host once both strands' device work is done (the two strands'
    // passes side by side)
    std::vector<uint32_t> meta_s[2];
    std::vector<int32_t> pos_s[2], perf_s[2];
    std::vector<int8_t> flag_s[2];
    for (int dr : {0, 4}) {
        if (!(strands & (dr ? 2 : 1))) continue;
        a.dr = dr;
        G->last_lists += nl;
        // reads per block: CREADS while that fills the chip twice over, fewer below
        const uint32_t per = (uint32_t)std::min<size_t>(CREADS, std::max<size_t>(4, n_reads / 512));
        const unsigned grid = (unsigned)((n_reads + per - 1) / per);
        FL_TRY(hipMemsetAsync(a.list_cnt + nl, 0, 4, G->st));
        hipLaunchKernelGGL(fl_count, dim3(grid), dim3(FB), 0, G->st, a, per);
        FL_TRY(hipGetLastError());
        size_t tmp = 0;
        FL_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, a.list_cnt, G->list_start.as<uint32_t>(),
                                                (int)(nl + 1), G->st));
        FL_RC(G->cub_tmp.ensure(tmp));
        FL_TRY(hipcub::DeviceScan::ExclusiveSum(G->cub_tmp.p, tmp, a.list_cnt,
                                                G->list_start.as<uint32_t>(), (int)(nl + 1), G->st));
        uint32_t total = 0;
        FL_TRY(hipMemcpyAsync(&total, G->list_start.as<uint32_t>() + nl, 4, hipMemcpyDeviceToHost,
                              G->st));
        FL_TRY(hipStreamSynchronize(G->st));
        G->last_flat += total;
        FL_RC(G->flat.ensure((size_t)total * 4 + 4));
        a.flat = G->flat.as<uint32_t>();
        hipLaunchKernelGGL(fl_fill, dim3(grid), dim3(FB), 0, G->st, a, per);
        FL_TRY(hipGetLastError());

        std::vector<uint32_t> &meta = meta_s[dr ? 1 : 0];
        std::vector<int32_t> &pos = pos_s[dr ? 1 : 0], &perf = perf_s[dr ? 1 : 0];
        std::vector<int8_t> &flag = flag_s[dr ? 1 : 0];
        FL_RC(G->pair(a, false, nullptr, (uint32_t)n_reads, ECAP, PCAP, meta, pos, flag, perf));
        // reads that outgrew the LDS slots run again with slots in HBM
        std::vector<uint32_t> over;
        for (size_t r = 0; r < n_reads; ++r)
            if (meta[3 * r + 2] == OVERFLOW_MARK) over.push_back((uint32_t)r);
        G->last_overflow += over.size();
        // (65534: a count word of 0xFFFF | 0xFFFF << 16 would read as the overflow mark)
        for (uint32_t cap : {1024u, 65534u}) {
            if (over.empty()) break;
            const size_t per = std::max<size_t>(1, ((size_t)256 << 20) / ((size_t)cap * 9));
            std::vector<uint32_t> still;
            for (size_t b = 0; b < over.size(); b += per) {
                const uint32_t m = (uint32_t)std::min(per, over.size() - b);
                std::vector<uint32_t> m2;
                std::vector<int32_t> p2, q2;
                std::vector<int8_t> f2;
                FL_RC(G->pair(a, true, over.data() + b, m, cap, cap, m2, p2, f2, q2));
                const uint32_t es = (uint32_t)pos.size(), ps = (uint32_t)perf.size();
                pos.insert(pos.end(), p2.begin(), p2.end());
                flag.insert(flag.end(), f2.begin(), f2.end());
                perf.insert(perf.end(), q2.begin(), q2.end());
                for (uint32_t t = 0; t < m; ++t) {
                    const uint32_t r = over[b + t];
                    if (m2[3 * t + 2] == OVERFLOW_MARK) {
                        still.push_back(r);
                        continue;
                    }
                    meta[3 * r + 0] = es + m2[3 * t + 0];
                    meta[3 * r + 1] = ps + m2[3 * t + 1];
                    meta[3 * r + 2] = m2[3 * t + 2];
                }
            }
            over.swap(still);
        }
        if (!over.empty())
            return srm::set_error(SRM_ENOMEM, "read %u holds more than 65534 filter entries",
                                  over[0]);
        FL_TRY(hipEventRecord(G->ev[1], G->st));
        FL_TRY(hipEventSynchronize(G->ev[1]));
        FL_TRY(hipEventElapsedTime(&G->last_ms, G->ev[0], G->ev[1]));
    }
    auto pass = [&](int x) {
        *(x ? out_rev : out_fwd) =
            batch_pass(MetaAcc{meta_s[x], pos_s[x], flag_s[x], perf_s[x]}, n_reads, read_len,
                       read_k, G->glen, blocked, chunk_value);
    };
    if ((strands & 3) == 3) {
        std::thread other;
        try {
            other = std::thread(pass, 1);
        } catch (...) {   // no thread to be had: both passes on this one
            pass(1);
        }
        pass(0);
        if (other.joinable()) other.join();
    } else {
        pass((strands & 1) ? 0 : 1);
    }
    return SRM_OK;
}

}  // namespace

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
        return rc;
    };
    if (hipSetDevice(G->device) != hipSuccess ||
        hipEventCreate(&G->ev[0]) != hipSuccess || hipEventCreate(&G->ev[1]) != hipSuccess)
        return fail(srm::set_error(SRM_EDEVICE, "event creation failed"));
    int rc = G->upload(G->genome, genome, glen);
    if (!rc) rc = G->pack(G->genome, glen, G->gen_pk, G->gen_odd);
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
    const int rc = run_device(G, blocked, reads, read_off, read_len, read_k, n_reads,
                              do_reverse ? 2 : 1, chunk_value, &F, &F);
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
    *out_fwd = nullptr;
    *out_rev = nullptr;
    if (!G || chunk_value < 1) return srm::set_error(SRM_EINVAL, "bad filter arguments");
    if (n_reads == 0) {
        *out_fwd = new srm_filter();
        *out_rev = new srm_filter();
        return SRM_OK;
    }
    srm_filter *Ff = nullptr, *Fr = nullptr;
    const int rc = run_device(G, blocked, reads, read_off, read_len, read_k, n_reads, 3,
                              chunk_value, &Ff, &Fr);
    if (rc != SRM_OK) {
        delete Ff;
        delete Fr;
        return rc;
    }
    *out_fwd = Ff;
    *out_rev = Fr;
    return SRM_OK;
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
    (void)hipStreamSynchronize(G->st);
    delete G;
}

}  // extern "C"
