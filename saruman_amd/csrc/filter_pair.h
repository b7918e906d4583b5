// filter_pair.h -- the per-read part of the q-gram filter as host/device code:
// q-gram lookup in the device copy of the index, run_seashore's pairing
// (src/hash.c:502-834) and add_start_position (src/hash.c:40-178) over the flat
// position-list array.  Compiled into the kernels of filter_gpu.hip; the same
// functions also compile for the host, which lets a CPU build check the
// kernels' indexing.
#pragma once

#include <stdint.h>

#include <vector>

#include "filter_internal.h"

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define SRM_HD __host__ __device__
#else
#define SRM_HD
#endif

namespace srm_pair {

constexpr uint32_t OVERFLOW_MARK = 0xFFFFFFFFu;

struct DQ {                  // one q's index on the device
    const uint64_t *keys;    // (code << pos_bits) | offset, ascending
    const uint32_t *pre;     // [4^pre_bases + 1] key ranges by the first bases
    const uint64_t *odd_hash;   // FNV-1a of the q-gram text, ascending, then offset
    const uint32_t *odd_pos;
    uint32_t n_odd;
    int q, pos_bits, pre_bases;
};

struct DParam {
    int L, k, q, rest, n, half, exact;
    uint32_t gram_off;       // into FArgs::gram (no kernel reads it: gram_offset)
};

struct FArgs {
    const DQ *qix;           // [32], indexed by q
    const DParam *par;
    const uint16_t *gram;    // for checks on the host, as rlen: the kernels take neither
    const char *genome;
    uint64_t glen;
    const char *reads;
    const uint64_t *roff;
    const uint16_t *rlen;
    const uint16_t *pid;
    uint32_t n_reads;
    int dr;                  // 0 forward, 4 reverse
    uint32_t cv;             // chunk_value
    const uint32_t *list_base;   // [n_reads + 1] first list of every read
    uint32_t *list_cnt;          // [n_lists + 1] list length + 1 (terminator)
    uint32_t *list_lo;           // [n_lists] first key of the list (NO_RANGE: search again)
    const uint32_t *list_start;  // [n_lists + 1] exclusive sum of list_cnt
    uint32_t *flat;
    // pairing
    const uint32_t *todo;    // reads to pair; null = all reads
    uint32_t n_todo;
    bool packed;             // entries one after another instead of at the reads' places
    int32_t *slot_pos;       // HBM slots (second and later passes)
    int8_t *slot_flag;
    int32_t *slot_perf;
    uint32_t cap, pcap;
    uint32_t *counters;      // [3] compact entries / perfect hits written so far, overflows
    int32_t *out_pos;
    int8_t *out_flag;
    int32_t *out_perf;
    uint32_t *meta;          // [3 * n_reads]: ent_off, perf_off, n_ent | n_perf << 16
    // the reads' bytes as 2-bit codes and as a mask of the bytes other than ACGT
    // (pack16), at the same offsets
    const uint32_t *read_pk;
    const uint32_t *read_odd;
    const uint32_t *gen_pk;      // the genome's, likewise
    const uint32_t *gen_odd;
    // list_start[0]: nonzero where another strand's lists come before in one sum.
    // Offsets into flat count from it, modulo 2^32
    uint32_t list_org;
    uint32_t *over;              // reads that outgrew their slots (counters[2] of them)
};

// where list i starts in flat
SRM_HD inline uint32_t list_at(const FArgs &a, uint64_t i) { return a.list_start[i] - a.list_org; }

// The starts are sums modulo 2^32, and so is a strand's total, which says whether its
// lists fit: a total past 2^32 may say so wrongly.  Until the true sum passes 2^32 every
// start is true, so the list at which it does is one that ends past any room below 2^32:
// a list that does not fit where the total does means that the total is not true.  A
// strand's room is at most MAX_FLAT elements (a wave's steps past the last one must not
// wrap either)
constexpr uint64_t MAX_FLAT = 0xFFFFFF00ull;
SRM_HD inline bool list_fits(uint32_t at, uint32_t len, uint64_t room) { return (uint64_t)at + len <= room; }

SRM_HD inline char dcomp(char c)
{
    switch (c) {
    case 'A': return 'T';
    case 'C': return 'G';
    case 'G': return 'C';
    case 'T': return 'A';
    default: return c;
    }
}

SRM_HD inline int dcode(char c)
{
    switch (c) {
    case 'A': return 0;
    case 'C': return 1;
    case 'G': return 2;
    case 'T': return 3;
    default: return -1;
    }
}

// byte j of the read as the filter sees it (reverse complement for strand 4,
// util.c:35-57)
SRM_HD inline char obyte(const char *rd, int L, int dr, int j)
{
    return dr ? dcomp(rd[L - 1 - j]) : rd[j];
}

// 16 bytes as 16 codes, the first in the top two bits (q-gram codes are read as
// numbers with the first base most significant); a byte other than ACGT gives some
// code and sets its bit (byte i: bit i) in odd
SRM_HD inline uint32_t pack16(const uint32_t (&w)[4], uint32_t &odd)
{
    uint32_t pk = 0;
    odd = 0;
    for (int i = 0; i < 16; ++i) {
        const uint32_t c = (w[i >> 2] >> (8 * (i & 3))) & 0xFFu;
        const uint32_t x = (c >> 1) & 3u, code = x ^ (x >> 1);   // A 0, C 1, G 2, T 3
        pk = (pk << 2) | code;
        odd |= (uint32_t)(((0x54474341u >> (8 * code)) & 0xFFu) != c) << i;
    }
    return pk;
}

// 32 codes from code index o, the first in the top bits (words o >> 4 .. + 2)
SRM_HD inline uint64_t codes32(const uint32_t *pk, uint64_t o)
{
    const uint32_t *p = pk + (o >> 4);
    const int sh = 2 * (int)(o & 15);
    const uint64_t x = ((uint64_t)p[0] << 32) | p[1];
    return sh ? (x << sh) | (p[2] >> (32 - sh)) : x;
}

// 32 mask bits from index o (words o >> 5, + 1)
SRM_HD inline uint32_t odd32(const uint32_t *odd, uint64_t o)
{
    const uint32_t *p = odd + (o >> 5);
    return (uint32_t)((((uint64_t)p[1] << 32) | p[0]) >> (o & 31));
}

// the 32 codes of x in reverse order
SRM_HD inline uint64_t reverse_codes(uint64_t x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    x = __brevll(x);
    return ((x >> 1) & 0x5555555555555555ull) | ((x & 0x5555555555555555ull) << 1);
#else
    x = __builtin_bswap64(x);
    x = ((x >> 4) & 0x0F0F0F0F0F0F0F0Full) | ((x & 0x0F0F0F0F0F0F0F0Full) << 4);
    return ((x >> 2) & 0x3333333333333333ull) | ((x & 0x3333333333333333ull) << 2);
#endif
}

// the code of the q-gram (q <= 31) at offset g of the read at byte `at`, L bases, as
// strand dr sees it; false when it holds another byte
SRM_HD inline bool gram_code(const uint32_t *pk, const uint32_t *odd, uint64_t at, int L, int dr,
                             int q, int g, uint64_t &code)
{
    const uint64_t o = at + (uint64_t)(dr ? L - g - q : g);
    const uint64_t x = codes32(pk, o);
    if (odd32(odd, o) & ((1u << q) - 1u)) return false;
    code = dr ? reverse_codes(~x) & (((uint64_t)1 << (2 * q)) - 1) : x >> (64 - 2 * q);
    return true;
}

// 16 codes from code index o, the first in the top bits (words o >> 4, + 1)
SRM_HD inline uint32_t codes16(const uint32_t *pk, uint64_t o)
{
    const uint32_t *p = pk + (o >> 4);
    return (uint32_t)(((((uint64_t)p[0] << 32) | p[1]) << (2 * (o & 15))) >> 32);
}

// bases 16x .. of the read (at most 16, to its end) as strand dr sees it against the
// genome's from S + 16x: equal as bytes.  at: the read's first byte in a.reads.
SRM_HD inline bool same16(const FArgs &a, uint64_t at, int L, int dr, uint64_t S, int x)
{
    const int j = 16 * x, m = L - j < 16 ? L - j : 16;
    const uint64_t o = at + (uint64_t)(dr ? L - j - m : j);
    const uint32_t some = (uint32_t)((1ull << m) - 1u);
    // all words before the first test: one wait for memory
    uint32_t c = codes16(a.read_pk, o);
    const uint32_t g = codes16(a.gen_pk, S + (uint64_t)j);
    if ((odd32(a.read_odd, o) | odd32(a.gen_odd, S + (uint64_t)j)) & some) {
        for (int t = 0; t < m; ++t)
            if (a.genome[S + (uint64_t)(j + t)] != obyte(a.reads + at, L, dr, j + t)) return false;
        return true;
    }
    if (dr)   // the m codes complemented and in reverse order, the first on top again
        c = (uint32_t)(reverse_codes(~(uint64_t)c << 32)) << (2 * (16 - m));
    return ((c ^ g) >> (2 * (16 - m))) == 0u;
}

// offset of q-gram list x: ascending from the read's start, then, when q does not
// divide L, descending from its end (saruman.c:42-75)
SRM_HD inline int gram_offset(int L, int q, int x)
{
    const int m = L / q;
    return x < m ? x * q : L - (x - m + 1) * q;
}

// FNV-1a, 64 bit
SRM_HD inline uint64_t fnv_step(uint64_t h, unsigned char c)
{
    return (h ^ c) * 1099511628211ull;
}
constexpr uint64_t FNV_BASIS = 14695981039346656037ull;

// list_lo of a q-gram whose positions are not one run of keys (it holds a byte
// other than ACGT: its positions come from the hash table and a byte compare)
constexpr uint32_t NO_RANGE = 0xFFFFFFFFu;

// the run of keys of the q-gram `code`: its length, the first one's index in lo
SRM_HD inline uint32_t lookup_code(const DQ &X, uint64_t code, uint32_t &lo)
{
    const uint64_t p = code >> (2 * (X.q - X.pre_bases));
    lo = X.pre[p];
    const uint32_t end = X.pre[p + 1];
    uint32_t hi = end;
    const uint64_t key = code << X.pos_bits;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (X.keys[mid] < key) lo = mid + 1;
        else hi = mid;
    }
    uint32_t i = lo;
    while (i < end && (X.keys[i] >> X.pos_bits) == code) ++i;
    return i - lo;
}

// positions of the q-gram at read offset g, ascending; writes them to out when
// FILL, returns their number; lo_out (when given) receives the index of the first
// key (the positions are keys lo .. lo + count - 1), or NO_RANGE for a q-gram
// holding another byte
template <bool FILL>
SRM_HD uint32_t lookup(const DQ &X, const char *genome, const char *rd, int L, int dr, int g,
                       uint32_t *out, uint32_t *lo_out = nullptr)
{
    const int q = X.q;
    uint64_t code = 0;
    bool odd = false;
    // all q bytes, with no exit from the loop (on gfx950 a loop that left at the
    // first other byte gave fl_count wrong list lengths for some lanes once the key
    // range was stored as well; the same source on the host gave the right ones)
    for (int i = 0; i < q; ++i) {
        const int c = dcode(obyte(rd, L, dr, g + i));
        odd |= c < 0;
        code = (code << 2) | (uint64_t)(c & 3);
    }
    uint32_t cnt = 0;
    if (odd) {
        if (lo_out) *lo_out = NO_RANGE;
        uint64_t h = FNV_BASIS;
        for (int i = 0; i < q; ++i) h = fnv_step(h, (unsigned char)obyte(rd, L, dr, g + i));
        uint32_t lo = 0, hi = X.n_odd;
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (X.odd_hash[mid] < h) lo = mid + 1;
            else hi = mid;
        }
        for (uint32_t i = lo; i < X.n_odd && X.odd_hash[i] == h; ++i) {
            const uint32_t p = X.odd_pos[i];
            bool same = true;
            for (int t = 0; t < q && same; ++t) same = genome[p + t] == obyte(rd, L, dr, g + t);
            if (same) {
                if (FILL) out[cnt] = p;
                ++cnt;
            }
        }
        return cnt;
    }
    uint32_t lo;
    cnt = lookup_code(X, code, lo);
    if (lo_out) *lo_out = lo;
    if (FILL) {
        const uint64_t mask = ((uint64_t)1 << X.pos_bits) - 1;
        for (uint32_t i = 0; i < cnt; ++i) out[i] = (uint32_t)(X.keys[lo + i] & mask);
    }
    return cnt;
}

// a read's result-hash entries (pos, flag) and printed perfect hits
struct Store {
    int32_t *pos;
    int8_t *flag;
    int32_t *perf;
    uint32_t stride, cap, pcap;
    uint32_t n = 0, np = 0;
    bool ovf = false;
    SRM_HD int32_t &P(uint32_t i) { return pos[i * stride]; }
    SRM_HD int8_t &F(uint32_t i) { return flag[i * stride]; }
    SRM_HD int32_t &Q(uint32_t i) { return perf[i * stride]; }
    SRM_HD void push(int32_t p, int f)
    {
        if (n == cap) {
            ovf = true;
            return;
        }
        P(n) = p;
        F(n) = (int8_t)f;
        ++n;
    }
};

// A read's lists (lb: its first): list x starts at flat index start(x), and val(i) is
// the flat array's element i.  A kernel holds the first n_starts starts and the n_vals
// elements from index v0 in LDS; the rest, and elements of later reads that a scan
// runs into (Q12), are read from HBM.
struct ReadLists {
    const FArgs &a;
    uint32_t lb;
    const uint32_t *starts = nullptr;
    uint32_t n_starts = 0;
    const uint32_t *vals = nullptr;
    uint32_t v0 = 0, n_vals = 0;
    SRM_HD uint32_t start(int x) const { return (uint32_t)x < n_starts ? starts[x] : list_at(a, lb + (uint32_t)x); }
    SRM_HD uint32_t val(uint32_t i) const { return i - v0 < n_vals ? vals[i - v0] : a.flat[i]; }
};

// first index of the ascending run of elements [lo, hi) whose value is >= u
SRM_HD inline uint32_t run_lower(const ReadLists &ls, uint32_t lo, uint32_t hi, uint32_t u)
{
    while (lo < hi) {
        const uint32_t m = lo + ((hi - lo) >> 1);
        if (ls.val(m) < u) lo = m + 1;
        else hi = m;
    }
    return lo;
}

// The pair passes' matches of one list in the reference's scan order.  The scan
// compares every target tg(err), err = -lim .. lim, with the ascending run
// [lo, min(hi, end)) of elements -- cut at its first 0, as the reference's 0-terminated
// scans are -- and, in the first pass, first with one more value p0 (p0 == 0:
// none).  The targets are consecutive (ascending from t_lo when up, descending
// from t_hi otherwise), so the matches are the run's values in [t_lo, t_hi] found
// by one search and a walk, p0 merged in before a run value of the same target.
// Counts them into *hits and returns true when the count reaches need.
SRM_HD inline bool scan_run(const ReadLists &ls, uint32_t lo, uint32_t hi, uint32_t end,
                            int64_t t_lo, int64_t t_hi, bool up, uint32_t p0, int need, int &hits)
{
    if (t_hi < 0) return false;
    // positions are below 2^31, so the targets that one can equal fit 32 bits
    const uint32_t u_lo = t_lo > 0 ? (uint32_t)t_lo : 0u, u_hi = (uint32_t)t_hi;
    if (hi > end) hi = end;
    if (lo >= hi || ls.val(lo) == 0) hi = lo;    // an empty run
    bool p0_left = p0 != 0 && p0 >= u_lo && p0 <= u_hi;
    if (up) {
        uint32_t i = run_lower(ls, lo, hi, u_lo);
        for (;;) {
            const uint32_t v = i < hi ? ls.val(i) : 0xFFFFFFFFu;
            const bool run_next = v <= u_hi;
            if (p0_left && (!run_next || p0 <= v)) {
                p0_left = false;
                if (++hits == need) return true;
                continue;
            }
            if (!run_next) return false;
            if (++hits == need) return true;
            ++i;
        }
    }
    // descending (second pass only: no p0)
    uint32_t i = run_lower(ls, lo, hi, u_hi + 1u);
    while (i > lo && ls.val(i - 1) >= u_lo) {
        if (++hits == need) return true;
        --i;
    }
    return false;
}

// what entry (ep, ef) makes of a start (pos, flag): 1 rejected, 2 its flag is lowered,
// 0 the next entry decides
SRM_HD inline int entry_rule(int32_t ep, int ef, int32_t pos, int flag, int k)
{
    const int dir = flag > 3 ? 1 : 0, tdir = ef > 3 ? 1 : 0;
    const int64_t d1 = (int64_t)ep - pos, d2 = (int64_t)ep + pos;
    if (ef <= flag && ((d1 >= -k && d1 <= k) || (d2 >= -k && d2 <= k))) return 1;
    if (ep == pos && tdir == dir && ef > flag) return 2;
    return (ep == pos || ep == -pos) && tdir == dir ? 1 : 0;
}

// add_start_position, hash.c:40-178: 0 first entry, 1 rejected, 2 added or
// flag lowered.  |pos - e| <= k is the reference's scan of pos + i, i in [-k, k].
SRM_HD inline int add_start(Store &s, int32_t pos, int flag, int possible, int exact, int k)
{
    if (possible != exact) return 1;
    if (s.n == 0) {
        s.push(pos, flag);
        return 0;
    }
    for (uint32_t e = 0; e < s.n; ++e) {
        const int rule = entry_rule(s.P(e), s.F(e), pos, flag, k);
        if (rule == 2) s.F(e) = (int8_t)flag;
        if (rule) return rule;
    }
    s.push(pos, flag);
    return 2;
}

// the end of the position lists a read's list indexes may run into: its chunk's
SRM_HD inline uint32_t chunk_end(const FArgs &a, uint32_t r)
{
    const uint64_t next_chunk = ((uint64_t)(r / a.cv) + 1) * a.cv;
    return list_at(a, a.list_base[next_chunk < a.n_reads ? next_chunk : a.n_reads]);
}

// |v - (gs + d)| <= lim, for positions v and gs below 2^31 and gs + 1 above -2^16, 0 <= lim
// < 2^16: modulo 2^32 no other difference comes that near
SRM_HD inline bool near(uint32_t v, int64_t gs, int d, int lim)
{
    return v - (uint32_t)gs - (uint32_t)d + (uint32_t)lim <= 2u * (uint32_t)lim;
}

// the pair passes of one start position (hash.c:606-794): list aa's element off,
// value Pa, genome start gs + 1; lb: the read's first list.  Every match raises
// `possible` and calls add_start_position, which acts only when possible equals
// exact_tresh (Q13): the need-th match of the two passes in scan order, need =
// exact_tresh - 1, is the only one that can insert, and the scan stops there.
// True when there is one, with what it inserts.
SRM_HD inline bool pair_matches(const ReadLists &ls, const DParam &P, uint32_t flat_end, int aa,
                                uint32_t off, uint32_t Pa, int64_t gs, int32_t &hpos, int &hflag)
{
    const int q = P.q, half = P.half, k = P.k, L = P.L, dr = ls.a.dr;
    const bool fqm = (aa == 0);
    const int need = P.exact - 1;
    if (need < 1) return false;
    int hits = 0;
    // first pass, hash.c:606-692.  For every err the reference scans D(b, off), then
    // D(b, 1), D(b, 2), ... up to the next 0 (Q12): the element at a's index, then
    // one ascending run of list b (or of the list after b when b is empty).
    for (int b = aa + 1; b < half; ++b) {
        const uint32_t sb = ls.start(b), nb = ls.start(b + 1);
        const uint64_t at = (uint64_t)sb + off;
        const uint32_t P0 = at < flat_end ? ls.val((uint32_t)at) : 0u;
        if (P0 == 0) continue;                 // the scan never starts
        const int rstart = b * q + 1;
        const uint32_t lo = sb + 1;
        if (nb - sb == 2) {
            // a list of one element, nearly every list of a read that maps once: the scan
            // of the rest is empty
            if (!near(P0, gs, rstart, k) || ++hits != need) continue;
        }
        // list b from index 1, or the next list (b + 2 <= half + 1 <= P.n: the read's)
        else if (!scan_run(ls, lo, (lo < nb ? nb : ls.start(b + 2)) - 1, flat_end, gs + rstart - k,
                           gs + rstart + k, true, P0, need, hits))
            continue;
        if (b == half - 1 && fqm) {
            hflag = 1 + dr;
            hpos = (int32_t)(gs + 1);
        } else if (aa == half - 1) {
            hflag = ((int64_t)Pa + q > L ? 3 : 2) + dr;
            hpos = (int32_t)(gs - k + 1);
        } else if (fqm) {
            hflag = 1 + dr;
            hpos = (int32_t)(gs + 1);
        } else {
            hflag = 3 + dr;
            hpos = (int32_t)(gs - k + 1);
        }
        return true;
    }
    // second pass, hash.c:695-794: each err scans list half + j from its start up to
    // its 0; the targets gs + nin + err run downwards when j < a (the reference's err
    // is negated there)
    for (int j = 0; j < half; ++j) {
        const int lim = half - 1 - j - aa < 0 ? -(half - 1 - j - aa) : half - 1 - j - aa;
        const int nin = (half - j - 1) * q + 1 + P.rest;
        const uint32_t lo = ls.start(half + j), hi = ls.start(half + j + 1) - 1;
        if (lo == hi) continue;
        if (hi - lo == 1 && hi <= flat_end) {   // one element: either way the same
            const uint32_t v = ls.val(lo);
            if (v == 0 || !near(v, gs, nin, lim) || ++hits != need) continue;
        } else if (!scan_run(ls, lo, hi, flat_end, gs + nin - lim, gs + nin + lim, j - aa >= 0, 0u, need,
                      hits))
            continue;
        if (j == 0 && fqm) {
            hflag = 1 + dr;
            hpos = (int32_t)(gs + 1);
        } else if (j == 0) {
            hflag = (nin + q > L ? 3 : 2) + dr;
            hpos = (int32_t)(gs - k + 1);
        } else if (fqm) {
            hflag = 1 + dr;
            hpos = (int32_t)(gs + 1);
        } else {
            hflag = 3 + dr;
            hpos = (int32_t)(gs - k + 1);
        }
        return true;
    }
    return false;
}

// run_seashore of one read, its start positions one after another (the kernels
// take several at a time); ls: its lists
SRM_HD inline void seashore(const FArgs &a, uint32_t r, Store &s, const ReadLists &ls)
{
    const DParam P = a.par[a.pid[r]];
    const int L = P.L, dr = a.dr;
    const char *rd = a.reads + a.roff[r];
    const uint32_t flat_end = chunk_end(a, r);
    for (int aa = 0; aa < P.half; ++aa) {
        for (uint64_t off = 0;; ++off) {
            const uint64_t at = (uint64_t)ls.start(aa) + off;
            const uint32_t Pa = at < flat_end ? ls.val((uint32_t)at) : 0u;
            if (Pa == 0) break;
            const long gs = (long)Pa - ((long)aa * P.q + 1);
            if (gs + 1 <= 0) continue;
            // perfect check (strncpy + strcmp, hash.c:550-583)
            const long S = gs + 1;
            if ((uint64_t)S + (uint64_t)L <= a.glen) {
                bool perfect = true;
                const char *g = a.genome + S;
                for (int j = 0; j < L && perfect; ++j) perfect = g[j] == obyte(rd, L, dr, j);
                if (perfect && add_start(s, (int32_t)(-S), 0, P.exact, P.exact, P.k) != 1) {
                    if (s.np == s.pcap) s.ovf = true;
                    else s.Q(s.np++) = (int32_t)S;
                }
                if (s.ovf) return;
            }
            int32_t hpos;
            int hflag;
            if (pair_matches(ls, P, flat_end, aa, (uint32_t)off, Pa, gs, hpos, hflag)) {
                add_start(s, hpos, hflag, P.exact, P.exact, P.k);
                if (s.ovf) return;
            }
        }
    }
}

SRM_HD inline void seashore(const FArgs &a, uint32_t r, Store &s)
{
    seashore(a, r, s, ReadLists{a, a.list_base[r]});
}

// the device copies of the per-read parameter sets and their q-gram offsets
inline void device_params(const std::vector<srm_filter_impl::Params> &params,
                          std::vector<DParam> &dpar, std::vector<uint16_t> &gram)
{
    for (auto &p : params) {
        dpar.push_back({p.L, p.k, p.q, p.rest, p.n, p.half, p.exact_tresh, (uint32_t)gram.size()});
        for (int g : p.gram) gram.push_back((uint16_t)g);
    }
}

// the device copy of one q's index: the odd (non-ACGT) q-grams as (FNV-1a of
// the text, offset) pairs in ascending order
inline void odd_table(const srm_filter_impl::QIndex &X, std::vector<uint64_t> &hash,
                      std::vector<uint32_t> &pos)
{
    std::vector<std::pair<uint64_t, uint32_t>> odd;
    for (auto &kv : X.odd) {
        uint64_t h = FNV_BASIS;
        for (char c : kv.first) h = fnv_step(h, (unsigned char)c);
        for (uint32_t p : kv.second) odd.emplace_back(h, p);
    }
    std::sort(odd.begin(), odd.end());
    hash.resize(odd.size());
    pos.resize(odd.size());
    for (size_t t = 0; t < odd.size(); ++t) {
        hash[t] = odd[t].first;
        pos[t] = odd[t].second;
    }
}

}  // namespace srm_pair
