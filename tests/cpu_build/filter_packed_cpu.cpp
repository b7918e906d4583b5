// CPU build of the packed-code helpers of the device filter (filter_pair.h: pack16,
// codes16, codes32, odd32, gram_code, gram_offset, same16), with exactly the words the device arrays
// hold, against a byte-by-byte reading of the same bases: every q-gram of reads of
// 1..300 bases at every alignment, q 1..31, both strands, with other bytes mixed in,
// and every 16-base step of reads against genome stretches equal to them or one
// byte off.
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "filter_internal.h"
#include "filter_pair.h"

using namespace srm_filter_impl;
using namespace srm_pair;

namespace {

struct Packed {
    std::vector<uint32_t> pk, odd;
    explicit Packed(const std::string &s)
    {
        const size_t n16 = (s.size() + 15) / 16;
        std::vector<uint32_t> bytes(n16 * 4, 0);
        std::memcpy(bytes.data(), s.data(), s.size());
        pk.assign(n16 + 2, 0);                       // two words past the last
        std::vector<uint16_t> o16((n16 + 3) / 2 * 2 + 2, 0);   // and a mask word
        for (size_t i = 0; i < n16; ++i) {
            const uint32_t w[4] = {bytes[4 * i], bytes[4 * i + 1], bytes[4 * i + 2], bytes[4 * i + 3]};
            uint32_t o;
            pk[i] = pack16(w, o);
            o16[i] = (uint16_t)o;
        }
        odd.resize(o16.size() / 2);
        std::memcpy(odd.data(), o16.data(), odd.size() * 4);
    }
};

uint64_t g_state;
uint64_t next()
{
    g_state ^= g_state << 13;
    g_state ^= g_state >> 7;
    g_state ^= g_state << 17;
    return g_state;
}

std::string random_bases(size_t n, unsigned other)   // one byte in `other` is no base
{
    static const char others[] = "NacgtR\0\xff@B";
    std::string s(n, 'A');
    for (char &c : s) c = other && next() % other == 0 ? others[next() % 10] : "ACGT"[next() & 3];
    return s;
}

}  // namespace

int main()
{
    g_state = 88172645463325252ull;
    size_t checks = 0;
    for (int round = 0; round < 400; ++round) {
        const unsigned other = round % 4 == 0 ? 0 : 3 + (unsigned)(next() % 60);
        const int L = 1 + (int)(next() % 300);
        const size_t at = next() % 70;
        const std::string buf = random_bases(at + (size_t)L, other);
        const Packed P(buf);
        const char *rd = buf.data() + at;
        for (int dr : {0, 4})
            for (int q = 1; q <= 31 && q <= L; ++q)
                for (int g = 0; g + q <= L; ++g) {
                    uint64_t want = 0, got = 0;
                    bool other_byte = false;
                    for (int i = 0; i < q; ++i) {
                        const int c = dcode(obyte(rd, L, dr, g + i));
                        other_byte |= c < 0;
                        want = (want << 2) | (uint64_t)(c & 3);
                    }
                    const bool ok = gram_code(P.pk.data(), P.odd.data(), at, L, dr, q, g, got);
                    if (ok == other_byte || (ok && got != want)) {
                        printf("MISMATCH L=%d at=%zu dr=%d q=%d g=%d\n", L, at, dr, q, g);
                        return 1;
                    }
                    ++checks;
                }
    }
    for (int round = 0; round < 20000; ++round) {
        const unsigned other = round % 3 == 0 ? 0 : 2 + (unsigned)(next() % 60);
        const int L = 1 + (int)(next() % 90);
        const size_t at = next() % 40, S = next() % 70;
        const int dr = round & 1 ? 4 : 0;
        const std::string reads = random_bases(at + (size_t)L, other);
        std::string genome = random_bases(S + (size_t)L, other);
        for (int j = 0; j < L; ++j) genome[S + (size_t)j] = obyte(reads.data() + at, L, dr, j);
        if (next() % 2) genome[S + next() % (size_t)L] = random_bases(1, 2)[0];
        const Packed R(reads), G(genome);
        FArgs a{};
        a.reads = reads.data();
        a.genome = genome.data();
        a.read_pk = R.pk.data();
        a.read_odd = R.odd.data();
        a.gen_pk = G.pk.data();
        a.gen_odd = G.odd.data();
        for (int x = 0; 16 * x < L; ++x) {
            bool want = true;
            for (int j = 16 * x; j < L && j < 16 * x + 16; ++j)
                want &= genome[S + (size_t)j] == obyte(reads.data() + at, L, dr, j);
            if (same16(a, at, L, dr, S, x) != want) {
                printf("MISMATCH same16 L=%d at=%zu S=%zu dr=%d x=%d\n", L, at, S, dr, x);
                return 1;
            }
            ++checks;
        }
    }
    for (int L = 1; L <= 400; ++L)
        for (int k = 0; k <= 40; ++k) {
            const Params p = derive(L, k);
            for (int x = 0; x < p.n; ++x)
                if (gram_offset(L, p.q, x) != p.gram[(size_t)x]) {
                    printf("MISMATCH gram L=%d k=%d x=%d\n", L, k, x);
                    return 1;
                }
        }
    printf("OK %zu\n", checks);
    return 0;
}
