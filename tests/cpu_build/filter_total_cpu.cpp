// The device filter's test of whether a strand's lists fit (filter_pair.h: list_fits),
// over starts and totals modulo 2^32 as its scan leaves them: lists that fit the room are
// all taken; lists of 2^32 elements or more are found out whatever their total wraps to;
// and none is taken that ends past the room.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "filter_pair.h"

using namespace srm_pair;

static uint64_t state = 88172645463325252ull;
static uint32_t rnd()
{
    state ^= state << 13;
    state ^= state >> 7;
    state ^= state << 17;
    return (uint32_t)(state >> 20);
}

int main()
{
    long wrapped_totals = 0, taken = 0;
    for (int t = 0; t < 4000; ++t) {
        // a true total around m 2^32, of lists of 1 .. 2^24 elements
        const uint64_t m = rnd() % 4;
        uint64_t want = (m << 32) + (t % 5 == 0 ? rnd() % 3 - 1 : t % 2 ? rnd() : rnd() % 5000);
        if (want >> 40) want = 4096;   // (m = 0 and one below)
        std::vector<uint32_t> len;
        uint64_t sum = 0;
        while (sum < want) {
            const uint64_t x = 1 + rnd() % (1u << 24), left = want - sum;
            len.push_back((uint32_t)(x < left ? x : left));
            sum += len.back();
        }
        const uint32_t total = (uint32_t)sum, org = rnd();
        // room as the host makes it from the total it is told
        uint64_t room = (uint64_t)total + (t % 3 ? total / 8 : 0) + t % 7;
        if (room > MAX_FLAT) room = MAX_FLAT;
        if (total > room) continue;    // (told to be too many)
        uint32_t start = org;          // another strand's lists before, in one sum
        bool all = true;
        for (uint32_t n : len) {
            const uint32_t at = start - org;
            if (!list_fits(at, n, room)) all = false;
            else if ((uint64_t)at + n > room) return printf("a list outside the room\n"), 1;
            start += n;
        }
        if (sum > room && all) return printf("a total of %llu in a room of %llu\n", (unsigned long long)sum, (unsigned long long)room), 1;
        if (sum <= room && !all) return printf("lists that fit refused\n"), 1;
        (all ? taken : wrapped_totals) += 1;
    }
    printf("OK taken %ld wrapped %ld\n", taken, wrapped_totals);
    return taken > 100 && wrapped_totals > 1000 ? 0 : 1;
}
