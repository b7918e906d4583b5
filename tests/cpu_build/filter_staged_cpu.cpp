// filter_pair_cpu.cpp's checks with every read's list starts and elements staged as
// fl_pair stages them in LDS, cut short at several sizes: what lies beyond comes from
// the flat array.
#include <algorithm>
#include <vector>

#include "filter_internal.h"
#include "filter_pair.h"

namespace srm_pair {

inline void staged_seashore(const FArgs &a, uint32_t r, Store &s)
{
    static const uint32_t caps[][2] = {{33, 64}, {1, 1}, {5, 3}, {0, 64}, {33, 0}, {2, 200}};
    const DParam P = a.par[a.pid[r]];
    const uint32_t *cap = caps[r % 6];
    ReadLists ls{a, a.list_base[r]};
    const uint32_t i0 = ls.start(0), end = ls.start(P.n);
    std::vector<uint32_t> starts, vals;   // exactly sized
    for (uint32_t x = 0; x < std::min<uint32_t>((uint32_t)P.n + 1, cap[0]); ++x) starts.push_back(ls.start((int)x));
    for (uint32_t i = 0; i < std::min(end - i0, cap[1]); ++i) vals.push_back(a.flat[i0 + i]);
    starts.shrink_to_fit();
    vals.shrink_to_fit();
    seashore(a, r, s, ReadLists{a, a.list_base[r], starts.data(), (uint32_t)starts.size(), vals.data(),
                                i0, (uint32_t)vals.size()});
}

}  // namespace srm_pair

#define seashore staged_seashore
#include "filter_pair_cpu.cpp"
