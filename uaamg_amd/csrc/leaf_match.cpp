// Host side of the leaf matching (leaf_match.h).
#include "leaf_match.h"

#include <cstring>

#include "leaf_topology.h"

namespace uaamg {

namespace {

int table_bits(int64_t n) {   // load at most 1/2, as LeafLookup
    int bits = 4;
    while ((int64_t(1) << bits) < 2 * n) ++bits;
    return bits;
}

size_t aligned(size_t b) { return (b + 255) & ~size_t(255); }

}  // namespace

int LeafMatch::add(int64_t n, const int32_t* origins) {
    for (size_t i = 0; i < src_.size(); ++i)
        if (src_[i].n == n &&
            (n == 0 || src_[i].origins == origins || !std::memcmp(src_[i].origins, origins, size_t(n) * 12)))
            return int(i);
    src_.push_back({n, origins});
    return int(src_.size()) - 1;
}

size_t LeafMatch::bytes() const {
    size_t b = 256;
    for (const Src& r : src_) b += aligned(size_t(r.n) * 12) + aligned((size_t(1) << table_bits(r.n)) * 12);
    return b;
}

hipError_t LeafMatch::build(char* mem, hipStream_t s) {
    if (src_.size() > size_t(kMatchSets)) return hipErrorInvalidValue;
    // [bad][tables][origins]: one fill empties the tables and the flag
    sets_ = MatchSets{};
    sets_.nset = int32_t(src_.size());
    sets_.bad = reinterpret_cast<int32_t*>(mem);
    char* at = mem + 256;
    for (size_t i = 0; i < src_.size(); ++i) {
        MatchSet& m = sets_.set[i];
        const int bits = table_bits(src_[i].n);
        m.n = src_[i].n;
        m.mask = (uint64_t(1) << bits) - 1;
        m.shift = 64 - bits;
        m.keys = reinterpret_cast<uint64_t*>(at);
        m.vals = reinterpret_cast<int32_t*>(m.keys + m.mask + 1);
        at += aligned((m.mask + 1) * 12);
    }
    if (hipError_t e = hipMemsetAsync(mem, 0xff, size_t(at - mem), s)) return e;
    for (size_t i = 0; i < src_.size(); ++i) {
        sets_.set[i].origins = reinterpret_cast<int32_t*>(at);
        const size_t b = size_t(src_[i].n) * 12;
        if (b)
            if (hipError_t e = hipMemcpyAsync(at, src_[i].origins, b, hipMemcpyHostToDevice, s)) return e;
        at += aligned(b);
    }
    return launch_match_build(sets_, s);
}

hipError_t LeafMatch::query(int from, const std::vector<MatchColumn>& cols, int32_t* tab, hipStream_t s) const {
    if (cols.size() > size_t(kMatchCols)) return hipErrorInvalidValue;
    MatchQuery q{};
    q.from = from;
    q.ncol = int32_t(cols.size());
    q.tab = tab;
    for (size_t i = 0; i < cols.size(); ++i) q.col[i] = cols[i];
    return launch_match_query(sets_, q, s);
}

bool bad_origins(int64_t n, const int32_t* origins, LeafLookup& lookup, bool* misaligned) {
    std::vector<Coord> o(static_cast<size_t>(n));
    for (int64_t i = 0; i < n; ++i) {
        o[size_t(i)] = {origins[3 * i], origins[3 * i + 1], origins[3 * i + 2]};
        if ((o[size_t(i)].x | o[size_t(i)].y | o[size_t(i)].z) & 7) {
            *misaligned = true;
            return true;
        }
    }
    *misaligned = false;
    lookup.build(o);
    for (size_t i = 0; i < o.size(); ++i)
        if (lookup.find(o[i]) != int32_t(i)) return true;
    return false;
}

bool bad_origins(int64_t n, const int32_t* origins, bool* misaligned) {
    LeafLookup lookup;
    return bad_origins(n, origins, lookup, misaligned);
}

}  // namespace uaamg
