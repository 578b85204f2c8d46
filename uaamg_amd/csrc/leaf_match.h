// Matching leaves of one grid to leaves of others by origin, on the device, for
// the length of one call: every set of origins goes into an open-addressing
// table (the packing and hash of LeafLookup), and a query writes, per leaf of
// one set, the leaf of another set at its origin or one leaf beside it.
//
// The host tables this replaced took most of the calls that use them (a hash
// insert and up to twenty finds per leaf, one thread): right-hand side and
// pressure gradient together 3.06 ms at 13115 leaves, 1.95 with the matching here.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

namespace uaamg {

class LeafLookup;

constexpr int kMatchSets = 8;    // different sets of origins of one call
constexpr int kMatchCols = 20;   // columns of one query

struct MatchSet {
    const int32_t* origins;   // [n][3]
    int64_t n;
    uint64_t* keys;           // all ones: empty
    int32_t* vals;
    uint64_t mask;
    int32_t shift;
};

struct MatchSets {
    MatchSet set[kMatchSets];
    int32_t nset;
    int32_t* bad;   // -1, or 1 where an origin is no multiple of 8 or comes twice in a set
};

struct MatchColumn {
    int32_t set;     // < 0: matches nothing
    int32_t d[3];    // voxels from the leaf's origin
};

struct MatchQuery {
    int32_t from, ncol;
    int32_t* tab;    // [n of from][ncol], -1: no such leaf
    MatchColumn col[kMatchCols];
};

hipError_t launch_match_build(const MatchSets& s, hipStream_t stream);
hipError_t launch_match_query(const MatchSets& s, const MatchQuery& q, hipStream_t stream);

// The sets of one call. Arrays of equal content share a set, so each is
// uploaded and inserted once.
class LeafMatch {
public:
    // set of a host array of n origins; the array is read until the stream has run what build() issues
    int add(int64_t n, const int32_t* origins);
    size_t bytes() const;   // device memory that build() lays out
    int64_t leaves(int set) const { return int64_t(src_[size_t(set)].n); }
    hipError_t build(char* mem, hipStream_t s);
    hipError_t query(int from, const std::vector<MatchColumn>& cols, int32_t* tab, hipStream_t s) const;
    const int32_t* bad() const { return sets_.bad; }

private:
    struct Src {
        int64_t n;
        const int32_t* origins;
    };
    std::vector<Src> src_;
    MatchSets sets_{};
};

// The refusal of a grid's origins (misaligned, then duplicate), or false with
// the grid's lookup built
bool bad_origins(int64_t n, const int32_t* origins, LeafLookup& lookup, bool* misaligned);
bool bad_origins(int64_t n, const int32_t* origins, bool* misaligned);

}  // namespace uaamg
