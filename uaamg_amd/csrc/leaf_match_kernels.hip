// Kernels of the leaf matching (leaf_match.h). A few memory latencies each;
// at 13115 leaves 8 us for two sets and 6 us for twenty columns.
#include "leaf_match.h"
#include "leaf_topology.h"

namespace uaamg {
namespace {

constexpr int kThreads = 256;
constexpr uint64_t kEmpty = ~uint64_t(0);   // packed origins use 63 bits

__device__ __forceinline__ uint64_t slot_of(const MatchSet& m, uint64_t key) {
    return (key * 0x9E3779B97F4A7C15ull) >> m.shift;
}

// blockIdx.y: the set. A table is at most half full, so every probe ends.
__global__ __launch_bounds__(kThreads) void match_build_kernel(MatchSets s) {
    const MatchSet& m = s.set[blockIdx.y];
    const int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= m.n) return;
    const Coord o{m.origins[3 * i], m.origins[3 * i + 1], m.origins[3 * i + 2]};
    if ((o.x | o.y | o.z) & 7) {
        *s.bad = 1;
        return;
    }
    const uint64_t key = pack_origin(o);
    for (uint64_t h = slot_of(m, key);; h = (h + 1) & m.mask) {
        const uint64_t old = atomicCAS(reinterpret_cast<unsigned long long*>(m.keys + h), kEmpty, key);
        if (old == kEmpty) {
            m.vals[h] = int32_t(i);
            return;
        }
        if (old == key) {
            *s.bad = 1;
            return;
        }
    }
}

// blockIdx.y: the column
__global__ __launch_bounds__(kThreads) void match_query_kernel(MatchSets s, MatchQuery q) {
    const MatchSet& f = s.set[q.from];
    const int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= f.n) return;
    const MatchColumn& c = q.col[blockIdx.y];
    int32_t found = -1;
    if (c.set >= 0) {
        const MatchSet& m = s.set[c.set];
        const uint64_t key =
            pack_origin({f.origins[3 * i] + c.d[0], f.origins[3 * i + 1] + c.d[1], f.origins[3 * i + 2] + c.d[2]});
        for (uint64_t h = slot_of(m, key);; h = (h + 1) & m.mask) {
            const uint64_t k = m.keys[h];
            if (k == key) found = m.vals[h];
            if (k == key || k == kEmpty) break;
        }
    }
    q.tab[size_t(i) * q.ncol + blockIdx.y] = found;
}

}  // namespace

hipError_t launch_match_build(const MatchSets& s, hipStream_t stream) {
    int64_t most = 0;
    for (int i = 0; i < s.nset; ++i) most = s.set[i].n > most ? s.set[i].n : most;
    if (most == 0) return hipSuccess;
    if (most > INT32_MAX) return hipErrorInvalidValue;
    match_build_kernel<<<dim3(unsigned((most + kThreads - 1) / kThreads), unsigned(s.nset)), kThreads, 0, stream>>>(s);
    return hipGetLastError();
}

hipError_t launch_match_query(const MatchSets& s, const MatchQuery& q, hipStream_t stream) {
    const int64_t n = s.set[q.from].n;
    if (n == 0) return hipSuccess;
    match_query_kernel<<<dim3(unsigned((n + kThreads - 1) / kThreads), unsigned(q.ncol)), kThreads, 0, stream>>>(s, q);
    return hipGetLastError();
}

}  // namespace uaamg
