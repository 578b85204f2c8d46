// Device build of the pressure Poisson right-hand side (rhs_device.h).
#include "rhs_device.h"
#include "stencil_device.h"

namespace uaamg {
namespace {

using namespace dev;

__device__ __forceinline__ float grid_value(const RhsGridDev& g, int32_t leaf, int off, int comp) {
    return leaf >= 0 ? g.values[(size_t(leaf) * 512 + off) * size_t(g.ncomp) + comp] : g.bg[comp];
}

// One wavefront per x-plane of a level-0 DOF leaf, a lane per voxel (the term
// order of BuildPoissonRhs::operator(), simd_vdb_poisson.cpp:43-84). 76 us at
// 12193 leaves, where a lane per z-row, whose voxels lie 32 and 96 bytes from
// the next lane's, took 320. 173 MB pass through HBM, 2.3 TB/s, under half of a
// copy's rate: what bounds it is latency, with three quarters of a wavefront's
// life spent waiting for its chain of leaf table, operands (the weights at a
// stride of 12 bytes) and store.
__global__ __launch_bounds__(kBlockThreads) void poisson_rhs_kernel(LevelView L, RhsArgs a, float* out) {
    const int gw = __builtin_amdgcn_readfirstlane(logical_block() * kWavesPerBlock + int(threadIdx.x >> 6));
    const int leaf = gw >> 3, lx = gw & 7;
    if (leaf >= L.nleaf) return;
    if (a.bad && *a.bad >= 0) return;
    const int lane = threadIdx.x & 63, ly = lane >> 3, lz = lane & 7;
    const uint64_t* mask = L.mask + size_t(leaf) * 8;
    const uint64_t word = mask[lx];
    if (!((word >> lane) & 1u)) return;
    const int32_t* t = a.tab + size_t(leaf) * (kRhsGrids * 4);
    // weight, velocity and solid velocity of the faces x+, x-, y+, y-, z+, z-
    float w[6], v[6], sv[6];
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        const int ch = f >> 1;
        const bool positive = (f & 1) == 0;
        const int X = lx + (positive && ch == 0), Y = ly + (positive && ch == 1), Z = lz + (positive && ch == 2);
        // 0 own leaf, 1..3 the +x / +y / +z neighbour
        const bool past = positive && (ch == 0 ? X : (ch == 1 ? Y : Z)) == 8;
        const int nb = past ? 1 + ch : 0;
        const int off = ((X & 7) << 6) | ((Y & 7) << 3) | (Z & 7);
        w[f] = grid_value(a.g[kRhsWeight], t[kRhsWeight * 4 + nb], off, ch);
        v[f] = grid_value(a.g[kRhsVx + ch], t[(kRhsVx + ch) * 4 + nb], off, 0);
        sv[f] = grid_value(a.g[kRhsSolid], t[kRhsSolid * 4 + nb], off, ch);
    }
    float rhs = 0.f;
    bool nonzero_weight = false;
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        if (w[f] != 0.f) nonzero_weight = true;
        const float flux = a.invdx * (w[f] * v[f] + (1.0f - w[f]) * sv[f]);
        if ((f & 1) == 0) rhs -= flux;
        else rhs += flux;
    }
    if (!nonzero_weight) rhs = 0.f;
    int64_t k = L.dofbase[leaf];
    for (int i = 0; i < lx; ++i) k += __popcll(mask[i]);
    out[k + __popcll(word & ((uint64_t(1) << lane) - 1))] = rhs;
}

}  // namespace

hipError_t launch_poisson_rhs(const LevelView& L0, const RhsArgs& a, float* rhs_dof, hipStream_t s) {
    if (L0.nleaf <= 0) return hipSuccess;
    static_assert(8 % kWavesPerBlock == 0, "whole blocks of a leaf's planes");
    poisson_rhs_kernel<<<unsigned(L0.nleaf) * (8 / kWavesPerBlock), kBlockThreads, 0, s>>>(L0, a, rhs_dof);
    return hipGetLastError();
}

}  // namespace uaamg
