// Device kernels of the UAAMG-PCG Poisson solve (see poisson_kernels.h).
//
// Arithmetic follows LaplacianApplySIMD::LightWeightApplier
// (simd_vdb_poisson.cpp:755-1031) term by term: the six neighbour products are
// rounded separately and summed as ((x+ + x-) + (y+ + y-)) + (z+ + z-), then
// A*x = fma(x, diag, sum). The file is compiled with -ffp-contract=off so the
// only fused multiply-adds are the explicit fmaf calls.
#include <cfloat>

#include "stencil_device.h"
#include "stencil_half.h"

namespace uaamg {
namespace {

using namespace dev;

template <int MODE, bool kLevel0>
__global__ __launch_bounds__(kBlockThreads) void apply_kernel(LevelView L, const float* X, const float* B, float* Y,
                                                              float w, float one_minus_w) {
    const int leaf = wave_leaf();
    if (leaf >= L.nleaf) return;
    const int lane = threadIdx.x & 63;
    // every load is issued unconditionally (all in bounds) and rows without a
    // DOF skip only the store, so no load waits for the mask
    const uint32_t rm = row_mask(L, leaf, lane);
    const LeafRec R = leaf_rec(L, leaf);
    float xc[8], s[8], y[8];
    stencil_offdiag(L, R, PlainSrc{X}, leaf, lane, xc, s);
    const int sd = R.sd;
    const size_t row = size_t(leaf) * 512 + lane * 8;
    if (MODE == kModeRedGS || MODE == kModeBlackGS) {
        float b[8], inv[8];
        ld8(B + row, b);
        ld8_slot(L.invdiag, sd, lane, L.dflt_invdiag, inv);
        const int lx = lane >> 3, ly = lane & 7;
#pragma unroll
        for (int z = 0; z < 8; ++z) {
            float r = b[z] - s[z];
            r = r * inv[z];
            r = r * w;
            const float upd = fmaf(xc[z], one_minus_w, r);
            const bool red = ((lx + ly + z) & 1) == 0;
            y[z] = (red == (MODE == kModeRedGS)) ? upd : xc[z];
        }
    } else {
        float dg[8];
        ld8_slot(L.diag, sd, lane, L.dflt_diag, dg);
        float ax[8];
#pragma unroll
        for (int z = 0; z < 8; ++z) ax[z] = fmaf(xc[z], dg[z], s[z]);
        if (MODE == kModeLaplacian) {
#pragma unroll
            for (int z = 0; z < 8; ++z) y[z] = ax[z];
        } else {
            float b[8];
            ld8(B + row, b);
            if (MODE == kModeResidual) {
#pragma unroll
                for (int z = 0; z < 8; ++z) y[z] = b[z] - ax[z];
            } else {   // SPAI0
                float sp[8];
                ld8_slot(L.spai0, R.ssp, lane, L.dflt_spai0, sp);
#pragma unroll
                for (int z = 0; z < 8; ++z) {
                    const float r = b[z] - ax[z];
                    y[z] = fmaf(sp[z], r, xc[z]);
                }
            }
        }
    }
    if (rm == 0) return;
#pragma unroll
    for (int z = 0; z < 8; ++z)
        if (!((rm >> z) & 1u)) y[z] = 0.f;
    st8(Y + row, y);
}

// kind: 0 Jacobi, 1 SPAI0, 2 red half of RBGS
__global__ __launch_bounds__(kBlockThreads) void first_sweep_kernel(LevelView L, int kind, const float* B, float* Y,
                                                                    float w) {
    const int leaf = wave_leaf();
    if (leaf >= L.nleaf) return;
    const int lane = threadIdx.x & 63;
    const uint32_t rm = row_mask(L, leaf, lane);
    const LeafRec R = leaf_rec(L, leaf);
    const size_t row = size_t(leaf) * 512 + lane * 8;
    float b[8], c[8], y[8];
    ld8(B + row, b);
    if (kind == 1) {
        ld8_slot(L.spai0, R.ssp, lane, L.dflt_spai0, c);
#pragma unroll
        for (int z = 0; z < 8; ++z) y[z] = c[z] * b[z];
    } else {
        ld8_slot(L.invdiag, R.sd, lane, L.dflt_invdiag, c);
        const int par = ((lane >> 3) + (lane & 7)) & 1;
#pragma unroll
        for (int z = 0; z < 8; ++z) {
            float v = c[z] * b[z];
            v = w * v;
            if (kind == 2 && ((par + z) & 1)) v = 0.f;
            y[z] = v;
        }
    }
    if (rm == 0) return;
#pragma unroll
    for (int z = 0; z < 8; ++z)
        if (!((rm >> z) & 1u)) y[z] = 0.f;
    st8(Y + row, y);
}

__global__ __launch_bounds__(kBlockThreads) void restrict_kernel(LevelView C, const float* F, float* Cv) {
    const int leaf = wave_leaf();
    if (leaf >= C.nleaf) return;
    const int lane = threadIdx.x & 63;
    const uint32_t rm = row_mask(C, leaf, lane);
    const int cx = lane >> 3, cy = lane & 7;
    float out[8];
#pragma unroll
    for (int bz = 0; bz < 2; ++bz) {
        const int oct = ((cx >= 4) << 2) | ((cy >= 4) << 1) | bz;
        const int fl = C.child[size_t(leaf) * 8 + oct];
        if (fl < 0) {
#pragma unroll
            for (int c = 0; c < 4; ++c) out[4 * bz + c] = 0.f;
            continue;
        }
        const int fx = 2 * (cx & 3), fy = 2 * (cy & 3);
        float v[2][2][8];
#pragma unroll
        for (int ii = 0; ii < 2; ++ii)
#pragma unroll
            for (int jj = 0; jj < 2; ++jj) ld8(F + size_t(fl) * 512 + ((fx + ii) * 8 + (fy + jj)) * 8, v[ii][jj]);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float sum = 0.f;
#pragma unroll
            for (int ii = 0; ii < 2; ++ii)
#pragma unroll
                for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                    for (int kk = 0; kk < 2; ++kk) sum += v[ii][jj][2 * c + kk];
            out[4 * bz + c] = sum * 0.125f;
        }
    }
    if (rm == 0) return;
#pragma unroll
    for (int z = 0; z < 8; ++z)
        if (!((rm >> z) & 1u)) out[z] = 0.f;
    st8(Cv + size_t(leaf) * 512 + lane * 8, out);
}

__global__ __launch_bounds__(kBlockThreads) void prolong_add_kernel(LevelView Fl, const float* Cv, float* Fv,
                                                                    float alpha) {
    const int leaf = wave_leaf();
    if (leaf >= Fl.nleaf) return;
    const int lane = threadIdx.x & 63;
    const uint32_t rm = row_mask(Fl, leaf, lane);
    const int p = Fl.parent[leaf];
    if (p < 0 || rm == 0) return;
    const int cl = p >> 3, oct = p & 7;
    const int bx = (oct >> 2) & 1, by = (oct >> 1) & 1, bz = oct & 1;
    const int crow = (((lane >> 3) >> 1) + 4 * bx) * 8 + (((lane & 7) >> 1) + 4 * by);
    const float4 c4 = *reinterpret_cast<const float4*>(Cv + size_t(cl) * 512 + crow * 8 + 4 * bz);
    const float c[4] = {alpha * c4.x, alpha * c4.y, alpha * c4.z, alpha * c4.w};
    const size_t row = size_t(leaf) * 512 + lane * 8;
    float y[8];
    ld8(Fv + row, y);
#pragma unroll
    for (int z = 0; z < 8; ++z)
        if ((rm >> z) & 1u) y[z] += c[z >> 1];
    st8(Fv + row, y);
}

// ---- the Jacobi-family passes, on half rows (stencil_half.h). kLevel0 only
// names the level in profiles.
// Leaves a workgroup. With 2 / 4 / 8 the sweep takes 132 / 133 / 137 us at 92428
// leaves, the one after the prolongation 180 / 202 / 254: the more wavefronts
// meet at the barrier, the fewer hide each other's loads.
constexpr int kSweepLeaves = 2;
constexpr int kSweepThreads = 128 * kSweepLeaves;

// kEarly: the sweep's own operands are loaded before the barrier (JacobiHalf)
template <bool kEarly, class Src, class VB, class VY>
__device__ __forceinline__ void jacobi_half(const LevelView& L, const Src& src, const VB* B, VY* Y, float w) {
    __shared__ float tiles[kSweepLeaves][512];   // a workgroup holds whole leaves
    HalfPos p = half_pos<2 * kSweepLeaves>();
    const bool valid = p.leaf < L.nleaf;
    if (!valid) p.leaf = L.nleaf - 1;   // meets the others at the barrier, stores nothing
    const uint32_t rm = half_row_mask(L, p);
    const LeafRec R = leaf_rec(L, p.leaf);
    JacobiHalf j;
    if (kEarly) j.load(L, R, p, B);
    float xc[4], s[4], y[4];
    typename Src::Quad c;
    half_offdiag<kSweepLeaves>(L, R, src, p, tiles, c, xc, s);
    if (!kEarly) j.load(L, R, p, B);
    j.sweep(xc, s, w, rm >> p.z0, y);
    if (valid && rm) sth(Y + size_t(p.leaf) * 512 + p.row * 8 + p.z0, y);   // rows without a DOF are not written
}

// One weighted Jacobi sweep. Against full rows (one lane per z-row of eight),
// at 12193 / 92428 leaves of level 0: 16.0 / 132 us (17.2 / 157), 3.6 / 11.6 us
// at 282 / 12247 leaves (4.4 / 12.5); at 92428 leaves 0.74 GB pass through HBM, 5.6 TB/s.
template <bool kLevel0, class VX, class VB, class VY>
__global__ __launch_bounds__(kSweepThreads) void jacobi_half_kernel(LevelView L, const VX* X, const VB* B, VY* Y,
                                                                    float w) {
    jacobi_half<false>(L, PlainHalf<VX>{X}, B, Y, w);
}

// First two scheduled / weighted Jacobi sweeps from a zero guess in one pass:
// the first sweep's result is rebuilt where the second sweep reads it.
// 16.4 / 143 us at 12193 / 92428 leaves (full rows 21.5 / 191).
template <bool kLevel0, class VB, class VY>
__global__ __launch_bounds__(kSweepThreads) void jacobi_first2_half_kernel(LevelView L, const VB* B, VY* Y, float w0,
                                                                           float w1) {
    jacobi_half<true>(L, FirstHalf<VB>{B, L.invdiag, L.dflt_invdiag, w0}, B, Y, w1);
}

// Prolongation (x += P x_coarse) fused into the first post-smoothing sweep.
// 20.7 / 181 us at 12193 / 92428 leaves (full rows 23.4 / 206).
template <bool kLevel0, class V, class VB>
__global__ __launch_bounds__(kSweepThreads) void prolong_jacobi_half_kernel(LevelView L, const V* X, const V* Xc,
                                                                            const VB* B, V* Y, float w) {
    jacobi_half<false>(L, ProlongHalf<V>{X, Xc, L.mask}, B, Y, w);
}

// Residual r = b - A x of half a fine leaf, restricted in the same pass: each
// coarse voxel's eight children lie in one half, so the wavefront writes its
// half of the parent coarse leaf's 4^3 octant (restriction, :1624-1684, sums
// the children in x,y,z nested order and scales by 1/8).
template <bool kLevel0, class V, class VB>
__global__ __launch_bounds__(kBlockThreads) void residual_restrict_half_kernel(LevelView F, const V* X, const VB* B,
                                                                               V* Cv) {
    __shared__ float rs[kWavesPerBlock][256];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const HalfPos p = half_pos();
    const bool valid = p.leaf < F.nleaf;
    float r[4];
    fillh(r, 0.f);
    int par = -1;
    if (valid) {
        const uint32_t m = half_row_mask(F, p) >> p.z0;
        const LeafRec R = leaf_rec(F, p.leaf);
        par = R.par;
        const int off = p.row * 8 + p.z0;
        float xc[4], s[4], dg[4], b[4];
        typename PlainHalf<V>::Quad c;
        half_offdiag<0>(F, R, PlainHalf<V>{X}, p, nullptr, c, xc, s);
        ldh_slot(F.diag, R.sd, off, F.dflt_diag, dg);
        ldh(B + size_t(p.leaf) * 512 + off, b);
#pragma unroll
        for (int z = 0; z < 4; ++z) {
            const float v = b[z] - fmaf(xc[z], dg[z], s[z]);
            r[z] = ((m >> z) & 1u) ? v : 0.f;
        }
    }
    sth(&rs[wave][lane * 4], r);   // row (within the half) * 8 + z
    __syncthreads();
    if (!valid || par < 0 || lane >= 32) return;   // every DOF leaf has a parent; par is a bounds guard
    const int cx = lane >> 4, cy = (lane >> 2) & 3, cz = lane & 3;   // cx within the half
    float sum = 0.f;
#pragma unroll
    for (int ii = 0; ii < 2; ++ii)
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) sum += rs[wave][((2 * cx + ii) * 8 + (2 * cy + jj)) * 8 + 2 * cz + kk];
    const int cl = par >> 3, oct = par & 7;
    const int off = ((cx + 2 * (p.row >> 5) + 4 * ((oct >> 2) & 1)) * 8 + (cy + 4 * ((oct >> 1) & 1))) * 8 + cz +
                    4 * (oct & 1);
    st1(Cv + size_t(cl) * 512 + off, sum * 0.125f);
}

__global__ __launch_bounds__(kBlockThreads) void scatter_dof_kernel(LevelView L, const float* dv, float* Y) {
    const int leaf = wave_leaf();
    if (leaf >= L.nleaf) return;
    const int lane = threadIdx.x & 63;
    const uint32_t rm = row_mask(L, leaf, lane);
    float y[8];
    fill8(y, 0.f);
    if (rm) {
        int64_t k = row_dof_base(L, leaf, lane);
#pragma unroll
        for (int z = 0; z < 8; ++z)
            if ((rm >> z) & 1u) y[z] = dv[k++];
    }
    st8(Y + size_t(leaf) * 512 + lane * 8, y);
}

__global__ __launch_bounds__(kBlockThreads) void gather_dof_kernel(LevelView L, const float* X, float* dv) {
    const int leaf = wave_leaf();
    if (leaf >= L.nleaf) return;
    const int lane = threadIdx.x & 63;
    const uint32_t rm = row_mask(L, leaf, lane);
    if (!rm) return;
    float x[8];
    ld8(X + size_t(leaf) * 512 + lane * 8, x);
    int64_t k = row_dof_base(L, leaf, lane);
#pragma unroll
    for (int z = 0; z < 8; ++z)
        if ((rm >> z) & 1u) dv[k++] = x[z];
}


// level 0 and the coarse levels run the same code under two names
template <class F0, class F1>
hipError_t by_level(const LevelView& L, const F0& level0, const F1& coarse) {
    if (L.nleaf <= 0) return hipSuccess;
    if (L.level == 0) level0();
    else coarse();
    return hipGetLastError();
}

template <class VX, class VB, class VY>
hipError_t jacobi_t(const LevelView& L, const VX* x, const VB* b, VY* y, float w, hipStream_t s) {
    const unsigned g = half_grid(L.nleaf, 2 * kSweepLeaves);
    return by_level(
        L, [&] { jacobi_half_kernel<true><<<g, kSweepThreads, 0, s>>>(L, x, b, y, w); },
        [&] { jacobi_half_kernel<false><<<g, kSweepThreads, 0, s>>>(L, x, b, y, w); });
}

template <class VB, class VY>
hipError_t jacobi_first2_t(const LevelView& L, const VB* b, VY* y, float w0, float w1, hipStream_t s) {
    const unsigned g = half_grid(L.nleaf, 2 * kSweepLeaves);
    return by_level(
        L, [&] { jacobi_first2_half_kernel<true><<<g, kSweepThreads, 0, s>>>(L, b, y, w0, w1); },
        [&] { jacobi_first2_half_kernel<false><<<g, kSweepThreads, 0, s>>>(L, b, y, w0, w1); });
}

template <class V, class VB>
hipError_t prolong_jacobi_t(const LevelView& L, const V* x, const V* xc, const VB* b, V* y, float w, hipStream_t s) {
    const unsigned g = half_grid(L.nleaf, 2 * kSweepLeaves);
    return by_level(
        L, [&] { prolong_jacobi_half_kernel<true><<<g, kSweepThreads, 0, s>>>(L, x, xc, b, y, w); },
        [&] { prolong_jacobi_half_kernel<false><<<g, kSweepThreads, 0, s>>>(L, x, xc, b, y, w); });
}

template <class V, class VB>
hipError_t residual_restrict_t(const LevelView& L, const V* x, const VB* b, V* cb, hipStream_t s) {
    const unsigned g = half_grid(L.nleaf);
    return by_level(
        L, [&] { residual_restrict_half_kernel<true><<<g, kBlockThreads, 0, s>>>(L, x, b, cb); },
        [&] { residual_restrict_half_kernel<false><<<g, kBlockThreads, 0, s>>>(L, x, b, cb); });
}

}  // namespace

hipError_t launch_apply(const LevelView& L, int mode, const float* x, const float* b, float* y, float w,
                        hipStream_t s) {
    if (L.nleaf <= 0) return hipSuccess;
    const dim3 g(grid_for(L.nleaf)), t(kBlockThreads);
    const float omw = 1.0f - w;
    if (mode == kModeJacobi) return jacobi_t(L, x, b, y, w, s);
    if (L.level == 0) {
        switch (mode) {
            case kModeLaplacian: apply_kernel<kModeLaplacian, true><<<g, t, 0, s>>>(L, x, b, y, w, omw); break;
            case kModeResidual: apply_kernel<kModeResidual, true><<<g, t, 0, s>>>(L, x, b, y, w, omw); break;
            case kModeSpai0: apply_kernel<kModeSpai0, true><<<g, t, 0, s>>>(L, x, b, y, w, omw); break;
            case kModeRedGS: apply_kernel<kModeRedGS, true><<<g, t, 0, s>>>(L, x, b, y, w, omw); break;
            case kModeBlackGS: apply_kernel<kModeBlackGS, true><<<g, t, 0, s>>>(L, x, b, y, w, omw); break;
            default: return hipErrorInvalidValue;
        }
    } else {
        switch (mode) {
            case kModeLaplacian: apply_kernel<kModeLaplacian, false><<<g, t, 0, s>>>(L, x, b, y, w, omw); break;
            case kModeResidual: apply_kernel<kModeResidual, false><<<g, t, 0, s>>>(L, x, b, y, w, omw); break;
            case kModeSpai0: apply_kernel<kModeSpai0, false><<<g, t, 0, s>>>(L, x, b, y, w, omw); break;
            case kModeRedGS: apply_kernel<kModeRedGS, false><<<g, t, 0, s>>>(L, x, b, y, w, omw); break;
            case kModeBlackGS: apply_kernel<kModeBlackGS, false><<<g, t, 0, s>>>(L, x, b, y, w, omw); break;
            default: return hipErrorInvalidValue;
        }
    }
    return hipGetLastError();
}

hipError_t launch_first_sweep(const LevelView& L, int kind, const float* b, float* y, float w, hipStream_t s) {
    if (L.nleaf <= 0) return hipSuccess;
    first_sweep_kernel<<<grid_for(L.nleaf), kBlockThreads, 0, s>>>(L, kind, b, y, w);
    return hipGetLastError();
}

hipError_t launch_restrict(const LevelView& coarse, const float* fine_v, float* coarse_v, hipStream_t s) {
    if (coarse.nleaf <= 0) return hipSuccess;
    restrict_kernel<<<grid_for(coarse.nleaf), kBlockThreads, 0, s>>>(coarse, fine_v, coarse_v);
    return hipGetLastError();
}

hipError_t launch_prolong_add(const LevelView& fine, const float* coarse_v, float* fine_v, float alpha,
                              hipStream_t s) {
    if (fine.nleaf <= 0) return hipSuccess;
    prolong_add_kernel<<<grid_for(fine.nleaf), kBlockThreads, 0, s>>>(fine, coarse_v, fine_v, alpha);
    return hipGetLastError();
}

hipError_t launch_scatter_dof(const LevelView& L, const float* dofvec, float* bricks, hipStream_t s) {
    if (L.nleaf <= 0) return hipSuccess;
    scatter_dof_kernel<<<grid_for(L.nleaf), kBlockThreads, 0, s>>>(L, dofvec, bricks);
    return hipGetLastError();
}

hipError_t launch_gather_dof(const LevelView& L, const float* bricks, float* dofvec, hipStream_t s) {
    if (L.nleaf <= 0) return hipSuccess;
    gather_dof_kernel<<<grid_for(L.nleaf), kBlockThreads, 0, s>>>(L, bricks, dofvec);
    return hipGetLastError();
}

hipError_t launch_jacobi_first2(const LevelView& L, const float* b, float* y, float w0, float w1, hipStream_t s) {
    return jacobi_first2_t(L, b, y, w0, w1, s);
}

hipError_t launch_prolong_jacobi(const LevelView& L, const float* x, const float* xc, const float* b, float* y,
                                 float w, hipStream_t s) {
    return prolong_jacobi_t(L, x, xc, b, y, w, s);
}

hipError_t launch_residual_restrict(const LevelView& fine, const float* x, const float* b, float* coarse_b,
                                    hipStream_t s) {
    return residual_restrict_t(fine, x, b, coarse_b, s);
}

// ---- mixed-precision W-cycle launchers (level 0 reads the FP32 PCG residual)
hipError_t launch_jacobi_first2(const LevelView& L, const float* b, bf16* y, float w0, float w1, hipStream_t s) {
    return jacobi_first2_t(L, b, y, w0, w1, s);
}
hipError_t launch_jacobi_first2(const LevelView& L, const bf16* b, bf16* y, float w0, float w1, hipStream_t s) {
    return jacobi_first2_t(L, b, y, w0, w1, s);
}

hipError_t launch_jacobi(const LevelView& L, const bf16* x, const float* b, bf16* y, float w, hipStream_t s) {
    return jacobi_t(L, x, b, y, w, s);
}
hipError_t launch_jacobi(const LevelView& L, const bf16* x, const float* b, float* y, float w, hipStream_t s) {
    return jacobi_t(L, x, b, y, w, s);
}
hipError_t launch_jacobi(const LevelView& L, const float* x, const float* b, bf16* y, float w, hipStream_t s) {
    return jacobi_t(L, x, b, y, w, s);
}
hipError_t launch_jacobi(const LevelView& L, const bf16* x, const bf16* b, bf16* y, float w, hipStream_t s) {
    return jacobi_t(L, x, b, y, w, s);
}

hipError_t launch_residual_restrict(const LevelView& fine, const bf16* x, const float* b, bf16* coarse_b,
                                    hipStream_t s) {
    return residual_restrict_t(fine, x, b, coarse_b, s);
}
hipError_t launch_residual_restrict(const LevelView& fine, const bf16* x, const bf16* b, bf16* coarse_b,
                                    hipStream_t s) {
    return residual_restrict_t(fine, x, b, coarse_b, s);
}

hipError_t launch_prolong_jacobi(const LevelView& L, const bf16* x, const bf16* xc, const float* b, bf16* y, float w,
                                 hipStream_t s) {
    return prolong_jacobi_t(L, x, xc, b, y, w, s);
}
hipError_t launch_prolong_jacobi(const LevelView& L, const bf16* x, const bf16* xc, const bf16* b, bf16* y, float w,
                                 hipStream_t s) {
    return prolong_jacobi_t(L, x, xc, b, y, w, s);
}

}  // namespace uaamg
