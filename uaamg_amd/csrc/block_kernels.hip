// One W-cycle level visit in two launches (coarse levels).
//
// On the small levels of the hierarchy every smoothing sweep is its own
// latency-bound launch. A block-visit kernel gives each leaf one workgroup
// that holds the leaf plus a halo of 4 voxels (from up to 26 neighbour
// leaves) and runs consecutive sweeps on a shrinking region: sweep k is valid
// k voxels further in, so the leaf's own 8^3 values come out exact. The halo
// voxels are recomputed redundantly by each neighbouring workgroup; every
// value is produced by the same arithmetic as the per-sweep kernels
// (stencil order ((x+ + x-) + (y+ + y-)) + (z+ + z-), fma(x, diag, s),
// fma(w, (b - Ax) * D^-1, x), non-DOF voxels 0), and with BF16 storage each
// sweep's output is rounded where the per-sweep kernels store it, so results
// are bit-identical to theirs in either precision.
//
//   kPreZero   x1 = w0 D^-1 b, two sweeps, residual, restriction
//              (first visit, muCyclePreconditioner from a zero guess)
//   kPreAgain  three sweeps from the level's x, residual, restriction
//   kPost      x + P x_coarse, three sweeps
//
// The region is 16^3 voxels, four of them in z per thread (1024 threads, one
// wavefront per x slab): every global load is an aligned row of four values,
// and each thread keeps its voxels' right-hand side and coefficients in
// registers for all sweeps. Only x crosses threads, between slabs and y rows
// through LDS (two buffers in turn, one barrier per sweep) and along z inside
// the quad of lanes that holds a row. What bounds the kernel is latency: the
// launch, two memory round trips (neighbourhood records, then operands) and
// the chain of sweeps.
//
// On the level above the coarsest, the post-visit can take the coarsest solve
// in with it (block_post_cg_kernel): every workgroup runs the coarsest CG on
// the whole coarsest system (the same routine and thread count as the
// standalone solve, so every workgroup gets the same values the standalone
// kernel stores), keeps the solution in LDS for its staging, and workgroup 0
// also stores it. The coarse correction then never crosses HBM and the
// W-cycle bottom loses a launch.
#include <type_traits>

#include "coarsest_device.h"
#include "stencil_device.h"

namespace uaamg {
namespace {

using namespace dev;

enum BlockMode { kPreZero = 0, kPreAgain = 1, kPost = 2 };
constexpr int kRegionQuads = 1024;   // 16 x 16 rows of four quads
// One quad per thread: with two per thread and half the threads the visit pair
// of a 282-leaf level took 34.1 us against 32.5 (VALU time per sweep is the
// same, fewer wavefronts hide less of the loads).
constexpr int kBlkThreads = 1024;

// Loads of four values in z: a z row of four of a brick
template <class V>
__device__ __forceinline__ void ldq(const V* p, float v[4]) {
    const float4 a = ld4(p);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}
__device__ __forceinline__ void stq(float* p, const float v[4]) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void stq(bf16* p, const float v[4]) {
    *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
}
__device__ __forceinline__ void ld2c(const float* p, float v[2]) {
    const float2 a = *reinterpret_cast<const float2*>(p);
    v[0] = a.x; v[1] = a.y;
}
__device__ __forceinline__ void ld2c(const bf16* p, float v[2]) {
    const uint32_t q = *reinterpret_cast<const uint32_t*>(p);
    v[0] = __uint_as_float(q << 16);
    v[1] = __uint_as_float(q & 0xffff0000u);
}

// value as the vector storage type holds it (the per-sweep kernels store
// every sweep's output, so the block form rounds where they would)
template <class V>
__device__ __forceinline__ float stored(float v) {
    if constexpr (std::is_same_v<V, float>) return v;
    else return float(V(v));
}

// v of the previous / next lane of the quad (a z row's four threads); the
// quad's first / last lane gets its own value, which only voxels outside the
// valid region use
__device__ __forceinline__ float quad_prev(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x90, 0xf, 0xf, true));   // [0,0,1,2]
}
__device__ __forceinline__ float quad_next(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xf9, 0xf, 0xf, true));   // [1,2,3,3]
}

// A thread's four voxels: their right-hand side, coefficients and DOF bits.
struct Quad {
    float b[4], dg[4], inv[4], cx[4], cxp[4], cy[4], cyp[4], cz[4];
    float czp;
    uint32_t m;
};

// A x of the quad at region index t, x being its own values and `buf` the
// region's (buf holds x of every quad; the caller has passed the barrier).
__device__ __forceinline__ void quad_ax(const Quad& Q, const float4* buf, int t, const float x[4], float ax[4]) {
    float s[4];
    {
        const float4 p = buf[t + 64], m = buf[t - 64];
        const float xp[4] = {p.x, p.y, p.z, p.w}, xm[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float f1 = xp[k] * Q.cxp[k];
            const float f2 = xm[k] * Q.cx[k];
            s[k] = f1 + f2;
        }
    }
    {
        const float4 p = buf[t + 4], m = buf[t - 4];
        const float yp[4] = {p.x, p.y, p.z, p.w}, ym[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float f3 = yp[k] * Q.cyp[k];
            const float f4 = ym[k] * Q.cy[k];
            s[k] = s[k] + (f3 + f4);
        }
    }
    const float zm = quad_prev(x[3]), zp = quad_next(x[0]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float f5 = (k < 3 ? x[k + 1] : zp) * (k < 3 ? Q.cz[k + 1] : Q.czp);
        const float f6 = (k > 0 ? x[k - 1] : zm) * Q.cz[k];
        s[k] = s[k] + (f5 + f6);
        ax[k] = fmaf(x[k], Q.dg[k], s[k]);
    }
}

// A workgroup of kT threads: 1024 / kT quads per thread, wavefront w holding
// slabs w, w + kT/64, ...
template <int kT>
struct Part {
    static constexpr int kPer = kRegionQuads / kT;
    Quad Q[kPer];
    float x[kPer][4];
    __device__ __forceinline__ static int slab(int h) {
        return __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)) + h * (kT / 64);
    }
    __device__ __forceinline__ static int at(int h) { return int(threadIdx.x) + h * kT; }
};

// One Jacobi sweep x <- J_w(x), rounded to the storage type V, on slabs LO ..
// 15 - LO (uniform per wavefront; rows outside LO .. 15 - LO in y, and the
// outer z voxels, get values that nothing valid reads). x enters published in
// `from`; it is published again in `to`.
template <int LO, class V, int kT>
__device__ __forceinline__ void sweep(Part<kT>& P, const float4* from, float4* to, float w) {
#pragma unroll
    for (int h = 0; h < Part<kT>::kPer; ++h) {
        const int slab = P.slab(h);
        if (slab >= LO && slab <= 15 - LO) {
            const Quad& Q = P.Q[h];
            float* x = P.x[h];
            float ax[4];
            quad_ax(Q, from, P.at(h), x, ax);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                float t = Q.b[k] - ax[k];
                t = t * Q.inv[k];
                const float r = fmaf(w, t, x[k]);
                x[k] = ((Q.m >> k) & 1u) ? stored<V>(r) : 0.f;
            }
            to[P.at(h)] = make_float4(x[0], x[1], x[2], x[3]);
        }
    }
    __syncthreads();
}

// The visit of one leaf. kCg (kPost only): the coarse correction comes from
// cgx, the coarsest solution in LDS indexed by coarsest DOF (dof_of maps a
// coarsest brick position to its DOF, -1 elsewhere), instead of Xc.
template <int MODE, class V, int kT, bool kCg>
__device__ __forceinline__ void visit_body(const LevelView& L, const V* Xin, const V* Xc, const V* B, V* Xout, V* Cv,
                                           float w0, float w1, float w2, const int32_t* dof_of, const float* cgx) {
    __shared__ float4 buf[2][kRegionQuads];
    // the first region row the mode reads, and the first it sweeps
    constexpr int kIn = MODE == kPreAgain ? 0 : 1;
    constexpr int kSw = kIn + 1;
    constexpr int kPer = Part<kT>::kPer;
    Part<kT> P;
    const int leaf = logical_block();
    const int tid = threadIdx.x;
    const int ry = (tid >> 2) & 15, qz = tid & 3;
    const int ay = ry < 4 ? 0 : (ry > 11 ? 2 : 1), az = qz < 1 ? 0 : (qz > 2 ? 2 : 1);
    const int ly = (ry + 4) & 7, lz = 4 * ((qz + 1) & 1);

    // the records of the neighbourhood leaves that hold the thread's voxels
    int4 ra[kPer];
    int2 rb[kPer];
    int sxp[kPer], syp[kPer];
#pragma unroll
    for (int h = 0; h < kPer; ++h) {
        const int slab = P.slab(h);
        const int ax = slab < 4 ? 0 : (slab > 11 ? 2 : 1), lx = (slab + 4) & 7;
        const int32_t* rec = L.nb27 + (size_t(leaf) * 27 + ax * 9 + ay * 3 + az) * kNb27Stride;
        ra[h] = *reinterpret_cast<const int4*>(rec);
        rb[h] = *reinterpret_cast<const int2*>(rec + 4);
        // slots of the rows at x + 1 and y + 1 (the next neighbourhood leaf's past a face)
        sxp[h] = rec[(lx == 7 && ax < 2 ? 9 * kNb27Stride : 0) + 2];
        syp[h] = rec[(ly == 7 && ay < 2 ? 3 * kNb27Stride : 0) + 3];
    }
#pragma unroll
    for (int h = 0; h < kPer; ++h) {
        const int slab = P.slab(h);
        const int lx = (slab + 4) & 7;
        const int n = ra[h].x;
        const int row = (lx << 6) | (ly << 3) | lz;
        Quad& Q = P.Q[h];
        float* x = P.x[h];
        Q.m = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            x[k] = 0.f;
            Q.b[k] = 0.f;
            Q.dg[k] = L.dflt_diag;
            Q.inv[k] = L.dflt_invdiag;
            Q.cx[k] = Q.cxp[k] = Q.cy[k] = Q.cyp[k] = Q.cz[k] = L.dflt_off;
        }
        if (slab >= kIn && slab <= 15 - kIn) {
            // vectors of absent leaves are 0, coefficients of absent leaves or
            // trimmed bricks the default constants
            uint32_t mb = 0;
            float c2[2] = {0.f, 0.f};
            int di0 = -1, di1 = -1;
            if (n >= 0) {
                const size_t at = size_t(n) * 512 + row;
                mb = reinterpret_cast<const uint8_t*>(L.mask)[size_t(n) * 64 + lx * 8 + ly];
                ldq(B + at, Q.b);
                if (MODE != kPreZero) ldq(Xin + at, x);
                if (MODE == kPost && rb[h].y >= 0) {
                    const int cl = rb[h].y >> 3, oct = rb[h].y & 7;
                    const int crow = ((lx >> 1) + 4 * ((oct >> 2) & 1)) * 8 + ((ly >> 1) + 4 * ((oct >> 1) & 1));
                    const size_t ci = size_t(cl) * 512 + crow * 8 + 4 * (oct & 1) + (lz >> 1);
                    if constexpr (kCg) {
                        const int2 d = *reinterpret_cast<const int2*>(dof_of + ci);
                        di0 = d.x;
                        di1 = d.y;
                    } else {
                        ld2c(Xc + ci, c2);
                    }
                }
            }
            if (ra[h].y >= 0) {
                ldq(L.diag + size_t(ra[h].y) * 512 + row, Q.dg);
                ldq(L.invdiag + size_t(ra[h].y) * 512 + row, Q.inv);
            }
            if (slab >= kSw && slab <= 15 - kSw) {
                if (ra[h].z >= 0) ldq(L.cx + size_t(ra[h].z) * 512 + row, Q.cx);
                if (sxp[h] >= 0) ldq(L.cx + size_t(sxp[h]) * 512 + ((row + 64) & 511), Q.cxp);
                if (ra[h].w >= 0) ldq(L.cy + size_t(ra[h].w) * 512 + row, Q.cy);
                if (syp[h] >= 0) ldq(L.cy + size_t(syp[h]) * 512 + ((row & ~56) | ((row + 8) & 56)), Q.cyp);
                if (rb[h].x >= 0) ldq(L.cz + size_t(rb[h].x) * 512 + row, Q.cz);
            }
            Q.m = (mb >> lz) & 15u;
            if (MODE == kPreZero) {
#pragma unroll
                for (int k = 0; k < 4; ++k) x[k] = w0 * (Q.inv[k] * Q.b[k]);
            }
            if (MODE == kPost) {
                if constexpr (kCg) {
                    // a fine DOF's parent voxel is a coarsest DOF, the only case where it is used
                    c2[0] = cgx[di0 >= 0 ? di0 : kMaxCoarsestDof];
                    c2[1] = cgx[di1 >= 0 ? di1 : kMaxCoarsestDof];
                }
                if (rb[h].y >= 0) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const float t = x[k] + c2[k >> 1];
                        x[k] = ((Q.m >> k) & 1u) ? t : x[k];
                    }
                }
            }
        }
        Q.czp = quad_next(Q.cz[0]);
        buf[0][P.at(h)] = make_float4(x[0], x[1], x[2], x[3]);
    }
    __syncthreads();

    if (MODE == kPreZero) {
        sweep<2, V, kT>(P, buf[0], buf[1], w1);
        sweep<3, V, kT>(P, buf[1], buf[0], w2);
    } else if (MODE == kPreAgain) {
        sweep<1, V, kT>(P, buf[0], buf[1], w0);
        sweep<2, V, kT>(P, buf[1], buf[0], w1);
        sweep<3, V, kT>(P, buf[0], buf[1], w2);
    } else {
        sweep<2, V, kT>(P, buf[0], buf[1], w0);
        sweep<3, V, kT>(P, buf[1], buf[0], w1);
        sweep<4, V, kT>(P, buf[0], buf[1], w2);
    }

    // the leaf's own values: slabs and rows 4 .. 11, the two middle quads;
    // then the residual on the own brick, in the buffer that the last sweep
    // read, and its restriction into the parent's octant
    const float4* fin = MODE == kPreZero ? buf[0] : buf[1];
    float* rs = reinterpret_cast<float*>(MODE == kPreZero ? buf[1] : buf[0]);
#pragma unroll
    for (int h = 0; h < kPer; ++h) {
        const int slab = P.slab(h);
        if (slab < 4 || slab > 11) continue;   // whole wavefronts: the quad exchange needs all four lanes
        const bool own = ry >= 4 && ry < 12 && (qz == 1 || qz == 2);
        const int row = (((slab + 4) & 7) << 6) | (ly << 3) | lz;
        if (own) stq(Xout + size_t(leaf) * 512 + row, P.x[h]);
        if (MODE == kPost) continue;
        float axv[4], rv[4];
        quad_ax(P.Q[h], fin, P.at(h), P.x[h], axv);
#pragma unroll
        for (int k = 0; k < 4; ++k) rv[k] = ((P.Q[h].m >> k) & 1u) ? P.Q[h].b[k] - axv[k] : 0.f;
        if (own) stq(rs + row, rv);
    }
    if (MODE == kPost) return;
    __syncthreads();
    if (tid < 64) {
        const int ccx = tid >> 4, ccy = (tid >> 2) & 3, ccz = tid & 3;
        float sum = 0.f;
#pragma unroll
        for (int ii = 0; ii < 2; ++ii)
#pragma unroll
            for (int jj = 0; jj < 2; ++jj) {
                const float2 r = *reinterpret_cast<const float2*>(rs + ((2 * ccx + ii) * 8 + (2 * ccy + jj)) * 8 + 2 * ccz);
                sum += r.x;
                sum += r.y;
            }
        const int p = L.parent[leaf];
        if (p < 0) return;
        const int cl = p >> 3, oct = p & 7;
        const int off = ((ccx + 4 * ((oct >> 2) & 1)) * 8 + (ccy + 4 * ((oct >> 1) & 1))) * 8 + ccz + 4 * (oct & 1);
        Cv[size_t(cl) * 512 + off] = V(sum * 0.125f);
    }
}

// two workgroups per CU
template <int MODE, class V>
__global__ __launch_bounds__(kBlkThreads) __attribute__((amdgpu_waves_per_eu(2 * kBlkThreads / 256))) void
block_visit_kernel(LevelView L, const V* Xin, const V* Xc, const V* B, V* Xout, V* Cv, float w0, float w1, float w2) {
    visit_body<MODE, V, kBlkThreads, false>(L, Xin, Xc, B, Xout, Cv, w0, w1, w2, nullptr, nullptr);
}

// The coarsest solve (right-hand side Bc, solution stored into Xc by
// workgroup 0) followed by the kPost visit of the level above it, on the
// CG's thread count. The CG's last barrier has passed when it writes its
// solution into cg.sp; the barrier here publishes it.
template <class V, int kMaxDof>
__global__ __launch_bounds__(kCgThreads) void block_post_cg_kernel(LevelView L, CoarsestView C, const int32_t* dof_of,
                                                                   const V* Bc, V* Xc, const V* Xin, const V* B,
                                                                   V* Xout, float w0, float w1, float w2) {
    __shared__ CgShared cg;
    coarsest_cg_block<kCgThreads, V, kMaxDof, true>(C, Bc, blockIdx.x == 0 ? Xc : nullptr, cg);
    __syncthreads();
    visit_body<kPost, V, kCgThreads, true>(L, Xin, nullptr, B, Xout, nullptr, w0, w1, w2, dof_of, cg.sp);
}

template <int MODE, class V>
hipError_t launch_mode(const LevelView& L, const V* xin, const V* xc, const V* b, V* xout, V* cv, float w0, float w1,
                       float w2, hipStream_t s) {
    block_visit_kernel<MODE, V><<<unsigned(L.nleaf), kBlkThreads, 0, s>>>(L, xin, xc, b, xout, cv, w0, w1, w2);
    return hipGetLastError();
}

template <class V>
hipError_t block_pre_t(const LevelView& L, bool from_zero, const V* x, const V* b, V* x_out, V* coarse_b, float w0,
                       float w1, float w2, hipStream_t s) {
    if (L.nleaf <= 0) return hipSuccess;
    if (!L.nb27) return hipErrorInvalidValue;
    if (from_zero) return launch_mode<kPreZero, V>(L, nullptr, nullptr, b, x_out, coarse_b, w0, w1, w2, s);
    return launch_mode<kPreAgain, V>(L, x, nullptr, b, x_out, coarse_b, w0, w1, w2, s);
}

template <class V>
hipError_t block_post_t(const LevelView& L, const V* x, const V* xc, const V* b, V* x_out, float w0, float w1, float w2,
                        hipStream_t s) {
    if (L.nleaf <= 0) return hipSuccess;
    if (!L.nb27) return hipErrorInvalidValue;
    return launch_mode<kPost, V>(L, x, xc, b, x_out, nullptr, w0, w1, w2, s);
}

template <class V>
hipError_t block_post_cg_t(const LevelView& L, const CoarsestView& C, const int32_t* dof_of, const V* bc, V* xc,
                           const V* x, const V* b, V* x_out, float w0, float w1, float w2, hipStream_t s) {
    if (L.nleaf <= 0) return hipSuccess;   // as block_post_t: nothing reads the coarse correction
    if (!L.nb27 || !dof_of || C.ndof <= 0 || C.ndof > kMaxCoarsestDof) return hipErrorInvalidValue;
    const unsigned g = unsigned(L.nleaf);
    if (C.ndof <= kCgSmallDof)
        block_post_cg_kernel<V, kCgSmallDof><<<g, kCgThreads, 0, s>>>(L, C, dof_of, bc, xc, x, b, x_out, w0, w1, w2);
    else
        block_post_cg_kernel<V, kMaxCoarsestDof>
            <<<g, kCgThreads, 0, s>>>(L, C, dof_of, bc, xc, x, b, x_out, w0, w1, w2);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_block_pre(const LevelView& L, bool from_zero, const float* x, const float* b, float* x_out,
                            float* coarse_b, float w0, float w1, float w2, hipStream_t s) {
    return block_pre_t<float>(L, from_zero, x, b, x_out, coarse_b, w0, w1, w2, s);
}

hipError_t launch_block_post(const LevelView& L, const float* x, const float* xc, const float* b, float* x_out,
                             float w0, float w1, float w2, hipStream_t s) {
    return block_post_t<float>(L, x, xc, b, x_out, w0, w1, w2, s);
}

hipError_t launch_block_pre(const LevelView& L, bool from_zero, const bf16* x, const bf16* b, bf16* x_out,
                            bf16* coarse_b, float w0, float w1, float w2, hipStream_t s) {
    return block_pre_t<bf16>(L, from_zero, x, b, x_out, coarse_b, w0, w1, w2, s);
}

hipError_t launch_block_post(const LevelView& L, const bf16* x, const bf16* xc, const bf16* b, bf16* x_out,
                             float w0, float w1, float w2, hipStream_t s) {
    return block_post_t<bf16>(L, x, xc, b, x_out, w0, w1, w2, s);
}

hipError_t launch_block_post_cg(const LevelView& L, const CoarsestView& C, const int32_t* dof_of, const float* bc,
                                float* xc, const float* x, const float* b, float* x_out, float w0, float w1, float w2,
                                hipStream_t s) {
    return block_post_cg_t<float>(L, C, dof_of, bc, xc, x, b, x_out, w0, w1, w2, s);
}

hipError_t launch_block_post_cg(const LevelView& L, const CoarsestView& C, const int32_t* dof_of, const bf16* bc,
                                bf16* xc, const bf16* x, const bf16* b, bf16* x_out, float w0, float w1, float w2,
                                hipStream_t s) {
    return block_post_cg_t<bf16>(L, C, dof_of, bc, xc, x, b, x_out, w0, w1, w2, s);
}

}  // namespace uaamg
