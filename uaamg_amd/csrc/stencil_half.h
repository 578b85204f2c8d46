// The 7-point stencil on half rows: a wavefront works on half a leaf (x 0-3 or
// 4-7), two lanes per z-row of four values each (lane = 2 * row + half).
//
// A wavefront's load is then 1 KiB of consecutive bytes (eight cache lines)
// where the full-row form's two 16-byte loads per lane each touch all sixteen
// lines of the brick, and a lane holds half the operands, so twice the
// wavefronts fit a SIMD. The value across the middle of a row comes from the
// other lane of the pair. Same terms, same order as stencil_device.h.
#pragma once

#include "stencil_device.h"

namespace uaamg {
namespace dev {

// (leaf, half) of the wavefront; row (0 .. 63) and first z (0 or 4) of the lane
struct HalfPos {
    int leaf, row, z0;
};
template <int kWaves = kWavesPerBlock>
__device__ __forceinline__ HalfPos half_pos() {
    const int w = logical_block() * kWaves + int(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    HalfPos p;
    p.leaf = __builtin_amdgcn_readfirstlane(w >> 1);
    p.row = (__builtin_amdgcn_readfirstlane(w & 1) << 5) | (lane >> 1);
    p.z0 = (lane & 1) * 4;
    return p;
}
inline unsigned half_grid(int32_t nleaf, int waves = kWavesPerBlock) {
    return unsigned((2 * int64_t(nleaf) + waves - 1) / waves);
}

// v of the other lane of the pair
__device__ __forceinline__ float pair_swap(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xb1, 0xf, 0xf, true));   // [1,0,3,2]
}

template <class V>
__device__ __forceinline__ void ldh(const V* p, float v[4]) {
    const float4 a = ld4(p);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}
__device__ __forceinline__ void sth(float* p, const float v[4]) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void sth(bf16* p, const float v[4]) {
    *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
}
__device__ __forceinline__ void fillh(float v[4], float c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = c;
}
__device__ __forceinline__ void ldh_slot(const float* base, int slot, int off, float dflt, float v[4]) {
    if (slot >= 0) ldh(base + size_t(slot) * 512 + off, v);
    else fillh(v, dflt);
}
// DOF bits of the lane's whole row
__device__ __forceinline__ uint32_t half_row_mask(const LevelView& L, const HalfPos& p) {
    return reinterpret_cast<const uint8_t*>(L.mask)[size_t(p.leaf) * 64 + p.row];
}

// Sources of the vector the stencil is applied to. A source loads its raw
// operands for four voxels or one (of a leaf that exists, with that leaf's
// diagonal slot sd and parent par), and forms the values from them later:
// nothing waits for a load before the loads of all sides are issued. (With
// the values formed side by side, the first two sweeps from zero took 184 us
// at 92428 leaves and the sweep after the prolongation 204.)

// the stored brick vector (PlainSrcT)
template <class V>
struct PlainHalf {
    struct Quad {
        float v[4];
    };
    struct One {
        float v;
    };
    const V* X;
    __device__ __forceinline__ void load(int leaf, int, int, int off, Quad& q) const {
        ldh(X + size_t(leaf) * 512 + off, q.v);
    }
    __device__ __forceinline__ void load(int leaf, int, int, int off, One& q) const {
        q.v = ld1(X + size_t(leaf) * 512 + off);
    }
    __device__ __forceinline__ float value(const Quad& q, int z) const { return q.v[z]; }
    __device__ __forceinline__ float value(const One& q) const { return q.v; }
};

// x1 = w0 * D^-1 b (FirstJacobiSrcT)
template <class VB>
struct FirstHalf {
    struct Quad {
        float b[4], inv[4];
    };
    struct One {
        float b, inv;
    };
    const VB* B;
    const float* invdiag;
    float dflt_inv, w0;
    __device__ __forceinline__ void load(int leaf, int sd, int, int off, Quad& q) const {
        ldh(B + size_t(leaf) * 512 + off, q.b);
        ldh_slot(invdiag, sd, off, dflt_inv, q.inv);
    }
    __device__ __forceinline__ void load(int leaf, int sd, int, int off, One& q) const {
        q.b = ld1(B + size_t(leaf) * 512 + off);
        q.inv = sd >= 0 ? invdiag[size_t(sd) * 512 + off] : dflt_inv;
    }
    __device__ __forceinline__ float value(const Quad& q, int z) const { return w0 * (q.inv[z] * q.b[z]); }
    __device__ __forceinline__ float value(const One& q) const { return w0 * (q.inv * q.b); }
};

// x + P x_coarse on DOF voxels (ProlongSrcT)
template <class V>
struct ProlongHalf {
    struct Quad {
        float x[4], c[2];
        uint32_t m;   // voxels that take the coarse value
    };
    struct One {
        float x, c;
        uint32_t m;
    };
    const V* X;
    const V* Xc;
    const uint64_t* mask;
    __device__ __forceinline__ uint32_t bits(int leaf, int off) const {
        return uint32_t(reinterpret_cast<const uint8_t*>(mask)[size_t(leaf) * 64 + (off >> 3)]) >> (off & 7);
    }
    __device__ __forceinline__ size_t coarse(int par, int off) const {
        const int cl = par >> 3, oct = par & 7;
        const int crow = ((off >> 7) + 4 * ((oct >> 2) & 1)) * 8 + (((off >> 4) & 3) + 4 * ((oct >> 1) & 1));
        return size_t(cl) * 512 + crow * 8 + 4 * (oct & 1) + ((off & 7) >> 1);
    }
    static __device__ __forceinline__ void ld2(const float* p, float v[2]) {
        const float2 a = *reinterpret_cast<const float2*>(p);
        v[0] = a.x; v[1] = a.y;
    }
    static __device__ __forceinline__ void ld2(const bf16* p, float v[2]) {
        const uint32_t a = *reinterpret_cast<const uint32_t*>(p);
        v[0] = __uint_as_float(a << 16);
        v[1] = __uint_as_float(a & 0xffff0000u);
    }
    // par < 0 (a bounds guard: every DOF leaf has a parent) reads coarse leaf 0 and adds nothing
    __device__ __forceinline__ void load(int leaf, int, int par, int off, Quad& q) const {
        ldh(X + size_t(leaf) * 512 + off, q.x);
        ld2(Xc + coarse(par >= 0 ? par : 0, off), q.c);
        q.m = par >= 0 ? bits(leaf, off) : 0u;
    }
    __device__ __forceinline__ void load(int leaf, int, int par, int off, One& q) const {
        q.x = ld1(X + size_t(leaf) * 512 + off);
        q.c = ld1(Xc + coarse(par >= 0 ? par : 0, off));
        q.m = par >= 0 ? bits(leaf, off) : 0u;
    }
    __device__ __forceinline__ float value(const Quad& q, int z) const {
        const float t = q.x[z] + q.c[z >> 1];
        return ((q.m >> z) & 1u) ? t : q.x[z];
    }
    __device__ __forceinline__ float value(const One& q) const {
        const float t = q.x + q.c;
        return (q.m & 1u) ? t : q.x;
    }
};

// p' = z + beta p (levelXPlusAlphaY, simd_vdb_poisson.cpp:2305-2320), both 0 off the DOFs
struct UpdateHalf {
    struct Quad {
        float z[4], p[4];
    };
    struct One {
        float z, p;
    };
    const float* Z;
    const float* P;
    float beta;
    __device__ __forceinline__ void load(int leaf, int, int, int off, Quad& q) const {
        ldh(Z + size_t(leaf) * 512 + off, q.z);
        ldh(P + size_t(leaf) * 512 + off, q.p);
    }
    __device__ __forceinline__ void load(int leaf, int, int, int off, One& q) const {
        q.z = Z[size_t(leaf) * 512 + off];
        q.p = P[size_t(leaf) * 512 + off];
    }
    __device__ __forceinline__ float value(const Quad& q, int z) const {
        const float t = beta * q.p[z];
        return q.z[z] + t;
    }
    __device__ __forceinline__ float value(const One& q) const {
        const float t = beta * q.p;
        return q.z + t;
    }
};

// Own operands c and values xc of the source and the off-diagonal sum of the
// stencil for the lane's four voxels (every lane of the wavefront must be
// active). With kTiles leaves a workgroup (0: none shared) the values inside
// the leaf come from LDS, where its two wavefronts put them once, and so does
// the value past a row's end where the workgroup holds the z-neighbour, one
// brick line a lane otherwise; only rows beyond the x and y faces are loaded. Every thread of the workgroup must call it.
template <int kTiles, class Src>
__device__ __forceinline__ void half_offdiag(const LevelView& L, const LeafRec& R, const Src& src, const HalfPos& p,
                                             float (*tiles)[512], typename Src::Quad& c, float xc[4], float s[4]) {
    const int row = p.row, lx = row >> 3, ly = row & 7, z0 = p.z0;
    const int off = row * 8 + z0;
    // an absent neighbour leaf reads the own leaf instead and counts as 0
    typename Src::Quad sq[4];
    bool have[4];
    const bool own[4] = {lx > 0, lx < 7, ly > 0, ly < 7};   // -x, +x, -y, +y inside the leaf
    const int o_own[4] = {off - 64, off + 64, off - 8, off + 8}, o_nb[4] = {off + 448, off - 448, off + 56, off - 56};
    src.load(p.leaf, R.sd, R.par, off, c);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        have[k] = own[k] || R.nb[k] >= 0;
        const bool nb = !own[k] && R.nb[k] >= 0;
        if (!kTiles || nb)
            src.load(nb ? R.nb[k] : p.leaf, nb ? R.nbsd[k] : R.sd, nb ? R.nbpar[k] : R.par,
                     own[k] ? o_own[k] : o_nb[k], sq[k]);
    }
    // the value past the row's end on the lane's side of the brick
    const bool hi = z0 != 0;
    const int nz = hi ? R.nb[5] : R.nb[4];
    typename Src::One oq;
    // (one brick line a lane: from LDS where the workgroup holds the neighbour too)
    const int first = kTiles > 0 ? logical_block() * kTiles : 0;
    const bool nz_in = kTiles > 0 && nz >= first && nz < first + kTiles;
    if (!nz_in) src.load(nz >= 0 ? nz : p.leaf, nz >= 0 ? (hi ? R.nbsd[5] : R.nbsd[4]) : R.sd,
             nz >= 0 ? (hi ? R.nbpar[5] : R.nbpar[4]) : R.par, row * 8 + (hi ? 0 : 7), oq);
    float cxm[4], cxp[4], cym[4], cyp[4], cz[4];
    const float d = L.dflt_off;
    ldh_slot(L.cx, R.sx, off, d, cxm);
    ldh_slot(L.cx, lx < 7 ? R.sx : R.sxp, lx < 7 ? off + 64 : off - 448, d, cxp);
    ldh_slot(L.cy, R.sy, off, d, cym);
    ldh_slot(L.cy, ly < 7 ? R.sy : R.syp, ly < 7 ? off + 8 : off - 56, d, cyp);
    ldh_slot(L.cz, R.sz, off, d, cz);
    const float czout = R.szp >= 0 ? L.cz[size_t(R.szp) * 512 + row * 8] : d;
#pragma unroll
    for (int z = 0; z < 4; ++z) xc[z] = src.value(c, z);
    float v[4][4];
    if constexpr (kTiles > 0) {
        float* tile = tiles[threadIdx.x >> 7];
        sth(tile + off, xc);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            ldh(tile + (own[k] ? o_own[k] : off), v[k]);
            if (!own[k]) {
#pragma unroll
                for (int z = 0; z < 4; ++z) v[k][z] = have[k] ? src.value(sq[k], z) : 0.f;
            }
        }
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int z = 0; z < 4; ++z) v[k][z] = have[k] ? src.value(sq[k], z) : 0.f;
    }
    float zout = nz >= 0 && !nz_in ? src.value(oq) : 0.f;
    if constexpr (kTiles > 0)
        if (nz_in) zout = tiles[nz - first][row * 8 + (hi ? 0 : 7)];
    const float xo = pair_swap(hi ? xc[0] : xc[3]), co = pair_swap(cz[0]);
    const float zm = hi ? xo : zout, zp = hi ? zout : xo, czp = hi ? czout : co;
#pragma unroll
    for (int z = 0; z < 4; ++z) {
        const float f1 = v[1][z] * cxp[z];
        const float f2 = v[0][z] * cxm[z];
        const float f3 = v[3][z] * cyp[z];
        const float f4 = v[2][z] * cym[z];
        const float f5 = (z < 3 ? xc[z + 1] : zp) * (z < 3 ? cz[z + 1] : czp);
        const float f6 = (z > 0 ? xc[z - 1] : zm) * cz[z];
        s[z] = ((f1 + f2) + (f3 + f4)) + (f5 + f6);
    }
}

// The remaining operands of a Jacobi sweep on the lane's voxels. Loaded behind
// the off-diagonal sum's barrier they cost a second memory latency; loaded
// before it, registers and with them wavefronts. At 92428 leaves, behind /
// before: the first two sweeps 149 / 143 us, the step's diagonal 270 / 258; but
// the plain sweep 132 / 132, with its dot product 142 / 145, and the one after
// the prolongation 180 / 211 (72 / 82 registers: six wavefronts a SIMD / five).
struct JacobiHalf {
    float dg[4], inv[4], b[4];
    template <class VB>
    __device__ __forceinline__ void load(const LevelView& L, const LeafRec& R, const HalfPos& p, const VB* B) {
        const int off = p.row * 8 + p.z0;
        ldh(B + size_t(p.leaf) * 512 + off, b);
        ldh_slot(L.diag, R.sd, off, L.dflt_diag, dg);
        ldh_slot(L.invdiag, R.sd, off, L.dflt_invdiag, inv);
    }
    // weighted Jacobi, 0 off the DOFs (jacobi_row, mask_row)
    __device__ __forceinline__ void sweep(const float xc[4], const float s[4], float w, uint32_t m, float y[4]) const {
#pragma unroll
        for (int z = 0; z < 4; ++z) {
            const float ax = fmaf(xc[z], dg[z], s[z]);
            float r = b[z] - ax;
            r = r * inv[z];
            const float v = fmaf(w, r, xc[z]);
            y[z] = ((m >> z) & 1u) ? v : 0.f;
        }
    }
};

}  // namespace dev
}  // namespace uaamg
