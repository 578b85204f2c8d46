// Device-side building blocks of the viscosity kernels: row loads and stores,
// wave records, and the fetch of a vector's or a coefficient grid's row at a
// voxel offset.
#pragma once

#include "stencil_device.h"
#include "viscosity_host.h"
#include "viscosity_kernels.h"

namespace uaamg {
namespace dev {

constexpr int nb_slot(int ax, int ay, int az) { return (ax + 1) * 9 + (ay + 1) * 3 + (az + 1); }

__device__ __forceinline__ int row_off(int X, int Y) { return ((X & 7) * 8 + (Y & 7)) * 8; }

__device__ __forceinline__ void ld8v(const float* p, float v[8]) {
    const float4 a = *reinterpret_cast<const float4*>(p);
    const float4 b = *reinterpret_cast<const float4*>(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ void st8v(float* p, const float v[8]) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
    *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}
// BF16-stored level vectors of the mixed form: a z-row is 16 bytes, widened
// exactly on load, rounded to nearest even on store; arithmetic stays FP32
__device__ __forceinline__ void ld8v(const bf16* p, float v[8]) { ld8(p, v); }
__device__ __forceinline__ void st8v(bf16* p, const float v[8]) { st8(p, v); }
__device__ __forceinline__ float ld1v(const float* p) { return *p; }
__device__ __forceinline__ float ld1v(const bf16* p) { return float(*p); }
__device__ __forceinline__ void st1v(float* p, float v) { *p = v; }
__device__ __forceinline__ void st1v(bf16* p, float v) { *p = bf16(v); }

// A wave record (layout at kVRecLeaf) in scalar registers.
struct VRec {
    int leaf;
    int nb[27];
    int own[14];
    int nbs[7];
};

__device__ __forceinline__ VRec load_vrec(const ViscLevelView& L, int e) {
    const int4* p = reinterpret_cast<const int4*>(L.wrec + size_t(e) * kVRec);
    int v[52];
#pragma unroll
    for (int i = 0; i < 13; ++i) {
        const int4 q = p[i];
        v[4 * i] = q.x; v[4 * i + 1] = q.y; v[4 * i + 2] = q.z; v[4 * i + 3] = q.w;
    }
    VRec r;
    r.leaf = v[kVRecLeaf];
#pragma unroll
    for (int k = 0; k < 27; ++k) r.nb[k] = v[kVRecNb + k];
#pragma unroll
    for (int k = 0; k < 14; ++k) r.own[k] = v[kVRecOwn + k];
#pragma unroll
    for (int k = 0; k < 7; ++k) r.nbs[k] = v[kVRecNbr + k];
    // One use of every field here, in the kernel's first basic block: the
    // record's scalar loads are then issued together and waited for once
    // (otherwise each is issued in the branch that first reads it). The
    // empty asm emits no instruction.
    int all = 0;
#pragma unroll
    for (int k = 0; k < 49; ++k) all ^= v[k];
    asm volatile("" ::"s"(all));
    return r;
}

// Leaf holding leaf-local row (lx + OX, ly + OY), shifted AZ leaves in z:
// one of four record entries chosen per lane.
template <int OX, int OY, int AZ>
__device__ __forceinline__ int vleaf(const VRec& R, int lx, int ly) {
    constexpr int sx = (OX > 0) - (OX < 0), sy = (OY > 0) - (OY < 0);
    const int X = lx + OX, Y = ly + OY;
    const bool ox = X < 0 || X > 7, oy = Y < 0 || Y > 7;
    const int l00 = R.nb[nb_slot(0, 0, AZ)], l10 = R.nb[nb_slot(sx, 0, AZ)];
    const int l01 = R.nb[nb_slot(0, sy, AZ)], l11 = R.nb[nb_slot(sx, sy, AZ)];
    return ox ? (oy ? l11 : l10) : (oy ? l01 : l00);
}

// channel ch of vector v at (lx + OX, ly + OY, z + OZ), z = 0..7 (a missing
// leaf, or one without vector bricks, reads 0)
template <int OX, int OY, int OZ, class V>
__device__ __forceinline__ void vfetch(const ViscLevelView& L, const V* v, int ch, const VRec& R, int lx, int ly,
                                       float out[8]) {
    const int X = lx + OX, Y = ly + OY;
    const int lf = vleaf<OX, OY, 0>(R, lx, ly);
    float row[8];
    if (lf >= 0 && lf < L.nleaf_dof) ld8v(v + (size_t(lf) * 3 + ch) * 512 + row_off(X, Y), row);
    else {
#pragma unroll
        for (int k = 0; k < 8; ++k) row[k] = 0.f;
    }
    if (OZ == 0) {
#pragma unroll
        for (int k = 0; k < 8; ++k) out[k] = row[k];
    } else if (OZ > 0) {
#pragma unroll
        for (int k = 0; k < 7; ++k) out[k] = row[k + 1];
        const int lz = vleaf<OX, OY, 1>(R, lx, ly);
        out[7] = (lz >= 0 && lz < L.nleaf_dof) ? ld1v(v + (size_t(lz) * 3 + ch) * 512 + row_off(X, Y)) : 0.f;
    } else {
#pragma unroll
        for (int k = 7; k > 0; --k) out[k] = row[k - 1];
        const int lz = vleaf<OX, OY, -1>(R, lx, ly);
        out[0] = (lz >= 0 && lz < L.nleaf_dof) ? ld1v(v + (size_t(lz) * 3 + ch) * 512 + row_off(X, Y) + 7) : 0.f;
    }
}

// coefficient grid GID at (lx + OX, ly + OY, z + OZ), at most one offset
// nonzero: rows inside the leaf read slot s_own, rows (or the shifted z
// value) beyond the face read s_nb; slot -1 reads the level default
template <int GID, int OX, int OY, int OZ>
__device__ __forceinline__ void cfetch(const ViscLevelView& L, int s_own, int s_nb, int lx, int ly, float out[8]) {
    static_assert((OX != 0) + (OY != 0) + (OZ != 0) <= 1, "single-axis coefficient offsets");
    const int X = lx + OX, Y = ly + OY;
    const bool beyond = X < 0 || X > 7 || Y < 0 || Y > 7;
    const int s = beyond ? s_nb : s_own;
    const float m = L.dflt[GID];
    float row[8];
    if (s >= 0) ld8v(L.pool + size_t(s) * 512 + row_off(X, Y), row);
    else {
#pragma unroll
        for (int k = 0; k < 8; ++k) row[k] = m;
    }
    if (OZ == 0) {
#pragma unroll
        for (int k = 0; k < 8; ++k) out[k] = row[k];
    } else if (OZ > 0) {
#pragma unroll
        for (int k = 0; k < 7; ++k) out[k] = row[k + 1];
        out[7] = s_nb >= 0 ? L.pool[size_t(s_nb) * 512 + row_off(X, Y)] : m;
    } else {
#pragma unroll
        for (int k = 7; k > 0; --k) out[k] = row[k - 1];
        out[0] = s_nb >= 0 ? L.pool[size_t(s_nb) * 512 + row_off(X, Y) + 7] : m;
    }
}

template <int A>
struct Unit {
    static constexpr int x = A == 0, y = A == 1, z = A == 2;
};

}  // namespace dev
}  // namespace uaamg
