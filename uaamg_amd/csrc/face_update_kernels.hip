// Device pressure-gradient update of the face velocities (face_update.h).
#include "face_update.h"
#include "fraction_inside.h"
#include "stencil_device.h"

namespace uaamg {
namespace {

using namespace dev;

// DOF bits of one x-plane (64 voxels, one mask word) of level-0 DOF leaf dl,
// and the plane's first DOF. The same for the whole wavefront.
struct DofPlane {
    uint64_t word;
    int64_t first;
};
__device__ __forceinline__ DofPlane dof_plane(const GradArgs& a, int32_t dl, int x) {
    if (dl < 0) return {0, 0};
    const uint64_t* m = a.dmask + size_t(dl) * 8;
    int64_t k = a.dofbase[dl];
#pragma unroll
    for (int i = 0; i < 7; ++i) k += i < x ? __popcll(m[i]) : 0;
    return {m[x], k};
}

// pressure at a voxel of a plane: (is a DOF, value; 0 off the DOFs)
__device__ __forceinline__ bool pressure_at(const GradArgs& a, const DofPlane& d, int bit, float& p) {
    p = 0.f;
    if (!((d.word >> bit) & 1u)) return false;
    p = a.pressure[d.first + __popcll(d.word & ((uint64_t(1) << bit) - 1))];
    return true;
}

// One wavefront per x-plane of a velocity leaf, a lane per voxel: every access
// to a vector is consecutive, the plane's masks are one word, and a lane's
// loads do not wait for each other. 72 us a channel at 13115 leaves, where a
// lane per z-row stepping through its eight voxels took 326. 240 MB pass
// through HBM (every channel reads the weights' three components), 3.3 TB/s,
// two thirds of a copy's rate; a wavefront waits for three quarters of its life.
__global__ __launch_bounds__(kBlockThreads) void pressure_gradient_kernel(int64_t nleaf, GradArgs a, uint64_t* active,
                                                                          float* vel, float* upd, float* refl) {
    const int gw = __builtin_amdgcn_readfirstlane(logical_block() * kWavesPerBlock + int(threadIdx.x >> 6));
    const int leaf = gw >> 3, lx = gw & 7;
    if (leaf >= nleaf) return;
    const int lane = threadIdx.x & 63, ly = lane >> 3, lz = lane & 7;
    const int off = lx * 64 + lane;
    const int c = a.channel;
    const int32_t* t = a.tab + size_t(leaf) * kGradTab;
    const uint64_t word = active[size_t(leaf) * 8 + lx];
    // the planes of the voxel and of the one below along c: inside the leaf, and past its low face
    const DofPlane here = dof_plane(a, t[kGradDof], lx);
    const DofPlane in = c == 0 && lx > 0 ? dof_plane(a, t[kGradDof], lx - 1) : here;
    const DofPlane past = dof_plane(a, t[kGradDofLow], c == 0 ? 7 : lx);
    const size_t at = size_t(leaf) * 512 + off;
    const float u0 = vel[at];
    float updated = u0, reflected = u0, du = 0.f;
    bool has_update = false;
    if ((word >> lane) & 1u) {
        // the voxel below along c: same leaf, or the -e_c neighbour at local coordinate 7
        const bool below_in = (c == 0 ? lx : (c == 1 ? ly : lz)) > 0;
        const int step = c == 0 ? 64 : (c == 1 ? 8 : 1);
        const int off_b = below_in ? off - step : off + 7 * step;
        const int32_t pl = below_in ? t[kGradPhi] : t[kGradPhiLow];
        const float weight = t[kGradW] >= 0 ? a.w[(size_t(t[kGradW]) * 512 + off) * 3 + c] : a.w_bg[c];
        const float phi_this = t[kGradPhi] >= 0 ? a.phi[size_t(t[kGradPhi]) * 512 + off] : a.phi_bg;
        const float phi_below = pl >= 0 ? a.phi[size_t(pl) * 512 + off_b] : a.phi_bg;
        float p_this, p_below;
        const bool has_p = pressure_at(a, here, lane, p_this);
        const bool has_pb = pressure_at(a, below_in ? in : past, off_b & 63, p_below);
        if (weight > 0.0f && (has_p || has_pb)) {
            has_update = true;
            float theta = 1.0f;
            if (phi_this >= 0 || phi_below >= 0) {
                theta = fraction_inside2(phi_below, phi_this);
                if (theta < 0.02f) theta = 0.02f;
            }
            du = -a.dt * (p_this - p_below) / a.dx / theta;
            updated += du;
            reflected = updated + du;
            if (weight < 1.0f) {
                const float svel =
                    t[kGradSolid] >= 0 ? a.sv[(size_t(t[kGradSolid]) * 512 + off) * 3 + c] : a.sv_bg[c];
                const float solid_fraction = (1.0f - weight) * a.friction;
                updated = (1.0f - solid_fraction) * updated + solid_fraction * svel;
            }
        }
    }
    if (has_update) vel[at] = updated;
    if (upd) upd[at] = has_update ? du : u0;
    if (refl) refl[at] = has_update ? reflected : u0;
    const uint64_t out_mask = __ballot(has_update);
    if (lane == 0) active[size_t(leaf) * 8 + lx] = out_mask;
}

}  // namespace

hipError_t launch_pressure_gradient(int64_t nleaf, const GradArgs& a, uint64_t* active, float* vel, float* upd,
                                    float* refl, hipStream_t s) {
    if (nleaf <= 0) return hipSuccess;
    if (nleaf > int64_t(INT32_MAX) / 64) return hipErrorInvalidValue;
    static_assert(8 % kWavesPerBlock == 0, "whole blocks of a leaf's planes");
    pressure_gradient_kernel<<<unsigned(nleaf * (8 / kWavesPerBlock)), kBlockThreads, 0, s>>>(nleaf, a, active, vel, upd, refl);
    return hipGetLastError();
}

}  // namespace uaamg
