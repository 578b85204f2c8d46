// The viscosity level above the coarsest as rows (visc_rows.h): the build of
// the rows from the level's bricks, and the visits.
#include "visc_rows.h"

#include "visc_coarsest_device.h"
#include "viscosity_device.h"

namespace uaamg {
namespace {

using namespace dev;

constexpr int kRowThreads = kVCgThreads;

// ------------------------------------------------------------------ build
// Maps hold row number + 1 as a float per brick entry (0: no DOF), so the
// fetch routines of the level kernels find a neighbour's row where they would
// find its value (a missing leaf reads 0).

// one wavefront per (leaf, channel) brick
__global__ __launch_bounds__(64) void rows_number_kernel(const uint64_t* mask, const int32_t* base, float* map,
                                                         int32_t* pos) {
    const int brick = blockIdx.x, lane = threadIdx.x;
    const int lx = lane >> 3, ly = lane & 7;
    const uint32_t m = uint32_t(mask[size_t(brick) * 8 + lx] >> (ly * 8)) & 0xffu;
    const uint32_t red = ((lx + ly) & 1) ? 0xaau : 0x55u;
    int count = __popc(m & red) | (__popc(m & ~red) << 16);
    const int own = count;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(count, o);
        if (lane >= o) count += t;
    }
    count -= own;
    int r[2] = {base[brick * 2] + (count & 0xffff), base[brick * 2 + 1] + (count >> 16)};
    for (int z = 0; z < 8; ++z) {
        const int off = lane * 8 + z;
        float v = 0.f;
        if ((m >> z) & 1u) {
            const int c = ((red >> z) & 1u) ? 0 : 1;
            pos[r[c]] = brick * 512 + off;
            v = float(++r[c]);
        }
        map[size_t(brick) * 512 + off] = v;
    }
}

__global__ void rows_coarse_map_kernel(int n, const int32_t* pos, float* map) {
    const int d = blockIdx.x * blockDim.x + threadIdx.x;
    if (d < n) map[pos[d]] = float(d + 1);
}

__global__ void rows_zero_kernel(size_t n, float* p) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.f;
}

__device__ __forceinline__ uint32_t row_id(float v, int none) { return v > 0.f ? uint32_t(v) - 1u : uint32_t(none); }

// one wavefront per wave record of channel C: the operands of visc_row, in its order
template <int C>
__device__ __forceinline__ void rows_fill(const ViscLevelView& L, const ViscRowsView& R, const float* map,
                                          const float* cmap, int e) {
    const int lane = threadIdx.x & 63, lx = lane >> 3, ly = lane & 7;
    const VRec W = load_vrec(L, e);
    constexpr int d0 = C, d1 = (C + 1) % 3, d2 = (C + 2) % 3;
    using E0 = Unit<d0>;
    using E1 = Unit<d1>;
    using E2 = Unit<d2>;
    constexpr int kN0 = kVNeg + 3 * C, kX2 = kVCross + 4 * d2, kX1 = kVCross + 4 * d1;
    float own[8];
    vfetch<0, 0, 0>(L, map, C, W, lx, ly, own);
    auto put = [&](int k, const float id[8], const float c[8]) {
        for (int z = 0; z < 8; ++z) {
            if (!(own[z] > 0.f)) continue;
            const size_t row = size_t(own[z]) - 1;
            reinterpret_cast<float*>(R.coef + size_t(k >> 2) * size_t(R.np) + row)[k & 3] = c[z];
            reinterpret_cast<uint16_t*>(R.idx + size_t(k >> 3) * size_t(R.np) + row)[k & 7] =
                uint16_t(row_id(id[z], R.n));
        }
    };
    float v[8], c[8];
    vfetch<1, 0, 0>(L, map, C, W, lx, ly, v);
    cfetch<kN0 + 0, 1, 0, 0>(L, W.own[0], W.nbs[0], lx, ly, c);
    put(0, v, c);
    vfetch<-1, 0, 0>(L, map, C, W, lx, ly, v);
    cfetch<kN0 + 0, 0, 0, 0>(L, W.own[0], -1, lx, ly, c);
    put(1, v, c);
    vfetch<0, 1, 0>(L, map, C, W, lx, ly, v);
    cfetch<kN0 + 1, 0, 1, 0>(L, W.own[1], W.nbs[1], lx, ly, c);
    put(2, v, c);
    vfetch<0, -1, 0>(L, map, C, W, lx, ly, v);
    cfetch<kN0 + 1, 0, 0, 0>(L, W.own[1], -1, lx, ly, c);
    put(3, v, c);
    vfetch<0, 0, 1>(L, map, C, W, lx, ly, v);
    cfetch<kN0 + 2, 0, 0, 1>(L, W.own[2], W.nbs[2], lx, ly, c);
    put(4, v, c);
    vfetch<0, 0, -1>(L, map, C, W, lx, ly, v);
    cfetch<kN0 + 2, 0, 0, 0>(L, W.own[2], -1, lx, ly, c);
    put(5, v, c);
    vfetch<0, 0, 0>(L, map, d1, W, lx, ly, v);
    cfetch<kX2 + 0, 0, 0, 0>(L, W.own[3], -1, lx, ly, c);
    put(6, v, c);
    vfetch<E1::x, E1::y, E1::z>(L, map, d1, W, lx, ly, v);
    cfetch<kX2 + 1, 0, 0, 0>(L, W.own[4], -1, lx, ly, c);
    put(7, v, c);
    vfetch<-E0::x, -E0::y, -E0::z>(L, map, d1, W, lx, ly, v);
    cfetch<kX2 + 2, -E0::x, -E0::y, -E0::z>(L, W.own[5], W.nbs[3], lx, ly, c);
    put(8, v, c);
    vfetch<E1::x - E0::x, E1::y - E0::y, E1::z - E0::z>(L, map, d1, W, lx, ly, v);
    cfetch<kX2 + 3, -E0::x, -E0::y, -E0::z>(L, W.own[6], W.nbs[4], lx, ly, c);
    put(9, v, c);
    vfetch<0, 0, 0>(L, map, d2, W, lx, ly, v);
    cfetch<kX1 + 0, 0, 0, 0>(L, W.own[7], -1, lx, ly, c);
    put(10, v, c);
    vfetch<-E0::x, -E0::y, -E0::z>(L, map, d2, W, lx, ly, v);
    cfetch<kX1 + 1, -E0::x, -E0::y, -E0::z>(L, W.own[8], W.nbs[5], lx, ly, c);
    put(11, v, c);
    vfetch<E2::x, E2::y, E2::z>(L, map, d2, W, lx, ly, v);
    cfetch<kX1 + 2, 0, 0, 0>(L, W.own[9], -1, lx, ly, c);
    put(12, v, c);
    vfetch<E2::x - E0::x, E2::y - E0::y, E2::z - E0::z>(L, map, d2, W, lx, ly, v);
    cfetch<kX1 + 3, -E0::x, -E0::y, -E0::z>(L, W.own[10], W.nbs[6], lx, ly, c);
    put(13, v, c);
    float inv[8], dg[8];
    cfetch<kVInvDiag + C, 0, 0, 0>(L, W.own[12], -1, lx, ly, inv);
    cfetch<kVDiag + C, 0, 0, 0>(L, W.own[11], -1, lx, ly, dg);
    const int p = L.parent[W.leaf];
    for (int z = 0; z < 8; ++z) {
        if (!(own[z] > 0.f)) continue;
        const size_t row = size_t(own[z]) - 1;
        float* cf = reinterpret_cast<float*>(R.coef + 3 * size_t(R.np) + row);
        cf[2] = inv[z];
        cf[3] = dg[z];
        uint32_t par = uint32_t(R.nc);
        if (p >= 0) {
            const int cl = p >> 3, oct = p & 7;
            const int cx = ((oct >> 2) & 1) * 4 + (lx >> 1), cy = ((oct >> 1) & 1) * 4 + (ly >> 1);
            const int cz = (oct & 1) * 4 + (z >> 1);
            par = row_id(cmap[(size_t(cl) * 3 + C) * 512 + cx * 64 + cy * 8 + cz], R.nc);
        }
        uint16_t* ix = reinterpret_cast<uint16_t*>(R.idx + size_t(R.np) + row);
        ix[6] = uint16_t(par);
        ix[7] = 0;
    }
}

__global__ __launch_bounds__(64) void rows_fill_kernel(ViscLevelView L, ViscRowsView R, const float* map,
                                                       const float* cmap) {
    const int e = blockIdx.x;
    if (e < L.chan_off[1]) rows_fill<0>(L, R, map, cmap, e);
    else if (e < L.chan_off[2]) rows_fill<1>(L, R, map, cmap, e);
    else rows_fill<2>(L, R, map, cmap, e);
}

// the eight children of each coarse row, in the restriction's order
__global__ void rows_child_kernel(ViscLevelView Cl, ViscRowsView R, const int32_t* cpos, const float* map) {
    const int d = blockIdx.x * blockDim.x + threadIdx.x;
    if (d >= R.nc) return;
    const int brick = cpos[d] >> 9, off = cpos[d] & 511;
    const int leaf = brick / 3, c = brick - 3 * leaf;
    const int lx = off >> 6, ly = (off >> 3) & 7, lz = off & 7;
    const int f = Cl.child[size_t(leaf) * 8 + (((lx >> 2) << 2) | ((ly >> 2) << 1) | (lz >> 2))];
    uint16_t* ch = reinterpret_cast<uint16_t*>(R.child + d);
    for (int k = 0; k < 8; ++k) {
        const int x = 2 * (lx & 3) + (k >> 2), y = 2 * (ly & 3) + ((k >> 1) & 1), z = 2 * (lz & 3) + (k & 1);
        ch[k] = uint16_t(f >= 0 ? row_id(map[(size_t(f) * 3 + c) * 512 + x * 64 + y * 8 + z], R.n) : uint32_t(R.n));
    }
}

// ------------------------------------------------------------------ visit
// value as the level vector's storage type holds it
template <class V>
__device__ __forceinline__ float stored(float v) {
    if constexpr (sizeof(V) == 4) return v;
    else return float(V(v));
}

// one row's operands
struct Row {
    float4 c[4];
    uint4 i[2];
    float b;
};

__device__ __forceinline__ Row load_row(const ViscRowsView& R, int row) {
    Row q;
#pragma unroll
    for (int k = 0; k < 4; ++k) q.c[k] = R.coef[size_t(k) * size_t(R.np) + size_t(row)];
#pragma unroll
    for (int k = 0; k < 2; ++k) q.i[k] = R.idx[size_t(k) * size_t(R.np) + size_t(row)];
    q.b = R.b[row];
    return q;
}

// the off-diagonal sum of a row: terms and order of visc_row
__device__ __forceinline__ float row_sum(const Row& q, const float* xs) {
    auto at = [&](uint32_t w, int h) { return xs[h ? (w >> 16) : (w & 0xffffu)]; };
    float s;
    {
        const float f1 = at(q.i[0].x, 0) * q.c[0].x, f2 = at(q.i[0].x, 1) * q.c[0].y;
        const float f3 = at(q.i[0].y, 0) * q.c[0].z, f4 = at(q.i[0].y, 1) * q.c[0].w;
        const float f5 = at(q.i[0].z, 0) * q.c[1].x, f6 = at(q.i[0].z, 1) * q.c[1].y;
        const float t = (f1 + f2) + (f3 + f4);
        s = t + (f5 + f6);
    }
    {
        const float a = at(q.i[0].w, 0) * q.c[1].z, b = at(q.i[0].w, 1) * q.c[1].w;
        const float c = at(q.i[1].x, 0) * q.c[2].x, d = at(q.i[1].x, 1) * q.c[2].y;
        s = s + ((a + b) + (c + d));
    }
    {
        const float a = at(q.i[1].y, 0) * q.c[2].z, b = at(q.i[1].y, 1) * q.c[2].w;
        const float c = at(q.i[1].z, 0) * q.c[3].x, d = at(q.i[1].z, 1) * q.c[3].y;
        s = s + ((a + b) + (c + d));
    }
    return s;
}

// One colour pass over group g, x in LDS. `cur` holds the thread's first row
// of the group; on return it holds its first row of group `next`: a row's
// loads do not depend on x, so they are issued one row ahead, across the
// barrier between passes too.
template <class V>
__device__ __forceinline__ void colour_pass(const ViscRowsView& R, const int* start, float* xs, int g, int next,
                                            Row& cur) {
    const int end = start[g + 1];
    int row = start[g] + int(threadIdx.x);
    for (;;) {
        const bool more = row + kRowThreads < end;
        const int ahead = more ? row + kRowThreads : start[next] + int(threadIdx.x);
        const Row nxt = load_row(R, ahead < R.n ? ahead : 0);
        if (row < end) {
            float t = cur.b - row_sum(cur, xs);
            t = t * cur.c[3].z;
            xs[row] = stored<V>(fmaf(xs[row], 0.0f, t));
        }
        cur = nxt;
        if (!more) break;
        row += kRowThreads;
    }
    __syncthreads();
}

// The visits (see visc_rows.h). Bounded by one CU's rate of reading rows:
// 96 + 4 bytes per row and pass, five passes over all rows per visit.
template <class V, int kPer>
__device__ __forceinline__ void rows_visit(const ViscRowsView& R, const ViscCoarsestView& C, const V* B, V* X,
                                           bool precon, int nvisits) {
    extern __shared__ float sm[];
    __shared__ ViscCgShared cg;
    __shared__ int start[7];
    float* xs = sm;                // [n + 1], the last zero
    float* sz = sm + R.n + 1;      // [nc + 1], the last zero
    const int tid = threadIdx.x;
    if (tid == 0) {
#pragma unroll
        for (int g = 0; g < 7; ++g) start[g] = R.start[g];
        xs[R.n] = 0.f;
        R.r[R.n] = 0.f;
    }
    for (int row = tid; row < R.n; row += kRowThreads) {
        const int p = R.pos[row];
        R.b[row] = ld1v(B + p);
        xs[row] = precon ? 0.f : ld1v(X + p);
    }
    __syncthreads();
#pragma unroll 1
    for (int v = 0; v < nvisits; ++v) {
        Row cur = load_row(R, tid < R.n ? tid : 0);
#pragma unroll 1
        for (int k = 0; k < 12; ++k) colour_pass<V>(R, start, xs, k % 6, (k + 1) % 6, cur);
        // residual of every row
        for (int row = tid; row < R.n; row += kRowThreads) {
            const Row nxt = load_row(R, row + kRowThreads < R.n ? row + kRowThreads : 0);
            const float ax = fmaf(xs[row], cur.c[3].w, row_sum(cur, xs));
            R.r[row] = stored<V>(cur.b - ax);
            cur = nxt;
        }
        __syncthreads();
        // restriction into the coarsest solve, whose solution stays in sz (the
        // empty asm keeps its rows' loads inside the loop over visits)
        ViscCoarsestView Cv = C;
        int at0 = 0;
        asm volatile("" : "+v"(at0));
        Cv.eval += at0;
        Cv.epair += at0;
        Cv.invdiag += at0;
        visc_cg_block<kPer>(
            Cv, sz, cg,
            [&](int d) {
                const uint4 ch = R.child[d];
                float sum = 0.f;
                const uint32_t w[4] = {ch.x, ch.y, ch.z, ch.w};
                float f[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) f[k] = R.r[(k & 1) ? (w[k >> 1] >> 16) : (w[k >> 1] & 0xffffu)];
#pragma unroll
                for (int k = 0; k < 8; ++k) sum += f[k];
                return stored<V>(sum * 0.125f * 0.5f * 2.0f);
            },
            [&](int d, float x) { sz[d] = stored<V>(x); });
        __syncthreads();
        // prolongation
        for (int row = tid; row < R.n; row += kRowThreads)
            xs[row] = stored<V>(xs[row] + sz[R.idx[size_t(R.np) + size_t(row)].w & 0xffffu]);
        cur = load_row(R, start[5] + tid < R.n ? start[5] + tid : 0);
        __syncthreads();
#pragma unroll 1
        for (int k = 0; k < 12; ++k) colour_pass<V>(R, start, xs, 5 - k % 6, 5 - (k + 1) % 6, cur);
    }
    for (int row = tid; row < R.n; row += kRowThreads) st1v(X + R.pos[row], xs[row]);
}

// workgroup i: problem i
template <class V, int kPer>
__global__ __launch_bounds__(kRowThreads) void visc_rows_visit_kernel(const ViscRowsView* __restrict__ views,
                                                                      const ViscCoarsestView* __restrict__ cviews, const V* B, V* X,
                                                                      int precon, int nvisits) {
    rows_visit<V, kPer>(views[blockIdx.x], cviews[blockIdx.x], B, X, precon != 0, nvisits);
}

template <class V, int kPer>
hipError_t visit_per(const ViscRowsView* views, const ViscCoarsestView* cviews, unsigned count, size_t lds, const V* b,
                     V* x, bool precon, int nvisits, hipStream_t s) {
    visc_rows_visit_kernel<V, kPer><<<count, kRowThreads, lds, s>>>(views, cviews, b, x, precon ? 1 : 0, nvisits);
    return hipGetLastError();
}

template <class V>
hipError_t visit(const ViscRowsView* views, const ViscCoarsestView* cviews, int count, int max_n, int max_nc,
                 const V* b, V* x, bool precon, int nvisits, hipStream_t s) {
    if (count <= 0) return hipSuccess;
    if (max_n <= 0 || max_n > kViscRowsMax || max_nc <= 0 || max_nc > kViscMaxCoarsest || nvisits < 1)
        return hipErrorInvalidValue;
    const size_t lds = (size_t(max_n) + size_t(max_nc) + 2) * sizeof(float);
    const unsigned g = unsigned(count);
    if (max_nc <= 2 * kVCgThreads) return visit_per<V, 2>(views, cviews, g, lds, b, x, precon, nvisits, s);
    if (max_nc <= 4 * kVCgThreads) return visit_per<V, 4>(views, cviews, g, lds, b, x, precon, nvisits, s);
    return visit_per<V, 8>(views, cviews, g, lds, b, x, precon, nvisits, s);
}

}  // namespace

hipError_t visc_rows_init() {
    const int most = int((kViscRowsMax + kViscMaxCoarsest + 2) * sizeof(float));
    const void* kernels[] = {reinterpret_cast<const void*>(&visc_rows_visit_kernel<float, 2>),
                             reinterpret_cast<const void*>(&visc_rows_visit_kernel<float, 4>),
                             reinterpret_cast<const void*>(&visc_rows_visit_kernel<float, 8>),
                             reinterpret_cast<const void*>(&visc_rows_visit_kernel<bf16, 2>),
                             reinterpret_cast<const void*>(&visc_rows_visit_kernel<bf16, 4>),
                             reinterpret_cast<const void*>(&visc_rows_visit_kernel<bf16, 8>)};
    for (const void* k : kernels)
        if (hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, most)) return e;
    return hipSuccess;
}

size_t visc_rows_bytes(int64_t n, int64_t nc) {
    const size_t np = (size_t(n) + 63) & ~size_t(63);
    // coef, idx, pos, b, r, child, each rounded up to an allocation unit
    return np * (4 * sizeof(float4) + 2 * sizeof(uint4) + 3 * 4) + 256 + size_t(nc) * sizeof(uint4) + 6 * 256;
}

hipError_t launch_visc_rows_build(const ViscLevelView& F, const ViscLevelView& Cl, const ViscRowsView& R,
                                  const int32_t* base, const int32_t* cpos, float* fmap, float* cmap, hipStream_t s) {
    if (R.n <= 0 || R.nc <= 0 || F.nleaf_dof <= 0 || Cl.nleaf_dof <= 0 || F.chan_off[3] <= 0 || !F.parent || !Cl.child)
        return hipErrorInvalidValue;
    const size_t nzero = size_t(Cl.nleaf_dof) * 3 * 512;
    rows_zero_kernel<<<unsigned((nzero + 255) / 256), 256, 0, s>>>(nzero, cmap);
    rows_coarse_map_kernel<<<unsigned((R.nc + 255) / 256), 256, 0, s>>>(R.nc, cpos, cmap);
    rows_number_kernel<<<unsigned(F.nleaf_dof * 3), 64, 0, s>>>(F.mask, base, fmap, R.pos);
    rows_fill_kernel<<<unsigned(F.chan_off[3]), 64, 0, s>>>(F, R, fmap, cmap);
    rows_child_kernel<<<unsigned((R.nc + 255) / 256), 256, 0, s>>>(Cl, R, cpos, fmap);
    return hipGetLastError();
}

hipError_t launch_visc_rows_visit(const ViscRowsView* views, const ViscCoarsestView* cviews, int count, int max_n,
                                  int max_nc, const float* b, float* x, bool precon, int nvisits, hipStream_t s) {
    return visit<float>(views, cviews, count, max_n, max_nc, b, x, precon, nvisits, s);
}
hipError_t launch_visc_rows_visit(const ViscRowsView* views, const ViscCoarsestView* cviews, int count, int max_n,
                                  int max_nc, const bf16* b, bf16* x, bool precon, int nvisits, hipStream_t s) {
    return visit<bf16>(views, cviews, count, max_n, max_nc, b, x, precon, nvisits, s);
}

}  // namespace uaamg
