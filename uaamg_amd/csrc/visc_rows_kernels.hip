// The viscosity level above the coarsest as rows (visc_rows.h): the build of
// the rows from the level's bricks, and the visits.
#include "visc_rows.h"

#include "visc_coarsest_device.h"
#include "viscosity_device.h"

namespace uaamg {
namespace {

using namespace dev;

constexpr int kStepLast = kViscStepLast;
constexpr int kMaxSteps = kViscMaxSteps;

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

// The views come from memory, so their pointers are generic to the compiler:
// its flat loads would count as LDS accesses too and each barrier would wait
// for them. Loads and stores here name the global address space.
typedef float vf4 __attribute__((ext_vector_type(4)));
typedef uint32_t vu4 __attribute__((ext_vector_type(4)));
#define UAAMG_GLOBAL __attribute__((address_space(1)))
template <class T>
__device__ __forceinline__ T gload(const void* base, uint32_t byte) {
    return *reinterpret_cast<const UAAMG_GLOBAL T*>((const UAAMG_GLOBAL char*)base + byte);
}
template <class T>
__device__ __forceinline__ void gstore(void* base, uint32_t byte, T v) {
    *reinterpret_cast<UAAMG_GLOBAL T*>((UAAMG_GLOBAL char*)base + byte) = v;
}

// one row's operands
struct Row {
    vf4 c[4];
    vu4 i[2];
    float b;
};

__device__ __forceinline__ Row load_row(const ViscRowsView& R, int row) {
    Row q;
    const uint32_t o16 = uint32_t(row) * 16u;
#pragma unroll
    for (int k = 0; k < 4; ++k) q.c[k] = gload<vf4>(R.coef + size_t(k) * size_t(R.np), o16);
#pragma unroll
    for (int k = 0; k < 2; ++k) q.i[k] = gload<vu4>(R.idx + size_t(k) * size_t(R.np), o16);
    q.b = gload<float>(R.b, uint32_t(row) * 4u);
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

// Rows in flight per thread: a row's operands do not depend on x, so they are
// loaded this many steps ahead, across the barriers between passes too. (At
// 6018 rows one, two and three ahead take the same time: what is left of a
// pass is the CU's own work, 100 KB of rows, 14 LDS reads and about 90 vector
// instructions a row.)
constexpr int kRowsAhead = 2;

// `sweeps` Gauss-Seidel sweeps (six colour passes each) over the steps of one
// direction (ViscRowsView::steps, in LDS), then, with RESIDUAL, the residual
// of every row into R.r; x in LDS.
template <class V, bool RESIDUAL>
__device__ __forceinline__ void run_passes(const ViscRowsView& R, const int2* steps, int nsteps, float* xs,
                                           int sweeps) {
    const int tid = threadIdx.x;
    const int gs = sweeps * nsteps, total = gs + (RESIDUAL ? nsteps : 0);
    Row buf[kRowsAhead];
    int2 st[kRowsAhead];
    int ahead = 0;   // the step to fetch next, modulo nsteps
    auto fetch = [&](int u) {
        st[u] = steps[ahead];
        ahead = ahead + 1 < nsteps ? ahead + 1 : 0;
        const int row = st[u].x + tid;
        buf[u] = load_row(R, row < R.n ? row : 0);
    };
#pragma unroll
    for (int u = 0; u < kRowsAhead; ++u) fetch(u);
#pragma unroll 1
    for (int i = 0; i < total; i += kRowsAhead) {
#pragma unroll
        for (int u = 0; u < kRowsAhead; ++u) {
            if (i + u >= total) break;
            const int row = st[u].x + tid, end = st[u].y & (kStepLast - 1);
            const bool last = __builtin_amdgcn_readfirstlane(st[u].y) >= kStepLast;
            if (row < end) {
                const float s = row_sum(buf[u], xs);
                if (!RESIDUAL || i + u < gs) {
                    float t = buf[u].b - s;
                    t = t * buf[u].c[3].z;
                    xs[row] = stored<V>(fmaf(xs[row], 0.0f, t));
                } else {
                    gstore<float>(R.r, uint32_t(row) * 4u, stored<V>(buf[u].b - fmaf(xs[row], buf[u].c[3].w, s)));
                }
            }
            fetch(u);
            if (last) __syncthreads();
        }
    }
}

// The visits (see visc_rows.h). Bounded by one CU's rates: 96 + 4 bytes per
// row, five times over all rows per visit. Two visits of a 6018-row level with
// the coarsest solves (934 rows) take 95 us; as launches a visit took 155 us.
template <class V, int kPer, int kT>
__device__ __forceinline__ void rows_visit(const ViscRowsView& R, const ViscCoarsestView& C, const V* B, V* X,
                                           bool precon, int nvisits) {
    extern __shared__ float sm[];
    __shared__ ViscCgShared cg;
    float* xs = sm;                // [n + 1], the last zero
    float* sz = sm + R.n + 1;      // [nc + 1], the last zero
    const int tid = threadIdx.x;
    __shared__ int2 steps[2 * kMaxSteps];
    const int nsteps = R.nsteps;
    for (int i = tid; i < 2 * nsteps; i += kT) steps[i] = make_int2(gload<int>(R.steps, uint32_t(i) * 8u), gload<int>(R.steps, uint32_t(i) * 8u + 4u));
    if (tid == 0) {
        xs[R.n] = 0.f;
        gstore<float>(R.r, uint32_t(R.n) * 4u, 0.f);
    }
    for (int row = tid; row < R.n; row += kT) {
        const int p = gload<int>(R.pos, uint32_t(row) * 4u);
        gstore<float>(R.b, uint32_t(row) * 4u, ld1v(B + p));
        xs[row] = precon ? 0.f : ld1v(X + p);
    }
    __syncthreads();
#pragma unroll 1
    for (int v = 0; v < nvisits; ++v) {
        run_passes<V, true>(R, steps, nsteps, xs, 2);
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
                const vu4 w = gload<vu4>(R.child, uint32_t(d) * 16u);
                float sum = 0.f, f[8];
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    f[k] = gload<float>(R.r, 4u * ((k & 1) ? (w[k >> 1] >> 16) : (w[k >> 1] & 0xffffu)));
#pragma unroll
                for (int k = 0; k < 8; ++k) sum += f[k];
                return stored<V>(sum * 0.125f * 0.5f * 2.0f);
            },
            [&](int d, float x) { sz[d] = stored<V>(x); });
        __syncthreads();
        // prolongation
        for (int row = tid; row < R.n; row += kT)
            xs[row] = stored<V>(xs[row] + sz[gload<uint32_t>(R.idx + size_t(R.np), uint32_t(row) * 16u + 12u) & 0xffffu]);
        __syncthreads();
        run_passes<V, false>(R, steps + nsteps, nsteps, xs, 2);
    }
    for (int row = tid; row < R.n; row += kT) st1v(X + gload<int>(R.pos, uint32_t(row) * 4u), xs[row]);
}

// one workgroup
template <class V, int kPer, int kT>
__global__ __launch_bounds__(kT) void visc_rows_visit_kernel(const ViscRowsView* view, const ViscCoarsestView* cview,
                                                             const V* B, V* X, int precon, int nvisits) {
    const ViscRowsView R = *view;
    const ViscCoarsestView C = *cview;
    rows_visit<V, kPer, kT>(R, C, B, X, precon != 0, nvisits);
}

template <class V>
hipError_t visit(const ViscRowsView* view, const ViscCoarsestView* cview, int n, int nc, const V* b, V* x, bool precon,
                 int nvisits, hipStream_t s) {
    if (n <= 0 || n > kViscRowsMax || nc <= 0 || nc > kViscMaxCoarsest || nvisits < 1) return hipErrorInvalidValue;
    const size_t lds = (size_t(n) + size_t(nc) + 2) * sizeof(float);
    const int p = precon ? 1 : 0;
    // (the steps of the view are cut for the same thread count)
    static_assert(2 * kVCgThreads == kViscRowsWideNc, "the wide form's coarsest size");
    if (visc_rows_step(nc) == 1024)
        visc_rows_visit_kernel<V, 2, 1024><<<1, 1024, lds, s>>>(view, cview, b, x, p, nvisits);
    else if (nc <= 4 * kVCgThreads)
        visc_rows_visit_kernel<V, 4, 512><<<1, 512, lds, s>>>(view, cview, b, x, p, nvisits);
    else
        visc_rows_visit_kernel<V, 8, 512><<<1, 512, lds, s>>>(view, cview, b, x, p, nvisits);
    return hipGetLastError();
}

}  // namespace

hipError_t visc_rows_init() {
    const int most = int((kViscRowsMax + kViscMaxCoarsest + 2) * sizeof(float));
    const void* kernels[] = {reinterpret_cast<const void*>(&visc_rows_visit_kernel<float, 2, 1024>),
                             reinterpret_cast<const void*>(&visc_rows_visit_kernel<float, 4, 512>),
                             reinterpret_cast<const void*>(&visc_rows_visit_kernel<float, 8, 512>),
                             reinterpret_cast<const void*>(&visc_rows_visit_kernel<bf16, 2, 1024>),
                             reinterpret_cast<const void*>(&visc_rows_visit_kernel<bf16, 4, 512>),
                             reinterpret_cast<const void*>(&visc_rows_visit_kernel<bf16, 8, 512>)};
    for (const void* k : kernels)
        if (hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, most)) return e;
    return hipSuccess;
}

size_t visc_rows_bytes(int64_t n, int64_t nc) {
    const size_t np = (size_t(n) + 63) & ~size_t(63);
    // coef, idx, pos, b, r, child, each rounded up to an allocation unit
    return np * (4 * sizeof(float4) + 2 * sizeof(uint4) + 3 * 4) + 256 + size_t(nc) * sizeof(uint4) + 2 * kMaxSteps * sizeof(int2) +
           7 * 256;
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

hipError_t launch_visc_rows_visit(const ViscRowsView* view, const ViscCoarsestView* cview, int n, int nc,
                                  const float* b, float* x, bool precon, int nvisits, hipStream_t s) {
    return visit<float>(view, cview, n, nc, b, x, precon, nvisits, s);
}
hipError_t launch_visc_rows_visit(const ViscRowsView* view, const ViscCoarsestView* cview, int n, int nc,
                                  const bf16* b, bf16* x, bool precon, int nvisits, hipStream_t s) {
    return visit<bf16>(view, cview, n, nc, b, x, precon, nvisits, s);
}

}  // namespace uaamg
