// Coarsest-level solve as a block-wide device routine: Eigen::ConjugateGradient
// with DiagonalPreconditioner, zero initial guess, maxIterations = 10,
// tolerance = float epsilon, restated (constructCoarsestLevelExactSolver,
// simd_vdb_poisson.cpp:2114-2126; Eigen ConjugateGradient.h conjugate_gradient()).
//
// The first kRowThreads threads of the block keep up to kPer DOFs' matrix rows
// and x, r, z, p, q = A p in registers; only z is shared through LDS for the
// neighbour reads. An absent neighbour reads slot kMaxCoarsestDof of the
// shared vector, which holds zero, so the six reads of a row are
// unconditional.
//
// An iteration is a serial chain on one CU (neighbour reads, sums over the
// block, divisions, barriers), so the form with one sum over the block per
// iteration is used (Chronopoulos and Gear, "s-step iterative methods for
// symmetric linear systems", J. Comput. Appl. Math. 25, 1989, with s = 1):
// with w = A z, one reduction gives ||r||^2, g = <r, z> and d = <z, w>; then
// beta = g / g_old, <p, A p> = d - beta^2 <p, A p>_old, alpha = g / <p, A p>,
// p = z + beta p and q = A p = w + beta q. The same vectors as Eigen's loop,
// rounded differently, for small right-hand sides too (cg_scale.h). Eigen's
// stopping test on ||r||^2 after an update is made by the next iteration's
// sums, before anything changes. With the sum of
// <p, A p> kept apart (two reductions per iteration) a solve of 1697 rows took
// 13.5 us, with one 11.9; the rows packed to 48 bytes.
#pragma once

#include <cfloat>

#include "cg_scale.h"
#include "poisson_kernels.h"
#include "wave_reduce.h"

namespace uaamg {
namespace dev {

struct CgShared {
    float4 red[2][1024 / 64];   // wavefronts of the largest row-thread count
    float sp[kMaxCoarsestDof + 1];   // the last slot stays zero
};

// Sums (a, b, c) over the row threads with one barrier; red alternates
// between two buffers, so the next call needs no barrier before it writes.
// Wavefronts without rows take part in the barrier and read the sums.
template <int kRowThreads>
__device__ __forceinline__ float3 cg_sum3(float a, float b, float c, CgShared& sh, int& parity) {
    const int w = threadIdx.x >> 6;
    if (w < kRowThreads / 64) {
        a = wave_sum_dpp(a);
        b = wave_sum_dpp(b);
        c = wave_sum_dpp(c);
        if ((threadIdx.x & 63) == 0) sh.red[parity][w] = make_float4(a, b, c, 0.f);
    }
    __syncthreads();
    float3 t = make_float3(0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < kRowThreads / 64; ++i) {
        const float4 v = sh.red[parity][i];
        t.x += v.x;
        t.y += v.y;
        t.z += v.z;
    }
    parity ^= 1;
    return t;
}

// Solves the coarsest system for right-hand side B (bricks) into X (bricks,
// DOF positions only); C.ndof <= kMaxDof (thread t owns rows t +
// j*kRowThreads, so a smaller kMaxDof only drops row slots that would be
// empty: the results do not depend on it, nor on the threads beyond
// kRowThreads). Every thread of the block must call it. kKeep: the solution,
// as X would hold it, also goes to sh.sp[d] (d < ndof; the zero slot stays
// zero), and X may be null; the caller's next barrier publishes it.
template <int kRowThreads, class V = float, int kMaxDof = kMaxCoarsestDof, bool kKeep = false>
__device__ void coarsest_cg_block(const CoarsestView& C, const V* B, V* X, CgShared& sh) {
    static_assert(kMaxDof <= kMaxCoarsestDof && kMaxDof % kRowThreads == 0, "row slots");
    constexpr int kPer = kMaxDof / kRowThreads;
    constexpr int kZero = kMaxCoarsestDof;
    int parity = 0;
    const int tid = threadIdx.x;
    const int n = tid < kRowThreads ? C.ndof : 0;   // rows d < n: none beyond the row threads
    int nb[kPer][6];
    float cf[kPer][8], x[kPer], r[kPer], z[kPer], p[kPer], q[kPer];
    if (tid == 0) sh.sp[kZero] = 0.f;   // published with z
    int4 row[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int d = tid + j * kRowThreads;
        row[j] = make_int4(0, 0, 0, 0);
        float4 c0 = make_float4(0.f, 0.f, 0.f, 0.f), c1 = c0;
        if (d < n) {
            row[j] = reinterpret_cast<const int4*>(C.row)[d];
            c0 = reinterpret_cast<const float4*>(C.coef)[size_t(d) * 2];
            c1 = reinterpret_cast<const float4*>(C.coef)[size_t(d) * 2 + 1];
        }
        cf[j][0] = c0.x; cf[j][1] = c0.y; cf[j][2] = c0.z; cf[j][3] = c0.w;
        cf[j][4] = c1.x; cf[j][5] = c1.y; cf[j][6] = c1.z; cf[j][7] = c1.w;
    }
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int d = tid + j * kRowThreads;
        x[j] = r[j] = z[j] = p[j] = q[j] = 0.f;
        if (d < n) r[j] = float(B[row[j].w]);
        nb[j][0] = row[j].x & 0xffff; nb[j][1] = int(uint32_t(row[j].x) >> 16);
        nb[j][2] = row[j].y & 0xffff; nb[j][3] = int(uint32_t(row[j].y) >> 16);
        nb[j][4] = row[j].z & 0xffff; nb[j][5] = int(uint32_t(row[j].z) >> 16);
    }
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int d = tid + j * kRowThreads;
        if (d < n) {
            z[j] = cf[j][7] * r[j];
            sh.sp[d] = z[j];
        }
    }
    __syncthreads();
    float threshold = 0.f, g_inv = 0.f, sigma = 0.f;
    for (int it = 0; it < C.max_iters; ++it) {
        float w[kPer];
        float rr = 0.f, rz = 0.f, zw = 0.f;
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int d = tid + j * kRowThreads;
            w[j] = 0.f;
            if (d < n) {
                float v[6];
#pragma unroll
                for (int k = 0; k < 6; ++k) v[k] = sh.sp[nb[j][k]];
                const float s1 = fmaf(v[1], cf[j][2], v[0] * cf[j][1]);
                const float s2 = fmaf(v[3], cf[j][4], v[2] * cf[j][3]);
                const float s3 = fmaf(v[5], cf[j][6], v[4] * cf[j][5]);
                w[j] = fmaf(z[j], cf[j][0], (s1 + s2) + s3);
                rr = fmaf(r[j], r[j], rr);
                rz = fmaf(r[j], z[j], rz);
                zw = fmaf(z[j], w[j], zw);
            }
        }
        // the barrier also orders this step's reads of z before the writes below
        float3 s = cg_sum3<kRowThreads>(rr, rz, zw, sh, parity);
        float beta = 0.f;
        if (it == 0) {
            threshold = fmaxf(C.tol * C.tol * s.x, FLT_MIN);
            if (s.x == 0.f || s.x < threshold) break;
            if (cg_needs_scale(s.y)) {   // the same step with c D^-1
                const float c = cg_scale(s.y);
                rz = zw = 0.f;
#pragma unroll
                for (int j = 0; j < kPer; ++j) {
                    cf[j][7] *= c;
                    z[j] *= c;
                    w[j] *= c;
                    rz = fmaf(r[j], z[j], rz);
                    zw = fmaf(z[j], w[j], zw);
                }
                s = cg_sum3<kRowThreads>(0.f, rz, zw, sh, parity);
            }
            sigma = s.z;
        } else {
            if (s.x < threshold) break;
            beta = s.y * g_inv;
            sigma = fmaf(-(beta * beta), sigma, s.z);
        }
        const float alpha = s.y / sigma;
        g_inv = 1.f / s.y;
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            p[j] = fmaf(beta, p[j], z[j]);
            q[j] = fmaf(beta, q[j], w[j]);
            x[j] = fmaf(alpha, p[j], x[j]);
            r[j] = fmaf(-alpha, q[j], r[j]);
            z[j] = cf[j][7] * r[j];
        }
        if (it + 1 < C.max_iters) {
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                const int d = tid + j * kRowThreads;
                if (d < n) sh.sp[d] = z[j];
            }
            __syncthreads();
        }
    }
    // every thread has passed the last barrier that follows a read of sh.sp
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int d = tid + j * kRowThreads;
        if (d < n) {
            const V xv = V(x[j]);
            if constexpr (kKeep) {
                sh.sp[d] = float(xv);
                if (X) X[row[j].w] = xv;
            } else {
                X[row[j].w] = xv;
            }
        }
    }
}

}  // namespace dev
}  // namespace uaamg
