// Coarsest-level viscosity solve as a block-wide device routine:
// Eigen::ConjugateGradient<RowMajor, Upper|Lower> with the diagonal
// preconditioner, zero guess, 10 iterations, tolerance = float epsilon
// (construct_exact_solver / solve_exact, simd_viscosity3d.cpp:2598-2657).
//
// Each thread keeps up to kPer rows in registers (15 values, 15 column
// offsets as 16-bit pairs) and only z is shared, so an iteration touches LDS
// alone; the form with one sum over the block per iteration is the one of
// coarsest_device.h (Chronopoulos and Gear), for small right-hand sides with a
// factor of the preconditioner (cg_scale.h). A row's padding multiplies the
// shared vector's last slot, which holds zero. With the rows streamed from
// memory in every iteration a system of more than 1024 rows took 52 us.
#pragma once

#include <cfloat>

#include "cg_scale.h"
#include "viscosity_kernels.h"
#include "wave_reduce.h"

namespace uaamg {
namespace dev {

constexpr int kVCgThreads = 512;

struct ViscCgShared {
    float4 red[2][kVCgThreads / 64];
};

// Sums (a, b, c) over the row threads with one barrier (cg_sum3).
__device__ __forceinline__ float3 visc_cg_sum3(float a, float b, float c, ViscCgShared& sh, int& par) {
    const int w = threadIdx.x >> 6;
    if (w < kVCgThreads / 64) {
        a = wave_sum_dpp(a);
        b = wave_sum_dpp(b);
        c = wave_sum_dpp(c);
        if ((threadIdx.x & 63) == 0) sh.red[par][w] = make_float4(a, b, c, 0.f);
    }
    __syncthreads();
    float3 s = make_float3(0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < kVCgThreads / 64; ++i) {
        const float4 v = sh.red[par][i];
        s.x += v.x;
        s.y += v.y;
        s.z += v.z;
    }
    par ^= 1;
    return s;
}

// Solves the system for the right-hand side ld(d) and hands the solution to
// st(d, x); sz has room for C.n + 1 floats. Row d belongs to thread d %
// kVCgThreads, C.n <= kPer * kVCgThreads (a larger kPer only adds empty rows).
// Every thread of the block, of kVCgThreads threads or more, must call it (the
// threads beyond only take part in the barriers); on return no thread reads sz
// any more.
template <int kPer, class Load, class Store>
__device__ __forceinline__ void visc_cg_block(const ViscCoarsestView& C, float* sz, ViscCgShared& sh, const Load& ld,
                                              const Store& st) {
    constexpr int kPairs = (kViscMaxRow + 1) / 2;
    const int tid = threadIdx.x, size = C.n;
    const int n = tid < kVCgThreads ? size : 0;   // rows d < n
    float ev[kPer][kViscMaxRow], inv[kPer], x[kPer], r[kPer], p[kPer], q[kPer];
    uint32_t ep[kPer][kPairs];
    int par = 0;
    if (tid == 0) sz[size] = 0.f;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int d = tid + j * kVCgThreads;
        x[j] = r[j] = p[j] = q[j] = inv[j] = 0.f;
#pragma unroll
        for (int k = 0; k < kViscMaxRow; ++k) ev[j][k] = 0.f;
#pragma unroll
        for (int k = 0; k < kPairs; ++k) ep[j][k] = 0;
        if (d < n) {
#pragma unroll
            for (int k = 0; k < kViscMaxRow; ++k) ev[j][k] = C.eval[size_t(k) * size_t(size) + size_t(d)];
#pragma unroll
            for (int k = 0; k < kPairs; ++k) ep[j][k] = C.epair[size_t(k) * size_t(size) + size_t(d)];
            inv[j] = C.invdiag[d];
            r[j] = ld(d);
            sz[d] = inv[j] * r[j];
        }
    }
    __syncthreads();
    float threshold = 0.f, g_inv = 0.f, sigma = 0.f;
    for (int it = 0; it < C.max_iters; ++it) {
        if constexpr (kPer > 4) {
            // eight rows fill the register file: the column offsets stay packed
            // (the empty asm keeps the compiler from unpacking them all before
            // the loop)
#pragma unroll
            for (int j = 0; j < kPer; ++j)
#pragma unroll
                for (int k = 0; k < kPairs; ++k) asm volatile("" : "+v"(ep[j][k]));
        }
        float w[kPer], rr = 0.f, rz = 0.f, zw = 0.f;
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int d = tid + j * kVCgThreads;
            w[j] = 0.f;
            if (d < n) {
                float t = 0.f;
#pragma unroll
                for (int k = 0; k < kViscMaxRow; ++k) {
                    const uint32_t e = ep[j][k >> 1];
                    const uint32_t at = (k & 1) ? (e >> 16) : (e & 0xffffu);
                    t = fmaf(ev[j][k], *reinterpret_cast<const float*>(reinterpret_cast<const char*>(sz) + at), t);
                }
                const float z = inv[j] * r[j];
                w[j] = t;
                rr = fmaf(r[j], r[j], rr);
                rz = fmaf(r[j], z, rz);
                zw = fmaf(z, t, zw);
            }
        }
        // the barrier also orders this step's reads of z before the writes below
        float3 s = visc_cg_sum3(rr, rz, zw, sh, par);
        float beta = 0.f;
        if (it == 0) {
            threshold = fmaxf(C.tol * C.tol * s.x, FLT_MIN);
            if (s.x == 0.f || s.x < threshold) break;
            if (cg_needs_scale(s.y)) {   // the same step with c D^-1
                const float c = cg_scale(s.y);
                rz = zw = 0.f;
#pragma unroll
                for (int j = 0; j < kPer; ++j) {
                    inv[j] *= c;
                    w[j] *= c;
                    const float z = inv[j] * r[j];
                    rz = fmaf(r[j], z, rz);
                    zw = fmaf(z, w[j], zw);
                }
                s = visc_cg_sum3(0.f, rz, zw, sh, par);
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
            p[j] = fmaf(beta, p[j], inv[j] * r[j]);
            q[j] = fmaf(beta, q[j], w[j]);
            x[j] = fmaf(alpha, p[j], x[j]);
            r[j] = fmaf(-alpha, q[j], r[j]);
        }
        if (it + 1 < C.max_iters) {
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                const int d = tid + j * kVCgThreads;
                if (d < n) sz[d] = inv[j] * r[j];
            }
            __syncthreads();
        }
    }
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int d = tid + j * kVCgThreads;
        if (d < n) st(d, x[j]);
    }
}

}  // namespace dev
}  // namespace uaamg
