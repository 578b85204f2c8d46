// The power of two that the coarsest CGs (coarsest_device.h,
// visc_coarsest_device.h) multiply their preconditioner D^-1 by.
//
// Their loop runs while ||r||^2 is at least FLT_EPSILON^2 ||b||^2 and FLT_MIN,
// but it divides by g = <r, D^-1 r>, smaller than ||r||^2 by the diagonal (1e3
// to 1e7 on fine grids): with a small b, g loses its digits and 1 / g overflows
// while the loop still runs. Deep in the W-cycle of a nearly converged solve b
// is that small. CG does not depend on a factor of its preconditioner: with
// c D^-1 in the place of D^-1, g becomes c g, <p, A p> c^2 <p, A p> and x stays.
// A power of two changes no digit, so a solve whose sums are ordinary, as
// nearly all are, is the same without one, and the others keep its accuracy.
// Where none is needed it costs one comparison a solve (whole solves at 32^3 to
// 512^3: 0.995 to 1.004 of the time without it); multiplying r and b instead,
// which the loop then has to hand back, cost 4%.
#pragma once

#include <hip/hip_runtime.h>

namespace uaamg {
namespace dev {

// Whether g of the first iteration is too small or large for the loop, in
// which g shrinks by FLT_EPSILON^2 (2^46) and somewhat more with an uneven D.
__device__ __forceinline__ bool cg_needs_scale(float g) { return !(g >= 0x1p-56f && g <= 0x1p100f); }

// The factor: g = 2^e becomes 2^(20 + e/2) and <p, A p>, about g, 2^40.
__device__ __forceinline__ float cg_scale(float g) {
    const int e = ((__float_as_int(g) >> 23) & 255) - 127;
    return __int_as_float((127 + 20 - e / 2) << 23);
}

}  // namespace dev
}  // namespace uaamg
