// One FP64 sample of a gridded velocity field, which the advection and the
// adjoint's forward share; each has an RK4 step of its own around it, in the
// same operation order and so with the same bits.
//
// Operation order (mirrored operation by operation in oracle/lm_oracle.c):
//   fx  = (x - x0) * inv_dx,          i = trunc(fx) clamped to nx-2, xi  = fx - i
//   fy  = (y - y0) * inv_dy,          j = trunc(fy) clamped to ny-2, eta = fy - j
//   u_b = fma(xi, u10 - u00, u00),   u_t = fma(xi, u11 - u01, u01)
//   u   = fma(eta, u_t - u_b, u_b)   (same for v)
//   u_deg = (u * (1/111120)) / cos_deg(y),   v_deg = v * (1/111120)
//   x1 = fma(u1, dt/2, x) ... x3 = fma(u3, dt, x)
//   x += fma(2, u2 + u3, u1 + u4) * (dt/6) as fma(., dt/6, x)
//
// These loops are bound by VALU issue (two thirds of it and more), so the
// forms below are the ones with the fewest vector instructions: no branch
// between a step's stages, one comparison for both ends of an axis, offsets to
// uniform row pointers, a division without its scaling steps, polynomial
// coefficients in scalar registers: 232 vector instructions for a step of the
// FP64 advection, where the straightforward forms take 297.  100 steps of
// 490,000 particles with the random walk went from 803 to 665 us, 24 float32
// steps of 4,000,000 from 721 to 637.
#pragma once

#include "lm_common.h"

namespace lm {

// cos_deg's coefficients in constant memory, from where they are loaded into
// scalar registers, which a fused multiply-add reads as an operand.  As
// literals each of the 11 needs a vector move into the accumulator first.
struct CosCoefs {
    double c[12];
};

#define LM_DEFINE_COS_COEFS(name)                                  \
    __constant__ double name[12] = {LM_COS_COEFS};                 \
    __device__ __forceinline__ CosCoefs load_##name() {            \
        CosCoefs k;                                                \
        _Pragma("unroll") for (int q = 0; q < 12; ++q) k.c[q] = name[q]; \
        return k;                                                  \
    }

__device__ __forceinline__ double cos_deg_from(const CosCoefs& K, double lat_deg) {
    const double t = lat_deg * LM_DEG2RAD;
    return lm_horner<12>(K.c, t * t);
}

// n / d by Newton-Raphson: the hardware's reciprocal, two steps, the quotient
// and one correction by its residual, whose last fma rounds as the IEEE division
// does (Markstein).  Without that division's scaling, which keeps the reciprocal,
// the quotient and the residual in range: here d is a cosine and n a velocity in
// degrees per second.  Equal to the IEEE quotient while |n| is zero or at least
// 2^-960 and the quotient is finite; smaller numerators, whose residual
// underflows, may be off by the last bit, and a finite n over so small a d that
// the quotient overflows gives NaN instead of infinity (as a position, outside
// every grid like it).  Zeros, infinities and NaN come from the fix-up, as in the
// division.
__device__ __forceinline__ double divide_near_one(double n, double d) {
    double r = __builtin_amdgcn_rcp(d);
    r = fma(r, fma(-d, r, 1.0), r);
    r = fma(r, fma(-d, r, 1.0), r);
    const double q = n * r;
    return __builtin_amdgcn_div_fixup(fma(fma(-d, q, n), r, q), d, n);
}

// trunc(v) saturated to int32, NaN to 0 (a C++ conversion is undefined there).
__device__ __forceinline__ int trunc_i32(double v) {
    int i;
    asm("v_cvt_i32_f64 %0, %1" : "=v"(i) : "v"(v));
    return i;
}

// Cell and fractional position along one axis of n nodes: index t =
// (v - v0) * inv (a zero product made +0 by the fma).  A position outside
// gets some cell inside and a fraction outside [0, 1].  Returns the wavefront's
// lanes inside: the fraction's bits, compared as an unsigned integer, are above
// 1.0's for every negative value, every one above 1 and every NaN.  (As lane
// masks, because the compiler otherwise packs a step's eight conditions into
// the bits of vector registers.)
using lanes_t = unsigned long long;

__device__ __forceinline__ lanes_t locate_axis(double v, double v0, double inv, int n, uint32_t* cell, double* frac) {
    const double t = fma(v - v0, inv, 0.0);
    const uint32_t i = min((uint32_t)trunc_i32(t), (uint32_t)(n - 2));
    const double f = t - (double)(int)i;
    *cell = i;
    *frac = f;
    return __builtin_amdgcn_ballot_w64((uint64_t)__double_as_longlong(f) <= 0x3ff0000000000000ull);
}

// Byte offset of node (j, i), nodes of SIZE bytes: in 32 bits, added to a
// uniform pointer by the load itself, while a field has less than 4 GB and
// fewer than 2^24 nodes along an axis (fits_offset32); BIG: in 64 bits.
inline bool fits_offset32(const lm_grid& g, int size) {
    return g.nx < (1 << 24) && g.ny < (1 << 24) && (int64_t)g.nx * g.ny * size < ((int64_t)1 << 32);
}

template <int SIZE, bool BIG>
__device__ __forceinline__ auto node_offset(const lm_grid& g, uint32_t i, uint32_t j) {
    if constexpr (BIG) return ((uint64_t)j * (uint64_t)g.nx + i) * SIZE;
    else return (__umul24(j, (uint32_t)g.nx) + i) * (uint32_t)SIZE;
}

// The sample at (x, y) of the field f and the lanes inside the grid; outside
// (or NaN) the velocity means nothing.
template <bool BIG>
__device__ __forceinline__ lanes_t sample_uv(const double* __restrict__ f, const lm_grid& g, const CosCoefs& K, double x,
                                          double y, double* ud, double* vd, uint32_t* ci, uint32_t* cj) {
    double xi, eta;
    const lanes_t in_x = locate_axis(x, g.x0, g.inv_dx, g.nx, ci, &xi);
    const lanes_t in_y = locate_axis(y, g.y0, g.inv_dy, g.ny, cj, &eta);
    const auto off = node_offset<16, BIG>(g, *ci, *cj);
    const char* row = reinterpret_cast<const char*>(f);  // uniform, as the next one
    const double2* r0 = reinterpret_cast<const double2*>(row + off);
    const double2* r1 = reinterpret_cast<const double2*>(row + 16 * (int64_t)g.nx + off);
    const double2 a = r0[0], b = r0[1], c = r1[0], d = r1[1];
    const double ub = fma(xi, b.x - a.x, a.x);
    const double ut = fma(xi, d.x - c.x, c.x);
    const double u = fma(eta, ut - ub, ub);
    const double vb = fma(xi, b.y - a.y, a.y);
    const double vt = fma(xi, d.y - c.y, c.y);
    const double v = fma(eta, vt - vb, vb);
    *ud = divide_near_one(u * LM_INV_M_PER_DEG, cos_deg_from(K, y));
    *vd = v * LM_INV_M_PER_DEG;
    return in_x & in_y;
}

}  // namespace lm
