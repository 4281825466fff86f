// Device helpers shared by the FCT, moment and field kernels.  Each follows
// the reference expression for expression (same operands, same association)
// because the FP64 path is bit-compared with the CPU oracle; the library is
// compiled with -ffp-contract=off so no multiply-add is fused.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "vx_consts.h"

namespace vxd {

// Rectangle.hpp:111-126
__device__ __forceinline__ double valmax(double a, double b) { return a > b ? a : b; }
__device__ __forceinline__ double valmin(double a, double b) { return a < b ? a : b; }
// std::min / std::max as used by the limiter-C sync (Rectangle.cpp:1646-1829)
__device__ __forceinline__ double stdmin(double a, double b) { return (b < a) ? b : a; }

// XCD-aware workgroup order: the dispatcher hands workgroup w of a launch to
// XCD w mod 8, so map w to a tile index that gives each XCD one contiguous
// run of tiles.  Neighbouring tiles (which read each other's halo rows and
// columns) then run on the same XCD and share those cache lines in its L2.
// A bijection of [0, nwg): XCD x takes q + (x < rem) workgroups and the run
// [x q + min(x, rem), ...) of that length.
__device__ __forceinline__ int xcd_order(int w, int nwg) {
    const int xcd = w & 7, q = nwg >> 3, rem = nwg & 7;
    return xcd * q + min(xcd, rem) + (w >> 3);
}

// The same in chunks of K consecutive tiles, dealt round-robin to the XCDs
// (chunk c to XCD c mod 8): neighbours within a chunk share one L2, and
// launches whose tiles differ in cost (several patches of different strip
// shapes) stay balanced over the XCDs.  Workgroups past the last whole round
// of 8 K keep their own index.  A bijection of [0, nwg).
template <int K>
__device__ __forceinline__ int xcd_chunk_order(int w, int nwg) {
    const int full = nwg - nwg % (8 * K);
    if (w >= full) return w;
    const int x = w & 7, k = w >> 3;
    return (x + 8 * (k / K)) * K + k % K;
}

// v_max_f64 / v_min_f64 as single instructions.  fmax/fmin compile to the
// same instruction, but first quiet possible signalling NaNs with a
// v_max_f64 x, x, x of every operand the compiler cannot prove canonical
// (loaded values, lane shifts, values carried around the row loop); the
// operands here are never NaN, so that step changes no bits and only costs
// issue slots.
__device__ __forceinline__ double hwmax(double a, double b) {
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ double hwmin(double a, double b) {
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// the larger, smaller of 0 and a
__device__ __forceinline__ double hwmax0(double a) {
    double r;
    asm("v_max_f64 %0, 0, %1" : "=v"(r) : "v"(a));
    return r;
}
__device__ __forceinline__ double hwmin0(double a) {
    double r;
    asm("v_min_f64 %0, 0, %1" : "=v"(r) : "v"(a));
    return r;
}

// Rectangle.hpp:86-88: lower p-face of cell j (pmin + dp * (j + p_pos))
__device__ __forceinline__ double momentum(double pmin, double dp, int j, int p_pos) {
    return pmin + dp * ((double)j + (double)p_pos);
}

// Rectangle::GetEfield(i) (Rectangle.cpp:1055-1067): mean of the finest-grid E
// over the rtb finest cells of patch column i.  EMFieldSolver::GetEfield
// (EMSolver.cpp:137-154) wraps each stencil index once, which equals the
// periodic index for finest indices in [-n_f, 2 n_f); callers check that the
// patch lies inside the finest grid, so rtb * (i + x_pos) + k stays there for
// the columns i in [-2, n_x + 2) the stage reads.
__device__ __forceinline__ double patch_E(const double *E, int n_f, int rtb, int x_pos, int i) {
    const int j = rtb * (i + x_pos);
    double t = 0.0;
    for (int k = 0; k < rtb; k++) {
        int m = j + k;
        m = m < 0 ? m + n_f : (m >= n_f ? m - n_f : m);
        t += E[m];
    }
    t *= (1.0 / (double)rtb);
    return t;
}

// sqrt(x) for x >= 1 (or NaN): the compiler's FP64 sequence without its
// scaling of arguments below 2^-767, so the same correctly rounded value; an
// infinite x (rsq 0) returns itself as there.  Measured on an MI355X: 86
// cycles per wave64 square root with the scaling, 70 without.
__device__ __forceinline__ double sqrt_ge1(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double s0 = x * y, h0 = 0.5 * y;
    const double r0 = __builtin_fma(-h0, s0, 0.5);
    const double s1 = __builtin_fma(s0, r0, s0), h1 = __builtin_fma(h0, r0, h0);
    const double s2 = __builtin_fma(__builtin_fma(-s1, s1, x), h1, s1);
    const double s3 = __builtin_fma(__builtin_fma(-s2, s2, x), h1, s2);
    return x == __builtin_inf() ? x : s3;
}

// Rectangle.hpp:181-183 with mc2inv = (m_inv*c_inv)*(m_inv*c_inv)
__device__ __forceinline__ double gamma_(double p, double a2, double mc2inv) {
    return sqrt_ge1(1.0 + ((p * p) + a2) * mc2inv);
}

// Rectangle.cpp:979-1030 (two-candidate WENO, upwind side takes the larger
// mapped weight); identical values to GetWenoEdgeValue (Rectangle.cpp:943-977).
__device__ __forceinline__ double weno(double f1, double f2, double f3, double f4, bool right) {
    double fL = (1.0 / 6) * (-f1 + 5 * f2 + 2 * f3);
    double fR = (1.0 / 6) * (2 * f2 + 5 * f3 - f4);
    double AL = f1 - 2 * f2 + f3;
    double BL = f3 - f1;
    double AR = f2 - 2 * f3 + f4;
    double BR = f4 - f2;
    double bL = 4.0 / 3 * (AL * AL) + 0.5 * AL * BL + 0.25 * (BL * BL);
    double bR = 4.0 / 3 * (AR * AR) - 0.5 * AR * BR + 0.25 * (BR * BR);
    const double mm = 1.0e-10;
    double oL = 0.5 / ((mm + bL) * (mm + bL));
    double oR = 0.5 / ((mm + bR) * (mm + bR));
    double wL = oL / (oL + oR);
    double wR = oR / (oL + oR);
    double wL0 = wL * (0.75 + wL * (wL - 0.5));
    double wR0 = wR * (0.75 + wR * (wR - 0.5));
    double s = wL0 + wR0;
    // right: the larger weight goes to fL; left: the smaller one does
    bool takeL = right ? (wL0 > wR0) : (wL0 < wR0);
    double w = (takeL ? wL0 : wR0) / s;
    double fwL = w;
    double fwR = 1 - w;
    return fwL * fL + fwR * fR;
}

// Division without the scaling and fix-up steps of the compiler's FP64
// sequence (v_div_scale, v_div_fmas, v_div_fixup): the same v_rcp_f64, Newton
// and remainder steps, so the same correctly rounded quotient wherever no
// intermediate leaves the normal range.  That holds for divisors in
// [2^-900, 2^900] and numerators that are 0 or in [2^-900, 2^900] with
// quotients in that range too (the remainder of a numerator n is a multiple of
// 2^-106 |n|).  Measured on an MI355X in independent streams: 50 cycles per
// wave64 division against 69 (v_div_scale_f64 alone takes 13, v_rcp_f64 18, an
// FMA 5), and one reciprocal serves several numerators.
__device__ __forceinline__ double rcp_refined(double d) {
    double r = __builtin_amdgcn_rcp(d);
    r = __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
    return __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
}
// n / d from r = rcp_refined(d)
__device__ __forceinline__ double div_refined(double n, double d, double r) {
    const double q = n * r;
    return __builtin_fma(__builtin_fma(-d, q, n), r, q);
}

// The parts of vxd::weno that belong to one cell, from the cell's value f and
// its lower and upper neighbours: its candidate and weight as the left cell of
// the face above it (fL, oL) and as the right cell of the face below it (fR,
// oR).  Both share A, B and their three products, which vxd::weno forms once
// per face and side.  The weights are 1 / (mm + b)^2, twice vxd::weno's: the
// ratios oL / (oL + oR) have the same bits.  Valid for |f| below WENO_MAX (the
// squares then stay below 2^770 and the weights above 2^-770, inside
// rcp_refined's range); the callers take vxd::weno for larger values and NaN.
constexpr double WENO_MAX = 0x1p190;
struct WenoCell {
    double fL, oL, fR, oR;
};
__device__ __forceinline__ WenoCell weno_cell(double fm, double f, double fp) {
    WenoCell c;
    const double m5 = 5 * f;
    c.fL = (1.0 / 6) * (-fm + m5 + 2 * fp);
    c.fR = (1.0 / 6) * (2 * fm + m5 - fp);
    const double A = fm - 2 * f + fp;
    const double B = fp - fm;
    const double aa = 4.0 / 3 * (A * A), ab = 0.5 * A * B, bb = 0.25 * (B * B);
    const double mm = 1.0e-10;
    const double sL = mm + (aa + ab + bb), sR = mm + (aa - ab + bb);
    const double dL = sL * sL, dR = sR * sR;
    const double rL = rcp_refined(dL), rR = rcp_refined(dR);
    c.oL = __builtin_fma(__builtin_fma(-dL, rL, 1.0), rL, rL);
    c.oR = __builtin_fma(__builtin_fma(-dR, rR, 1.0), rR, rR);
    return c;
}
// Face value from the left cell's (fL, oL) and the right cell's (fR, oR): the
// bits of vxd::weno.
__device__ __forceinline__ double weno_face(double fL, double oL, double fR, double oR, bool right) {
    const double d = oL + oR;
    const double r = rcp_refined(d);
    const double wL = div_refined(oL, d, r);
    const double wR = div_refined(oR, d, r);
    const double wL0 = wL * (0.75 + wL * (wL - 0.5));
    const double wR0 = wR * (0.75 + wR * (wR - 0.5));
    const double s = wL0 + wR0;
    // vxd::weno's choice: the larger weight for right, else the smaller (equal
    // weights give the same value either way)
    const double hi = hwmax(wL0, wR0), lo = hwmin(wL0, wR0);
    const double w = div_refined(right ? hi : lo, s, rcp_refined(s));
    return w * fL + (1 - w) * fR;
}
// Lanes whose value is outside weno_cell's range.
__device__ __forceinline__ uint64_t weno_wide(double f) {
    return __builtin_amdgcn_ballot_w64(!(__builtin_fabs(f) < WENO_MAX));
}

// A value that no lane of the launch writes, at a uniform index: read through
// the scalar cache (s_load), so that it does not queue behind the wavefront's
// vector loads (waiting for the youngest vector load waits for all of them).
__device__ __forceinline__ double ld_uniform(const double *p, int i) {
    typedef const double __attribute__((address_space(4))) *cptr;
    return ((cptr)(uintptr_t)p)[i];
}
// The same for a whole struct of 32-bit words at a uniform address.
template <class T>
__device__ __forceinline__ T ld_uniform_struct(const T *p) {
    typedef const uint32_t __attribute__((address_space(4))) *cptr;
    cptr src = (cptr)(uintptr_t)p;
    uint32_t w[sizeof(T) / 4];
#pragma unroll
    for (size_t k = 0; k < sizeof(T) / 4; k++) w[k] = src[k];
    T t;
    __builtin_memcpy(&t, w, sizeof(T));
    return t;
}
__device__ __forceinline__ bool same_bits(double a, double b) {
    return __builtin_bit_cast(uint64_t, a) == __builtin_bit_cast(uint64_t, b);
}

// EMSolver.cpp:558-585: plain two-candidate WENO for the face potentials
__device__ __forceinline__ double face_weno(double f1, double f2, double f3, double f4) {
    double fL = (1.0 / 6) * (-f1 + 5 * f2 + 2 * f3);
    double fR = (1.0 / 6) * (2 * f2 + 5 * f3 - f4);
    double AL = f1 - 2 * f2 + f3;
    double BL = f3 - f1;
    double AR = f2 - 2 * f3 + f4;
    double BR = f4 - f2;
    double bL = 4.0 / 3 * (AL * AL) + 0.5 * AL * BL + 0.25 * (BL * BL);
    double bR = 4.0 / 3 * (AR * AR) - 0.5 * AR * BR + 0.25 * (BR * BR);
    const double mm = 1.0e-10;
    double oL = 0.5 / ((mm + bL) * (mm + bL));
    double oR = 0.5 / ((mm + bR) * (mm + bR));
    double wL = oL / (oL + oR);
    double wR = oR / (oL + oR);
    return wL * fL + wR * fR;
}

// Element of row i (uniform) at the lane's byte lb of a row: the row's address
// stays in scalar registers and the lane adds a 32-bit offset.
__device__ __forceinline__ double *elem(double *pl, int pitch, int i, uint32_t lb) {
    return (double *)((char *)(pl + (long)(i + 2) * pitch) + lb);
}

// Row i of a plane at the lane's (clamped) column, with i clamped into the
// plane: no branch around the load, so that the loads in flight are counted
// one by one and a row waits only for its own; the caller masks the value (0
// outside the plane) where it uses it.
__device__ __forceinline__ double ldr(const double *pl, int pitch, int nx, int i, uint32_t lb) {
    const int ic = i < -2 ? -2 : (i > nx + 1 ? nx + 1 : i);
    return *elem(const_cast<double *>(pl), pitch, ic, lb);
}

// Whole-wavefront lane shifts by one lane (DPP wave_shl:1 / wave_shr:1, plain
// VALU moves instead of LDS permutes): shdn gives lane l the value of lane
// l + 1, shup the value of lane l - 1.  The end lane (63, resp. 0) receives 0;
// it is a halo lane, as are its neighbours that consume it.
template <int CTRL>
__device__ __forceinline__ double wave_shift1(double v) {
    const int lo = __double2loint(v), hi = __double2hiint(v);
    const int rlo = __builtin_amdgcn_mov_dpp(lo, CTRL, 0xf, 0xf, true);
    const int rhi = __builtin_amdgcn_mov_dpp(hi, CTRL, 0xf, 0xf, true);
    return __hiloint2double(rhi, rlo);
}
constexpr int DPP_WAVE_SHL1 = 0x130;
constexpr int DPP_WAVE_SHR1 = 0x138;
__device__ __forceinline__ double shdn1(double v) { return wave_shift1<DPP_WAVE_SHL1>(v); }
__device__ __forceinline__ double shup1(double v) { return wave_shift1<DPP_WAVE_SHR1>(v); }

// Mixed-precision helpers: f scaled by an exact power of two (sinv = 2^-k
// with 2^k near the patch's max |f|) and rounded to FP32 for the WENO weights
// and the Zalesak ratios; face values, fluxes and updates stay FP64.
// The parts of the mixed-precision WENO that belong to one cell, as vxd::WenoCell:
// candidates in FP64 and smoothness measures in FP32 (g: f * sinv in FP32), each
// formed once per cell instead of once per face and side.
struct WenoCellMp {
    double fL, fR;
    float bL, bR;
};
__device__ __forceinline__ WenoCellMp weno_cell_mp(double fm, double f, double fp, float gm, float g, float gp,
                                                   float eps) {
    WenoCellMp c;
    const double m5 = 5 * f;
    c.fL = (1.0 / 6) * (-fm + m5 + 2 * fp);
    c.fR = (1.0 / 6) * (2 * fm + m5 - fp);
    const float A = gm - 2 * g + gp, B = gp - gm;
    const float aa = 4.0f / 3 * (A * A), ab = 0.5f * A * B, bb = 0.25f * (B * B);
    c.bL = eps + (aa + ab + bb);
    c.bR = eps + (aa - ab + bb);
    return c;
}
// Face value from the left cell's (fL, bL) and the right cell's (fR, bR): weights in
// FP32, the blend in FP64; same candidate choice as vxd::weno.
__device__ __forceinline__ double weno_face_mp(double fL, float bL, double fR, float bR, bool right) {
    // oL / (oL + oR) with o = 0.5 / b^2 is bR^2 / (bL^2 + bR^2); both are
    // divided by the larger b first, so the squares stay in [0, 1]
    const float m = fmaxf(bL, bR);
    const bool ok = m > 1e-30f;
    const float rm = __builtin_amdgcn_rcpf(ok ? m : 1.0f);
    const float x = bL * rm, y = bR * rm, x2 = x * x, y2 = y * y;
    const float rden = __builtin_amdgcn_rcpf(x2 + y2);
    const float wL = ok ? y2 * rden : 0.5f, wR = ok ? x2 * rden : 0.5f;
    const float wL0 = wL * (0.75f + wL * (wL - 0.5f));
    const float wR0 = wR * (0.75f + wR * (wR - 0.5f));
    const bool takeL = right ? (wL0 > wR0) : (wL0 < wR0);
    const float w = (takeL ? wL0 : wR0) * __builtin_amdgcn_rcpf(wL0 + wR0);
    return fR + (double)w * (fL - fR);
}

// Zalesak ratio min(1, Q / P) for P > 0 in FP32 on the scaled values
__device__ __forceinline__ double zalesak_mp(double Q, double P, double sinv) {
    const float qf = (float)(Q * sinv), pf = (float)(P * sinv);
    if (pf > 1e-30f) return (double)fminf(1.0f, qf * __builtin_amdgcn_rcpf(pf));
    return qf > 0.0f ? 1.0 : 0.0;
}

// FP32 lane shifts for the scaled copies of f
__device__ __forceinline__ float shdn1f(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ float shup1f(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x138, 0xf, 0xf, true));
}

}  // namespace vxd
