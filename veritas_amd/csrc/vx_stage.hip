// Fused FCT stage for one patch whose four edges are domain walls (a single
// unrefined level): Rectangle::FCTTimeStep sub-steps 0-2 with the zero ghost
// fills between them (Mesh::Advance, Mesh.cpp:64-89; Rectangle.cpp:1255-1613)
// in one kernel, bit-identical to the sub-step kernels and the CPU oracle.
//
// Design (register streaming, no LDS):
//  * A wavefront owns 64 consecutive p-cells, lane l <-> j = jw - 3 + l.  Every
//    quantity of the stage depends on p-neighbours at most 3 cells away, so
//    lanes 3..60 produce exact results (58 outputs per wavefront) and p
//    neighbours are read from other lanes with cross-lane shuffles.
//  * The wavefront marches along x over a strip of TI output rows.  At march
//    row r it loads f_s(r) and f^n(r) (one coalesced 512-byte row each) and
//    advances a software pipeline held in registers:
//        x-face r-1 : WENO value and high-order flux FxH_s
//        column r   : WENO value; column r-1: high-order flux FpH_s
//        x-face r, column r: low-order fluxes of stage 0 (recomputed from f^n
//                     and the stage-0 fields instead of stored)
//        cell r-1   : low-order predictor f2
//        x-face r-1, column r-1: antidiffusive fluxes FxDS/FpDS
//        cell r-2   : Zalesak R+-
//        cell r-3   : limiter C on its faces and the corrected value f_{s+1}
//  * Store-flux design: FxH_s/FpH_s are written once (owned faces) for the
//    later stages' RK combinations instead of recomputing the WENO fluxes of
//    every earlier stage from stored stage values.  Stage 5 needs the earlier
//    fluxes only through its own combination, so stage 4 writes, in place of
//    FxH_4/FpH_4, stage 5's partial sum b_0 F_0 + ... + b_4 F_4 (left to
//    right, the order stage 5 would use), and stage 5 reads that one plane per
//    direction instead of five: the same bits, 64 B/cell less to read and
//    fewer registers held at stage 5.
// Every quantity is computed only inside the reference's loop range and is 0
// outside it, as the reference's never-written array entries are.
//
// Mixed-precision variant (MP): the divisions of the stage (the WENO weights
// of both face reconstructions, and the Zalesak ratios R+-) run in FP32 on f
// scaled by an exact power of two (f * 2^-k with 2^k near the patch's max |f|);
// the candidate face values, the fluxes, the RK combination and every
// accumulation into f stay FP64.  A face value is fR + w (fL - fR) with the
// FP32 weight w, so its error is of order 1e-7 |fL - fR|, not 1e-7 |f|.

#include <algorithm>
#include <cmath>
#include <functional>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "vx_dev.h"
#include "vx_internal.h"

using namespace vxi;
using namespace vxd;

namespace {

constexpr int HALO = 3;
constexpr int OUTW = 64 - 2 * HALO;  // p-cells produced per wavefront

struct StageArgs {
    vx_patch p;
    const double *fin;  // f_s (stage input), ghost ring zero
    double *fout;       // f_{s+1}; only interior cells are written
    const double *E, *a2;    // fields of this stage (finest grid)
    const double *E0, *a20;  // fields of stage 0 (for the low-order fluxes)
    int n_f;
    int step, ns;
    double a[6], aSum;
    double b5[6];  // stage 5's coefficients times dt (stage 4 forms its partial sum)
    int TI;       // output rows per strip
    int form;     // 0: k_stage; 1: held to four waves per SIMD (k_stage_w4); 2: k_stage_rows
    int nstrip;   // strips in x
    int nbx;      // tiles along p
    double sinv;  // MP: 2^-k, the scale of the FP32 copies of f
    float eps32;  // MP: the WENO epsilon (1e-10) in the scaled units
    double inv_rtb;  // 1.0 / relativeToBottom
};

// A^2 at x-face i (Rectangle.cpp:1280, 1296-1297; EMSolver.cpp:133-135)
__device__ __forceinline__ double face_a2(const StageArgs &A, const double *a2, int i) {
    int fi = A.p.rtb * (i + A.p.x_pos);
    int c = fi < 0 ? 0 : (fi > A.n_f ? A.n_f : fi);
    return ld_uniform(a2, c);
}

// q * Rectangle::GetEfield(i) (Rectangle.cpp:1055-1067, 1298; vxd::patch_E)
__device__ __forceinline__ double col_qE(const StageArgs &A, const double *E, int i) {
    const int j = A.p.rtb * (i + A.p.x_pos);
    double t = 0.0;
    for (int k = 0; k < A.p.rtb; k++) {
        int m = j + k;
        m = m < 0 ? m + A.n_f : (m >= A.n_f ? m - A.n_f : m);
        t += ld_uniform(E, m);
    }
    t *= A.inv_rtb;
    return A.p.q * t;
}

// XCD-aware tile order (vxd::xcd_order): p-neighbouring tiles march over the
// same rows on the same XCD and share their overlapping halos in its L2.
__device__ __forceinline__ int xcd_tile() { return xcd_order((int)blockIdx.x, (int)gridDim.x); }

// A strip of one wavefront: TI output rows [i0, i1) of the 58 p-cells from jw.
// IN (interior): the strip and its p-column lie so far from the patch edges
// that every reference loop-range test below holds for every lane and every
// march row (interior_strip states the margins), so IN only drops tests that
// are true, and the IN and general forms give the same bits.
// FULL: divisions over the whole FP64 range (vxd::weno).  The other form
// (vxd::weno_cell, weno_face) holds for |f| below vxd::WENO_MAX; it returns
// the lanes that met a larger value (or NaN), and the caller then runs the
// strip again as FULL: a strip reads nothing that it writes, so the second
// run replaces every value of the first.
//
// What bounds it (4096 x 4096, MI355X): FP64 VALU issue, about 345 wave64
// instructions per 58-cell row (461 before the parts that both sides of a face
// share were formed once per cell, the divisions shortened, the x-speeds kept
// where A^2 does not change and each limited flux formed once), two thirds of
// the issue slots at three waves per SIMD; at stages 3 and 4 the stored fluxes
// (88 and 104 B/cell) come close to the memory's rate as well.  The six stages
// of a step: 2.62 ms before, 2.04 ms now (stage 0..5: 262, 290, 330, 384, 472,
// 267 us).
template <int STEP, bool MP, bool IN, bool FULL>
__device__ __forceinline__ uint64_t stage_strip(const StageArgs &A, const int jw, const int i0) {
    const vx_patch &P = A.p;
    const int nx = P.n_x, np = P.n_p, pitch = P.pitch;
    const int lane = threadIdx.x & 63;
    const int i1 = min(i0 + A.TI, nx);       // output rows [i0, i1)
    const bool last_strip = i0 + A.TI >= nx;
    const int j = jw - HALO + lane;
    const bool mid_lane = lane >= HALO && lane < 64 - HALO;
    const bool out_lane = mid_lane && (IN || j < np);
    // faces this wavefront stores (each valid face has exactly one owner)
    const bool own_row_x = IN ? mid_lane
                              : (mid_lane && j < np) || (j == np && lane >= HALO && lane < 65 - HALO) ||
                                    (jw == 0 && j == -1);
    const bool own_row_p = IN ? mid_lane : (mid_lane && j < np) || (j == np && lane >= HALO && lane < 65 - HALO);
    constexpr bool store_flux = STEP < 5;

    // reference loop ranges in j (Rectangle.cpp:1279-1394) for this lane
    const bool jr_ex = IN || (j >= -1 && j < np + 1);   // ex, fx, FxH, FxL rows
    const bool jr_ep = IN || (j >= -1 && j < np + 2);   // ep
    const bool jr_fp = IN || (j >= 0 && j < np + 1);    // fp, FpH, FpL p-faces
    const bool jr_R = IN || (j >= -1 && j < np + 1);    // R
    const bool jint = IN || (j >= 0 && j < np);
    // update loop ranges (walls on all sides: xm = 1, xp = n_x, pm = 1, pp = n_p)
    const int xm = P.left ? 1 : 0, xp = P.right ? nx : nx + 1;
    const int pm = P.down ? 1 : 0, pp = P.up ? np : np + 1;
    const bool jr_u = IN || (j >= pm && j < pp), jr_u1 = IN || (j + 1 >= pm && j + 1 < pp);

    const double mc2 = P.mc2inv;
    const double dpcc = P.dp_inv * P.cc;
    const double ccdx = P.cc * P.dx_inv;
    const double w3 = 1 / 48.0;
    const double pj = momentum(P.pmin, P.dp, j, P.p_pos);

    const double *fin = A.fin, *f0p = P.f[0];
    const int r0 = i0 - HALO;

    // pipeline state (names: _mK = row/face r-K)
    double fs_m3 = 0, fs_m2 = 0, fs_m1 = 0, fs_0 = 0;  // (fs_m3: FULL only)
    double f0_m1 = 0, f0_0 = 0;
    double ep_m2 = 0, ep_m1 = 0, ep_0 = 0, fp_m2 = 0, fp_m1 = 0, fp_0 = 0;
    double xL_m1 = 0, xL_0 = 0, pL_m1 = 0, pL_0 = 0;  // stage-0 low-order fluxes times aSum
    double f2_m2 = 0, f2_m1 = 0;
    double hi_m3 = 0, hi_m2 = 0, hi_m1 = 0, lo_m3 = 0, lo_m2 = 0, lo_m1 = 0;  // larger, smaller of f^n and f^td
    double FxD_m2 = 0, FxD_m1 = 0, FpD_m2 = 0, FpD_m1 = 0;
    double Rp_m3 = 0, Rp_m2 = 0, Rm_m3 = 0, Rm_m2 = 0;
    double t_m3 = 0;  // corrected value of cell r-3 but for its upper x-face
    float gs_m2 = 0, gs_m1 = 0, gs_0 = 0;  // MP: FP32 copies of f_s rows
    double fL_m2 = 0, oL_m2 = 0;  // WENO candidate and weight of cell r-2 at its upper x-face
    float bL_m2 = 0;              // MP: its smoothness measure in place of the weight
    uint64_t wide = 0;
    const double sinv = A.sinv;
    const float eps32 = A.eps32;

    // Gamma(p_j, q^2 A^2 at x-face i), current fields and stage-0 fields.  It
    // changes along x only where A^2 does (inside a pulse), and so do the
    // x-speeds ex formed from it: each is formed again only where the face's
    // A^2 differs from the face before (a uniform branch).
    const double qq = P.q * P.q;
    double a2_0 = face_a2(A, A.a2, r0), a2_m1 = face_a2(A, A.a2, r0 - 1);
    double G_m1 = gamma_(pj, qq * a2_m1, mc2);
    double G_0 = same_bits(a2_0, a2_m1) ? G_m1 : gamma_(pj, qq * a2_0, mc2);
    double a20_0 = face_a2(A, A.a20, r0);
    double G0_0 = (STEP == 0 || same_bits(a20_0, a2_0)) ? G_0 : gamma_(pj, qq * a20_0, mc2);
    // ex at x-face r-1 and its difference over lanes j+1, j-1; ex of stage 0
    // at x-face r (lanes outside the p-range hold 0)
    double ex = 0.0, dex = 0.0, ex0 = 0.0;
    bool new_m1 = true, new_0 = true, new0_0 = true;  // face r-1, r / stage 0's face r differs from the one before
    double a2_p1 = face_a2(A, A.a2, r0 + 1), a20_p1 = face_a2(A, A.a20, r0 + 1);

    // software prefetch: rows r and r+1 are in flight before iteration r, the
    // stored fluxes of x-face / column r-1 one iteration ahead
    const bool in_j = IN || (j >= -2 && j < np + 2);
    const int jc = IN ? j : (j < -2 ? -2 : (j > np + 1 ? np + 1 : j));
    const uint32_t lb = 8u * (uint32_t)(jc + 2);  // the lane's byte in a row
    auto row_ok = [&](int i) { return IN || (i >= -2 && i < nx + 2 && in_j); };
    double pfs_a = ldr(fin, pitch, nx, r0, lb), pf0_a = ldr(f0p, pitch, nx, r0, lb);
    double pfs_b = ldr(fin, pitch, nx, r0 + 1, lb), pf0_b = ldr(f0p, pitch, nx, r0 + 1, lb);
    // stored flux planes read by this stage; stage 5 reads only plane 4, which
    // holds its partial sum
    constexpr int NH = STEP == 5 ? 1 : (STEP > 0 ? STEP : 1);
    double hx[NH], hp[NH];
    bool hvx = false, hvp = false;  // the loaded face lies in the FxH / FpH ranges
    auto load_h = [&](int face) {
        hvx = IN || (face >= 0 && face < nx + 1 && jr_ex);
        hvp = IN || (face >= -1 && face < nx + 1 && jr_fp);
#pragma unroll
        for (int k = 0; k < NH; k++) {
            const int plane = STEP == 5 ? 4 : k;
            hx[k] = (k < STEP) ? ldr(P.FxH[plane], pitch, nx, face, lb) : 0.0;
            hp[k] = (k < STEP) ? ldr(P.FpH[plane], pitch, nx, face, lb) : 0.0;
        }
    };
    load_h(r0 - 1);

    // The RK combination sum_k a_k FxH_k is evaluated left to right; the terms
    // of the earlier stages are folded into Sx/Sp as soon as their prefetched
    // values are consumed, which frees their registers a whole iteration early.
    // Stage 4 folds the same values into stage 5's partial sum Qx/Qp.
    double Sx = 0.0, Sp = 0.0, Qx = 0.0, Qp = 0.0;

    // One march row; each quantity is masked to its reference loop range.
    auto row = [&](int r) {
        // ---- ingest row r
        fs_0 = row_ok(r) ? pfs_a : 0.0;
        f0_0 = row_ok(r) ? pf0_a : 0.0;
        if (MP) gs_0 = (float)(fs_0 * sinv);
        pfs_a = pfs_b;
        pf0_a = pf0_b;
        pfs_b = ldr(fin, pitch, nx, r + 2, lb);
        pf0_b = ldr(f0p, pitch, nx, r + 2, lb);
        if (STEP == 5) {
            // b_0 F_0 + ... + b_4 F_4 as stage 4 formed it; outside the face
            // ranges the masked sum of the five terms is +0
            Sx = hvx ? hx[0] : 0.0;
            Sp = hvp ? hp[0] : 0.0;
        } else if (STEP > 0) {
            Sx = A.a[0] * (hvx ? hx[0] : 0.0);
            Sp = A.a[0] * (hvp ? hp[0] : 0.0);
#pragma unroll
            for (int k = 1; k < NH; k++) {
                Sx = Sx + A.a[k] * (hvx ? hx[k] : 0.0);
                Sp = Sp + A.a[k] * (hvp ? hp[k] : 0.0);
            }
            if (STEP == 4) {
                Qx = A.b5[0] * (hvx ? hx[0] : 0.0);
                Qp = A.b5[0] * (hvp ? hp[0] : 0.0);
#pragma unroll
                for (int k = 1; k < NH; k++) {
                    Qx = Qx + A.b5[k] * (hvx ? hx[k] : 0.0);
                    Qp = Qp + A.b5[k] * (hvp ? hp[k] : 0.0);
                }
            }
        }
        load_h(r);
        // the next row's A^2 is read one row ahead
        const double a2_p2 = face_a2(A, A.a2, r + 2), a20_p2 = STEP == 0 ? a2_p2 : face_a2(A, A.a20, r + 2);
        const bool new_p1 = !same_bits(a2_p1, a2_0);
        const bool new0_p1 = STEP == 0 ? new_p1 : !same_bits(a20_p1, a20_0);
        double G_p1 = G_0, dG = 0.0;  // dG: the force's Gamma term at column r
        if (new_p1) {
            G_p1 = gamma_(pj, qq * a2_p1, mc2);
            dG = ccdx * (G_p1 - G_0);
        }
        double G0_p1, dG0 = 0.0;
        if (STEP == 0) {
            G0_p1 = G_p1;
            dG0 = dG;
        } else {
            G0_p1 = G0_0;
            if (new0_p1) {
                G0_p1 = same_bits(a20_p1, a2_p1) ? G_p1 : gamma_(pj, qq * a20_p1, mc2);
                dG0 = ccdx * (G0_p1 - G0_0);
            }
        }

        // ---- x-face r-1: ex, fx (Rectangle.cpp:1278-1293), FxH_s (1313-1334)
        const int ix = r - 1;
        const bool vFx = IN || (ix >= 0 && ix < nx + 1 && jr_ex);
        if (new_m1) {  // (used on rows of the face range only)
            const double Gd = shdn1(G_m1);  // Gamma at p-face j+1
            ex = jr_ex ? dpcc * (Gd - G_m1) : 0.0;
            dex = shdn1(ex) - shup1(ex);
        }
        double fx = 0.0;
        if (MP) {
            const WenoCellMp c = weno_cell_mp(fs_m2, fs_m1, fs_0, gs_m2, gs_m1, gs_0, eps32);  // cell r-1
            if (vFx) fx = weno_face_mp(fL_m2, bL_m2, c.fR, c.bR, ex > 0.0);
            fL_m2 = c.fL;
            bL_m2 = c.bL;
        } else if (FULL) {
            if (vFx) fx = weno(fs_m3, fs_m2, fs_m1, fs_0, ex > 0.0);
        } else {
            wide |= weno_wide(fs_0);
            const WenoCell c = weno_cell(fs_m2, fs_m1, fs_0);  // cell r-1
            if (vFx) fx = weno_face(fL_m2, oL_m2, c.fR, c.oR, ex > 0.0);
            fL_m2 = c.fL;
            oL_m2 = c.oL;
        }
        double fx_u = shdn1(fx), fx_d = shup1(fx);
        double FxH = vFx ? P.dx_inv * (fx * ex + w3 * (fx_u - fx_d) * dex) : 0.0;

        // ---- column r: ep, fp (Rectangle.cpp:1294-1312)
        const bool cr = IN || (r >= -1 && r < nx + 1);
        double qE = cr ? col_qE(A, A.E, r) : 0.0;
        ep_0 = (cr && jr_ep) ? qE - dG : 0.0;
        double s1 = shup1(fs_0), s3 = shdn1(fs_0);
        fp_0 = 0.0;
        // the left cell's candidate and weight come from the lane below
        if (MP) {
            const WenoCellMp c = weno_cell_mp(s1, fs_0, s3, shup1f(gs_0), gs_0, shdn1f(gs_0), eps32);
            const double fl = shup1(c.fL);
            const float bl = shup1f(c.bL);
            if (cr && jr_fp) fp_0 = weno_face_mp(fl, bl, c.fR, c.bR, ep_0 > 0.0);
        } else if (FULL) {
            const double s2 = shup1(s1);
            if (cr && jr_fp) fp_0 = weno(s2, s1, fs_0, s3, ep_0 > 0.0);
        } else {
            const WenoCell c = weno_cell(s1, fs_0, s3);
            const double fl = shup1(c.fL), ol = shup1(c.oL);
            if (cr && jr_fp) fp_0 = weno_face(fl, ol, c.fR, c.oR, ep_0 > 0.0);
        }
        // ---- column r-1: FpH_s (Rectangle.cpp:1353-1375)
        const bool vFp = IN || (ix >= -1 && ix < nx + 1 && jr_fp);
        double FpH = vFp ? P.dp_inv * (fp_m1 * ep_m1 + w3 * (fp_0 - fp_m2) * (ep_0 - ep_m2)) : 0.0;
        if (store_flux) {
            const bool own_x = ix >= i0 && (ix < i0 + A.TI || last_strip);
            const bool own_c = (ix >= i0 || i0 == 0) && (ix < i0 + A.TI || last_strip);
            // read again only by the later stages: streamed past the caches;
            // stage 4 stores stage 5's partial sum instead of its fluxes
            const double hx_out = STEP == 4 ? Qx + A.b5[4] * FxH : FxH;
            const double hp_out = STEP == 4 ? Qp + A.b5[4] * FpH : FpH;
            if (vFx && own_x && own_row_x) __builtin_nontemporal_store(hx_out, elem(P.FxH[STEP], pitch, ix, lb));
            if (vFp && own_c && own_row_p) __builtin_nontemporal_store(hp_out, elem(P.FpH[STEP], pitch, ix, lb));
        }

        // ---- low-order fluxes of stage 0 at x-face r and column r
        // (Rectangle.cpp:1335-1352, 1376-1394 evaluated with the stage-0 fields)
        if (new0_0) ex0 = dpcc * (shdn1(G0_0) - G0_0);
        xL_0 = (IN || (r >= 0 && r < nx + 1 && jr_ex)) ? A.aSum * (P.dx_inv * ((ex0 > 0.0 ? f0_m1 : f0_0) * ex0)) : A.aSum * 0.0;
        double qE0 = cr ? col_qE(A, A.E0, r) : 0.0;
        double ep0 = qE0 - dG0;
        double f0_jm1 = shup1(f0_0);
        pL_0 = (cr && jr_fp) ? A.aSum * (P.dp_inv * ((ep0 > 0.0 ? f0_jm1 : f0_0) * ep0)) : A.aSum * 0.0;

        // ---- cell r-1: low-order predictor (Rectangle.cpp:1518-1534, gather form)
        {
            const int i = r - 1;
            double pL_up = shdn1(pL_m1);  // at (i, j+1)
            double t = 0.0;
            if (IN || (i >= 0 && i < nx && jint)) {
                t = f0_m1;
                const bool in0 = IN || (i >= xm && i < xp && jr_u);
                if (in0) {
                    t += xL_m1;
                    t += pL_m1;
                }
                if (IN || (i >= xm && i < xp && jr_u1)) t -= pL_up;
                if (IN || (i + 1 >= xm && i + 1 < xp && jr_u)) t -= xL_0;
            }
            f2_m1 = t;  // ghost cells: zero fill of the walls (BoundaryCondition.cpp:6-8)
            hi_m1 = hwmax(f0_m1, t);
            lo_m1 = hwmin(f0_m1, t);
        }

        // ---- x-face r-1 and column r-1: RK flux combination (Rectangle.cpp:1396-1517)
        {
            double sx = STEP == 0 ? A.a[0] * FxH : Sx + A.a[STEP] * FxH;
            double sp = STEP == 0 ? A.a[0] * FpH : Sp + A.a[STEP] * FpH;
            FxD_m1 = sx - xL_m1;
            FpD_m1 = sp - pL_m1;
        }

        // ---- cell r-2: Zalesak R+- (Rectangle.cpp:1538-1579)
        {
            const int i = r - 2;
            double FpDu = shdn1(FpD_m2);  // FpDS at (i, j+1)
            double hu = shdn1(hi_m2), hd = shup1(hi_m2);
            double lu = shdn1(lo_m2), ld = shup1(lo_m2);
            double rp = 0.0, rm = 0.0;
            if (IN || (i >= -1 && i < nx + 1 && jr_R)) {
                // hwmax/hwmin (one v_max_f64/v_min_f64 each) give the reference's
                // a > b ? a : b bits here: f is never -0 (every update adds to a
                // +0 or positive start), R and Q are never -0, nothing is NaN,
                // and a signed zero among the P terms reaches P only when P is
                // zero, where R is 0 either way
                double Pp = hwmax0(FxD_m2) - hwmin0(FxD_m1) + hwmax0(FpD_m2) - hwmin0(FpDu);
                double Pm = hwmax0(FxD_m1) - hwmin0(FxD_m2) + hwmax0(FpDu) - hwmin0(FpD_m2);
                double wMax = hwmax(hi_m2, hwmax(hi_m1, hwmax(hi_m3, hwmax(hu, hd))));
                double wMin = hwmin(lo_m2, hwmin(lo_m1, hwmin(lo_m3, hwmin(lu, ld))));
                double Qm = -wMin + f2_m2;
                double Qp = wMax - f2_m2;
                if (MP) {
                    rp = Pp > 0.0 ? zalesak_mp(Qp, Pp, sinv) : 0.0;
                    rm = Pm > 0.0 ? zalesak_mp(Qm, Pm, sinv) : 0.0;
                } else {
                    // min(1, Q / P) is 1 where Q >= P: only a wavefront with a
                    // lane below that (beside an extremum of f) divides
                    rp = Pp > 0.0 ? 1.0 : 0.0;
                    rm = Pm > 0.0 ? 1.0 : 0.0;
                    if (__builtin_amdgcn_ballot_w64(!(Qp - Pp >= 0.0) || !(Qm - Pm >= 0.0)) != 0) {
                        if (Pp > 0.0) rp = fmin(1.0, Qp / Pp);
                        if (Pm > 0.0) rm = fmin(1.0, Qm / Pm);
                    }
                }
            }
            Rp_m2 = rp;
            Rm_m2 = rm;
        }

        // ---- limiter C of cell r-2's lower faces (Rectangle.cpp:1581-1594) and
        // the corrected value (Rectangle.cpp:1596-1612, gather form): a cell
        // takes its lower x-face and its p-faces at this row and its upper x-face
        // at the next, each limited flux formed once, in the reference's order
        {
            const int i = r - 2;
            double Rpd = shup1(Rp_m2), Rmd = shup1(Rm_m2);  // R at (i, j-1)
            const bool lim = IN || (i >= 1 && i < nx && jint);
            double cx = lim ? (FxD_m2 > 0.0 ? hwmin(Rp_m2, Rm_m3) : hwmin(Rp_m3, Rm_m2)) : 1.0;
            double cp = lim ? (FpD_m2 > 0.0 ? hwmin(Rp_m2, Rmd) : hwmin(Rpd, Rm_m2)) : 1.0;
            const double lx = cx * FxD_m2, lp = cp * FpD_m2;
            const double lpu = shdn1(lp);  // the limited flux at (i, j+1), formed by the next lane
            if (out_lane && i - 1 >= i0 && i - 1 < i1) {
                double t = t_m3;
                if (IN || (i >= xm && i < xp && jr_u)) t -= lx;
                *elem(A.fout, pitch, i - 1, lb) = t;
            }
            double t = f2_m2;
            if (IN || (i >= xm && i < xp && jr_u)) {
                t += lx;
                t += lp;
            }
            if (IN || (i >= xm && i < xp && jr_u1)) t -= lpu;
            t_m3 = t;
        }

        // ---- shift the pipeline by one row
        if (FULL) fs_m3 = fs_m2;
        fs_m2 = fs_m1; fs_m1 = fs_0;
        gs_m2 = gs_m1; gs_m1 = gs_0;
        f0_m1 = f0_0;
        a2_0 = a2_p1; a2_p1 = a2_p2; a20_0 = a20_p1; a20_p1 = a20_p2;
        new_m1 = new_0; new_0 = new_p1; new0_0 = new0_p1;
        G_m1 = G_0; G_0 = G_p1; G0_0 = G0_p1;
        ep_m2 = ep_m1; ep_m1 = ep_0; fp_m2 = fp_m1; fp_m1 = fp_0;
        xL_m1 = xL_0; pL_m1 = pL_0;
        f2_m2 = f2_m1;
        hi_m3 = hi_m2; hi_m2 = hi_m1; lo_m3 = lo_m2; lo_m2 = lo_m1;
        FxD_m2 = FxD_m1; FpD_m2 = FpD_m1;
        Rp_m3 = Rp_m2; Rm_m3 = Rm_m2;
    };

    // Two rows at a time turn the pipeline's shifts (37 64-bit moves of 362 VALU
    // instructions a row) into register names.  Stage 4 holds eight stored
    // fluxes in flight and would spill (4096 x 4096: 472 us one row at a time,
    // 495 two), as would the mixed-precision stage 3.
    constexpr bool TWO = IN && STEP != 4 && !(MP && STEP == 3);
    if (TWO) {
        int r = r0;
        for (; r < i1 + HALO - 1; r += 2) {
            row(r);
            row(r + 1);
        }
        if (r == i1 + HALO - 1) row(r);
    } else {
        for (int r = r0; r <= i1 + HALO - 1; r++) row(r);
    }
    return wide;
}

// Whether a strip takes the IN form.  Lanes hold j in [jw - 3, jw + 60] and
// the march rows are r in [i0 - 3, i1 + 2] with i1 = i0 + TI; the tightest
// tests above are the updates of cells (r - 1, j) and (r - 3, j) with their
// +1 neighbours inside [1, n - 1) (xm, pm <= 1, xp >= n_x, pp >= n_p), which
// need 1 <= j <= n_p - 2 and 4 <= r <= n_x - 1, and the stored-flux faces
// r0 - 1 >= 0.  The margins below are wider than that.
__device__ __forceinline__ bool interior_strip(const StageArgs &A, int jw, int i0) {
    return jw >= 8 && jw + 64 <= A.p.n_p && i0 >= 8 && i0 + A.TI + 8 <= A.p.n_x;
}

// One workgroup's tile (4 strips of one 64-lane p-column) of a stage.
template <int STEP, bool MP>
__device__ __forceinline__ void stage_tile(const StageArgs &A, const int tile) {
    // the wavefront index is uniform: row loop, row ranges and field reads stay scalar
    const int bx = tile % A.nbx, by = tile / A.nbx;
    const int strip = by * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (strip >= A.nstrip) return;  // uniform per wavefront
    const int jw = bx * OUTW, i0 = strip * A.TI;
    const uint64_t wide = interior_strip(A, jw, i0) ? stage_strip<STEP, MP, true, false>(A, jw, i0)
                                                    : stage_strip<STEP, MP, false, false>(A, jw, i0);
    if (!MP && wide != 0) stage_strip<STEP, MP, false, true>(A, jw, i0);
}

// Compiled for at least three resident waves per SIMD (at most 168 VGPRs):
// the FP64 stages fit as they are; the mixed-precision stage 4 (173 otherwise)
// keeps a few values in scratch instead of running two waves per SIMD.
template <int STEP, bool MP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_stage(StageArgs A) {
    stage_tile<STEP, MP>(A, xcd_tile());
}
// The same stage compiled for four resident waves per SIMD (at most 128
// VGPRs; the stages after 0 then keep values in scratch): more waves to hide
// latency against a few more loads.  The strip-height timing picks between the two
// forms at stage 0 only (tile_rows has the figures); VX_TILE_ROWS pins either at
// every stage.  Both give the same bits.
template <int STEP, bool MP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_stage_w4(StageArgs A) {
    stage_tile<STEP, MP>(A, xcd_tile());
}

// The same stage with one wavefront per row, for patches too small to fill the
// device with long strips: a workgroup owns TI output rows of a p-column and
// runs TI + 4 wavefronts, wavefront w at row r = i0 - 2 + w (x-face r, column r
// and cell r).  What a row takes from the rows beside it goes through LDS, with
// a workgroup barrier per hand-over: (fp, ep), then (FxDS and the extrema of
// f^n and f^td), then R.  Each value is formed by the strip's operations, so
// the bits are the strip's.
// A strip of TI rows walks TI + 6 rows one after another, each a dependent
// chain of two reconstructions; here they run at once.  601 x 333 cells with a
// pulse (MI355X): 21 to 25 us a stage as strips, 10 to 12 here; 64 x 256 cells:
// 23 and 6 us.  The price is (TI + 4) / TI rows of work per output row,
// so strips win where they fill the device.
constexpr int RT_ARRAYS = 7;  // LDS rows of 64 doubles per wavefront

__device__ __forceinline__ double &lds_row(double *lds, int nw, int q, int w) {
    return lds[(q * nw + w) * 64 + (threadIdx.x & 63)];
}

template <int STEP, bool MP>
__device__ __forceinline__ void stage_rows(const StageArgs &A, const int tile, double *lds) {
    const vx_patch &P = A.p;
    const int nx = P.n_x, np = P.n_p, pitch = P.pitch;
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = A.TI + 4;
    const int bx = tile % A.nbx, by = tile / A.nbx;
    const int jw = bx * OUTW, i0 = by * A.TI, r = i0 - 2 + w;
    const int i1 = min(i0 + A.TI, nx);  // output rows [i0, i1)
    const bool last_strip = i0 + A.TI >= nx;
    const int j = jw - HALO + lane;
    const bool mid_lane = lane >= HALO && lane < 64 - HALO;
    const bool out_lane = mid_lane && j < np;
    const bool own_row_p = out_lane || (j == np && lane >= HALO && lane < 65 - HALO);
    const bool own_row_x = own_row_p || (jw == 0 && j == -1);
    // reference loop ranges (Rectangle.cpp:1279-1394, 1518-1612)
    const bool jint = j >= 0 && j < np;
    const bool jr_ex = j >= -1 && j < np + 1, jr_ep = j >= -1 && j < np + 2, jr_fp = j >= 0 && j < np + 1;
    const int xm = P.left ? 1 : 0, xp = P.right ? nx : nx + 1;
    const int pm = P.down ? 1 : 0, pp = P.up ? np : np + 1;
    const bool jr_u = j >= pm && j < pp, jr_u1 = j + 1 >= pm && j + 1 < pp;
    const bool in_r = r >= xm && r < xp, in_r1 = r + 1 >= xm && r + 1 < xp;
    const bool vFx = r >= 0 && r < nx + 1 && jr_ex;
    const bool cr = r >= -1 && r < nx + 1;
    const bool vFp = cr && jr_fp;

    // every load of the row at once
    const bool in_j = j >= -2 && j < np + 2;
    const int jc = j < -2 ? -2 : (j > np + 1 ? np + 1 : j);
    const uint32_t lb = 8u * (uint32_t)(jc + 2);
    auto row_ok = [&](int i) { return i >= -2 && i < nx + 2 && in_j; };
    double fs[4], f0[3];  // f_s at rows r-2 .. r+1, f^n at rows r-1 .. r+1
#pragma unroll
    for (int k = 0; k < 4; k++) fs[k] = ldr(A.fin, pitch, nx, r - 2 + k, lb);
#pragma unroll
    for (int k = 0; k < 3; k++) f0[k] = ldr(P.f[0], pitch, nx, r - 1 + k, lb);
    constexpr int NH = STEP == 5 ? 1 : (STEP > 0 ? STEP : 1);
    double hx[NH], hp[NH];
#pragma unroll
    for (int k = 0; k < NH; k++) {
        const int plane = STEP == 5 ? 4 : k;
        hx[k] = k < STEP ? ldr(P.FxH[plane], pitch, nx, r, lb) : 0.0;
        hp[k] = k < STEP ? ldr(P.FpH[plane], pitch, nx, r, lb) : 0.0;
    }
    const double qq = P.q * P.q, mc2 = P.mc2inv;
    const double dpcc = P.dp_inv * P.cc, ccdx = P.cc * P.dx_inv, w3 = 1 / 48.0;
    const double pj = momentum(P.pmin, P.dp, j, P.p_pos);

    // Gamma at x-faces r, r+1 (and r+1 of stage 0), the speeds
    const double a2_0 = face_a2(A, A.a2, r), a2_1 = face_a2(A, A.a2, r + 1);
    const double G_0 = gamma_(pj, qq * a2_0, mc2);
    double G_1 = G_0, dG = 0.0;
    if (!same_bits(a2_1, a2_0)) {
        G_1 = gamma_(pj, qq * a2_1, mc2);
        dG = ccdx * (G_1 - G_0);
    }
    const double Gd = shdn1(G_0);  // (lane shifts run with every lane active)
    const double ex = jr_ex ? dpcc * (Gd - G_0) : 0.0;
    const double dex = shdn1(ex) - shup1(ex);
    double G0_0 = G_0, G0_1 = G_1, dG0 = dG;
    if (STEP > 0) {
        const double b_0 = face_a2(A, A.a20, r), b_1 = face_a2(A, A.a20, r + 1);
        if (!same_bits(b_0, a2_0)) G0_0 = gamma_(pj, qq * b_0, mc2);
        if (!same_bits(b_1, a2_1)) G0_1 = gamma_(pj, qq * b_1, mc2);
        dG0 = ccdx * (G0_1 - G0_0);
    }
    const double ex0 = dpcc * (shdn1(G0_0) - G0_0), ex0_1 = dpcc * (shdn1(G0_1) - G0_1);

    uint64_t wide[4];
    float gs[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        fs[k] = row_ok(r - 2 + k) ? fs[k] : 0.0;
        if (MP) gs[k] = (float)(fs[k] * A.sinv);
        else wide[k] = weno_wide(fs[k]);
    }
#pragma unroll
    for (int k = 0; k < 3; k++) f0[k] = row_ok(r - 1 + k) ? f0[k] : 0.0;

    // ---- x-face r
    double fx = 0.0;
    if (MP) {
        const WenoCellMp cl = weno_cell_mp(fs[0], fs[1], fs[2], gs[0], gs[1], gs[2], A.eps32);
        const WenoCellMp ch = weno_cell_mp(fs[1], fs[2], fs[3], gs[1], gs[2], gs[3], A.eps32);
        if (vFx) fx = weno_face_mp(cl.fL, cl.bL, ch.fR, ch.bR, ex > 0.0);
    } else if (__builtin_expect((wide[0] | wide[1] | wide[2] | wide[3]) != 0, 0)) {
        if (vFx) fx = weno(fs[0], fs[1], fs[2], fs[3], ex > 0.0);
    } else {
        const WenoCell cl = weno_cell(fs[0], fs[1], fs[2]), ch = weno_cell(fs[1], fs[2], fs[3]);
        if (vFx) fx = weno_face(cl.fL, cl.oL, ch.fR, ch.oR, ex > 0.0);
    }
    const double fx_u = shdn1(fx), fx_d = shup1(fx);
    const double FxH = vFx ? P.dx_inv * (fx * ex + w3 * (fx_u - fx_d) * dex) : 0.0;

    // ---- column r
    const double qE = cr ? col_qE(A, A.E, r) : 0.0;
    const double ep = (cr && jr_ep) ? qE - dG : 0.0;
    const double s1 = shup1(fs[2]), s3 = shdn1(fs[2]);
    double fp = 0.0;
    if (MP) {
        const WenoCellMp c = weno_cell_mp(s1, fs[2], s3, shup1f(gs[2]), gs[2], shdn1f(gs[2]), A.eps32);
        const double fl = shup1(c.fL);
        const float bl = shup1f(c.bL);
        if (vFp) fp = weno_face_mp(fl, bl, c.fR, c.bR, ep > 0.0);
    } else if (__builtin_expect(wide[2] != 0, 0)) {
        const double s2 = shup1(s1);
        if (vFp) fp = weno(s2, s1, fs[2], s3, ep > 0.0);
    } else {
        const WenoCell c = weno_cell(s1, fs[2], s3);
        const double fl = shup1(c.fL), ol = shup1(c.oL);
        if (vFp) fp = weno_face(fl, ol, c.fR, c.oR, ep > 0.0);
    }
    lds_row(lds, nw, 0, w) = fp;
    lds_row(lds, nw, 1, w) = ep;

    // ---- stage-0 low-order fluxes of x-faces r, r+1 and column r, and the
    // low-order predictor of cell r
    const double qE0 = cr ? col_qE(A, A.E0, r) : 0.0;
    const double ep0 = qE0 - dG0;
    const double f0_jm1 = shup1(f0[1]);
    auto xl = [&](int face, double e, double lo, double hi) {
        return (face >= 0 && face < nx + 1 && jr_ex) ? A.aSum * (P.dx_inv * ((e > 0.0 ? lo : hi) * e)) : A.aSum * 0.0;
    };
    const double xL = xl(r, ex0, f0[0], f0[1]), xL_1 = xl(r + 1, ex0_1, f0[1], f0[2]);
    const double pL = vFp ? A.aSum * (P.dp_inv * ((ep0 > 0.0 ? f0_jm1 : f0[1]) * ep0)) : A.aSum * 0.0;
    const double pL_u = shdn1(pL);
    double f2 = 0.0;  // ghost cells: zero fill of the walls
    if (r >= 0 && r < nx && jint) {
        f2 = f0[1];
        if (in_r && jr_u) {
            f2 += xL;
            f2 += pL;
        }
        if (in_r && jr_u1) f2 -= pL_u;
        if (in_r1 && jr_u) f2 -= xL_1;
    }
    const double hi = hwmax(f0[1], f2), lo = hwmin(f0[1], f2);

    // ---- RK sums of the earlier stages' fluxes (left to right)
    double Sx = 0.0, Sp = 0.0, Qx = 0.0, Qp = 0.0;
    if (STEP == 5) {
        Sx = vFx ? hx[0] : 0.0;
        Sp = vFp ? hp[0] : 0.0;
    } else if (STEP > 0) {
        Sx = A.a[0] * (vFx ? hx[0] : 0.0);
        Sp = A.a[0] * (vFp ? hp[0] : 0.0);
#pragma unroll
        for (int k = 1; k < NH; k++) {
            Sx = Sx + A.a[k] * (vFx ? hx[k] : 0.0);
            Sp = Sp + A.a[k] * (vFp ? hp[k] : 0.0);
        }
        if (STEP == 4) {
            Qx = A.b5[0] * (vFx ? hx[0] : 0.0);
            Qp = A.b5[0] * (vFp ? hp[0] : 0.0);
#pragma unroll
            for (int k = 1; k < NH; k++) {
                Qx = Qx + A.b5[k] * (vFx ? hx[k] : 0.0);
                Qp = Qp + A.b5[k] * (vFp ? hp[k] : 0.0);
            }
        }
    }
    const double FxD = (STEP == 0 ? A.a[0] * FxH : Sx + A.a[STEP] * FxH) - xL;
    lds_row(lds, nw, 2, w) = FxD;
    lds_row(lds, nw, 3, w) = hi;
    lds_row(lds, nw, 4, w) = lo;
    __syncthreads();

    // ---- column r: FpH_s from the columns beside it (a wavefront at the end of
    // the workgroup reads its own row instead: its value is not used)
    const int wd = w > 0 ? w - 1 : w, wu = w + 1 < nw ? w + 1 : w;
    const double fp_d = lds_row(lds, nw, 0, wd), fp_u = lds_row(lds, nw, 0, wu);
    const double ep_d = lds_row(lds, nw, 1, wd), ep_u = lds_row(lds, nw, 1, wu);
    const double FpH = vFp ? P.dp_inv * (fp * ep + w3 * (fp_u - fp_d) * (ep_u - ep_d)) : 0.0;
    if (STEP < 5) {
        const bool own_x = r >= i0 && (r < i0 + A.TI || last_strip);
        const bool own_c = (r >= i0 || (i0 == 0 && r >= -1)) && (r < i0 + A.TI || last_strip);
        const double hx_out = STEP == 4 ? Qx + A.b5[4] * FxH : FxH;
        const double hp_out = STEP == 4 ? Qp + A.b5[4] * FpH : FpH;
        if (vFx && own_x && own_row_x) __builtin_nontemporal_store(hx_out, elem(P.FxH[STEP], pitch, r, lb));
        if (vFp && own_c && own_row_p) __builtin_nontemporal_store(hp_out, elem(P.FpH[STEP], pitch, r, lb));
    }
    const double FpD = (STEP == 0 ? A.a[0] * FpH : Sp + A.a[STEP] * FpH) - pL;

    // ---- cell r: Zalesak R+-
    const double FxDu = lds_row(lds, nw, 2, wu), FpDu = shdn1(FpD);
    const double hiu = lds_row(lds, nw, 3, wu), hid = lds_row(lds, nw, 3, wd);
    const double lou = lds_row(lds, nw, 4, wu), lod = lds_row(lds, nw, 4, wd);
    const double hju = shdn1(hi), hjd = shup1(hi), lju = shdn1(lo), ljd = shup1(lo);
    double Rp = 0.0, Rm = 0.0;
    if (r >= -1 && r < nx + 1 && jr_ex) {
        const double Pp = hwmax0(FxD) - hwmin0(FxDu) + hwmax0(FpD) - hwmin0(FpDu);
        const double Pm = hwmax0(FxDu) - hwmin0(FxD) + hwmax0(FpDu) - hwmin0(FpD);
        const double wMax = hwmax(hi, hwmax(hiu, hwmax(hid, hwmax(hju, hjd))));
        const double wMin = hwmin(lo, hwmin(lou, hwmin(lod, hwmin(lju, ljd))));
        const double Qm = -wMin + f2;
        const double Qu = wMax - f2;
        if (MP) {
            Rp = Pp > 0.0 ? zalesak_mp(Qu, Pp, A.sinv) : 0.0;
            Rm = Pm > 0.0 ? zalesak_mp(Qm, Pm, A.sinv) : 0.0;
        } else {
            Rp = Pp > 0.0 ? 1.0 : 0.0;
            Rm = Pm > 0.0 ? 1.0 : 0.0;
            if (__builtin_amdgcn_ballot_w64(!(Qu - Pp >= 0.0) || !(Qm - Pm >= 0.0)) != 0) {
                if (Pp > 0.0) Rp = fmin(1.0, Qu / Pp);
                if (Pm > 0.0) Rm = fmin(1.0, Qm / Pm);
            }
        }
    }
    lds_row(lds, nw, 5, w) = Rp;
    lds_row(lds, nw, 6, w) = Rm;
    __syncthreads();

    // ---- limiter C on the faces of cell r and the corrected value
    if (r < i0 || r >= i1) return;  // uniform; no barrier follows
    const double Rp_d = lds_row(lds, nw, 5, wd), Rm_d = lds_row(lds, nw, 6, wd);
    const double Rp_u = lds_row(lds, nw, 5, wu), Rm_u = lds_row(lds, nw, 6, wu);
    const double Rpl = shup1(Rp), Rml = shup1(Rm);  // R at (r, j-1)
    const bool lim = r >= 1 && r < nx && jint, lim_u = r + 1 >= 1 && r + 1 < nx && jint;
    const double cx = lim ? (FxD > 0.0 ? hwmin(Rp, Rm_d) : hwmin(Rp_d, Rm)) : 1.0;
    const double cxu = lim_u ? (FxDu > 0.0 ? hwmin(Rp_u, Rm) : hwmin(Rp, Rm_u)) : 1.0;
    const double cp = lim ? (FpD > 0.0 ? hwmin(Rp, Rml) : hwmin(Rpl, Rm)) : 1.0;
    const double lx = cx * FxD, lxu = cxu * FxDu, lp = cp * FpD;
    const double lpu = shdn1(lp);
    if (out_lane) {
        double t = f2;
        if (in_r && jr_u) {
            t += lx;
            t += lp;
        }
        if (in_r && jr_u1) t -= lpu;
        if (in_r1 && jr_u) t -= lxu;
        *elem(A.fout, pitch, r, lb) = t;
    }
}

template <int STEP, bool MP>
__global__ __launch_bounds__(1024) void k_stage_rows(StageArgs A) {
    extern __shared__ double lds[];
    stage_rows<STEP, MP>(A, xcd_tile(), lds);
}

// Several patches (of independent runs) at the same RK stage in one launch:
// workgroups [wg_start[k], wg_start[k+1]) of the XCD-ordered tile sequence
// belong to item k; the item's arguments come through the scalar cache.  Strips
// (k_stage_batch) or one wavefront per row (k_stage_rows_batch), one form for
// the launch (batch_form).
__device__ __forceinline__ int batch_item(const int *wg_start, int n, int tile) {
    int lo = 0, hi = n - 1;  // the last k with wg_start[k] <= tile (uniform)
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (wg_start[mid] <= tile) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}
template <int STEP, bool MP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_stage_batch(const StageArgs *items, const int *wg_start, int n) {
    const int tile = xcd_tile(), k = batch_item(wg_start, n, tile);
    const StageArgs A = ld_uniform_struct(items + k);
    stage_tile<STEP, MP>(A, tile - wg_start[k]);
}
template <int STEP, bool MP>
__global__ __launch_bounds__(1024) void k_stage_rows_batch(const StageArgs *items, const int *wg_start, int n) {
    extern __shared__ double lds[];
    const int tile = xcd_tile(), k = batch_item(wg_start, n, tile);
    const StageArgs A = ld_uniform_struct(items + k);
    stage_rows<STEP, MP>(A, tile - wg_start[k], lds);
}

template <bool MP>
void launch_stage_t(vx_ctx *ctx, const StageArgs &A) {
    const int strips_wg = A.form == 2 ? 1 : 4, waves = A.form == 2 ? A.TI + 4 : 4;
    const dim3 grid((unsigned)(A.nbx * ((A.nstrip + strips_wg - 1) / strips_wg))), block(64 * waves);
    const size_t lds = sizeof(double) * 64 * RT_ARRAYS * waves;
#define VX_STAGE(S)                                                        \
    if (A.form == 2) k_stage_rows<S, MP><<<grid, block, lds, ctx->stream>>>(A);  \
    else if (A.form == 1) k_stage_w4<S, MP><<<grid, block, 0, ctx->stream>>>(A); \
    else k_stage<S, MP><<<grid, block, 0, ctx->stream>>>(A);
    switch (A.step) {
        case 0: VX_STAGE(0) break;
        case 1: VX_STAGE(1) break;
        case 2: VX_STAGE(2) break;
        case 3: VX_STAGE(3) break;
        case 4: VX_STAGE(4) break;
        default: VX_STAGE(5) break;
    }
#undef VX_STAGE
}

void launch_stage(vx_ctx *ctx, StageArgs &A, bool mp) {
    A.nstrip = (A.p.n_x + A.TI - 1) / A.TI;
    if (mp) launch_stage_t<true>(ctx, A);
    else launch_stage_t<false>(ctx, A);
}

// Rows per strip (the tile height) of a patch shape and RK stage (the later
// stages hold more registers and read more planes).  A strip costs its rows
// plus 6 pipeline warm-up rows, and a wavefront walks them one after another,
// so small patches want short strips (more wavefronts) and large ones long
// strips (less warm-up).  The first call for a shape times the candidates on
// the call's own launch, which is idempotent (it reads f_s, f^n and the fluxes
// of earlier stages and writes only f_(s+1) and this stage's fluxes, the same
// values for every strip height), and keeps the fastest (a shorter strip must
// beat the taller ones by more than 3 %).  While a step graph
// is being recorded the choice falls back to the shortest strip that still
// gives 2048 wavefronts.
//
// A choice is kept as rows, rows + W4_FORM for the four-wave form (k_stage_w4)
// and rows + 2 W4_FORM for the row form (k_stage_rows), which is timed
// where a SIMD gets at most ROWS_PER_SIMD rows of the patch: it redoes 4 rows
// in 12, strips that fill the device about 6 in 50.  Measured, all stages of
// 1024 x 1024 (18 rows a SIMD): 31 to 45 us as rows, 54 to 64 as strips before
// this form; 2048 x 1024 mixed (36 rows): 49 to 59 us as rows, 45 to 60 as strips.
// The choices are kept per device for the whole process (every context on the
// device shares them: a serving loop's runs of one shape time it once).
struct TileKey {
    int device, nx, np, mp, step;
    bool operator<(const TileKey &o) const {
        return std::tie(device, nx, np, mp, step) < std::tie(o.device, o.nx, o.np, o.mp, o.step);
    }
};
constexpr int W4_FORM = 4096, ROWS_MAX = 12, ROWS_PER_SIMD = 64;
std::mutex g_tile_mu;
std::map<TileKey, int> g_tiles;

int tile_lookup(int device, int nx, int np, int mp, int step) {
    std::lock_guard<std::mutex> g(g_tile_mu);
    auto it = g_tiles.find(TileKey{device, nx, np, mp, step});
    return it == g_tiles.end() ? 0 : it->second;
}

void tile_store(vx_ctx *ctx, int nx, int np, int ti, int mp, int step) {
    ctx->ti_cache.push_back({nx, np, ti, mp, step});
    std::lock_guard<std::mutex> g(g_tile_mu);
    g_tiles[TileKey{ctx->device, nx, np, mp, step}] = ti;
}

// Workgroups of k_stage<step, mp> resident per compute unit (0 if unknown).
int stage_blocks_per_cu(int step, bool mp) {
    int n = 0;
    hipError_t e = hipSuccess;
#define VX_OCC(S, M) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_stage<S, M>, 256, 0)
    if (mp) {
        switch (step) {
            case 0: VX_OCC(0, true); break;
            case 1: VX_OCC(1, true); break;
            case 2: VX_OCC(2, true); break;
            case 3: VX_OCC(3, true); break;
            case 4: VX_OCC(4, true); break;
            default: VX_OCC(5, true); break;
        }
    } else {
        switch (step) {
            case 0: VX_OCC(0, false); break;
            case 1: VX_OCC(1, false); break;
            case 2: VX_OCC(2, false); break;
            case 3: VX_OCC(3, false); break;
            case 4: VX_OCC(4, false); break;
            default: VX_OCC(5, false); break;
        }
    }
#undef VX_OCC
    return e == hipSuccess ? n : 0;
}

// VX_TILE_ROWS pins the choice of every launch, shared ones among them (one value,
// or six comma-separated values, one per RK stage; rows + 4096 for the four-wave
// form, + 8192 for the row form), e.g. to profile the configuration a timed run
// chose.  The value of a stage, 0 without one.
int pinned_tile(int step) {
    const char *env = std::getenv("VX_TILE_ROWS");
    if (!env) return 0;
    int v[6], n = 0;
    for (const char *q = env; *q && n < 6;) {
        v[n++] = std::atoi(q);
        while (*q && *q != ',') q++;
        if (*q == ',') q++;
    }
    const int ti = n == 6 ? v[step] : (n >= 1 ? v[0] : 0);
    const bool ok = (ti >= 1 && ti <= 1024) || (ti > W4_FORM && ti <= W4_FORM + 1024) ||
                    (ti > 2 * W4_FORM && ti <= 2 * W4_FORM + ROWS_MAX);
    return ok ? ti : 0;
}

int tile_rows(vx_ctx *ctx, const StageArgs &A0, bool mp) {
    const int nx = A0.p.n_x, np = A0.p.n_p;
    for (auto &c : ctx->ti_cache)
        if (c[0] == nx && c[1] == np && c[3] == (int)mp && c[4] == A0.step) return c[2];
    static const int cand[] = {64, 32, 16, 8, 4, 2};
    if (const int pin = pinned_tile(A0.step)) {
        ctx->ti_cache.push_back({nx, np, pin, (int)mp, A0.step});  // this context only
        return pin;
    }
    if (const int known = tile_lookup(ctx->device, nx, np, (int)mp, A0.step)) {
        ctx->ti_cache.push_back({nx, np, known, (int)mp, A0.step});
        return known;
    }
    int guess = 2;
    for (int ti : cand)
        if ((long)A0.nbx * ((nx + ti - 1) / ti) >= 2048) {
            guess = ti;
            break;
        }
    if (ctx->capturing) return guess;
    // Besides the powers of two, the strip heights at which the launch's
    // workgroups just fill k rounds of the device's resident slots (k = 1..4):
    // the tallest strips (least warm-up) without a part-empty last round.
    std::vector<int> cands(std::begin(cand), std::end(cand));
    const int slots = ctx->n_cu * stage_blocks_per_cu(A0.step, mp);
    if (slots > 0)
        for (int k = 1; k <= 4; k++) {
            const long wg_max = (long)k * slots;
            // smallest strip height whose ceil(strips / 4) * nbx workgroups fit in wg_max
            for (int ti = 1; ti <= 1024 && ti <= nx; ti++) {
                const long strips = (nx + ti - 1) / ti;
                if ((long)A0.nbx * ((strips + 3) / 4) <= wg_max) {
                    if (ti > 2) cands.push_back(ti);
                    break;
                }
            }
        }
    std::sort(cands.begin(), cands.end(), std::greater<int>());
    cands.erase(std::unique(cands.begin(), cands.end()), cands.end());
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int best = guess;
    if (hipEventCreate(&e0) == hipSuccess && hipEventCreate(&e1) == hipSuccess) {
        bool failed = false;
        // one launch of (strip height, form) timed on its own
        auto timed = [&](int code) {
            StageArgs A = A0;
            A.TI = code % W4_FORM;
            A.form = code / W4_FORM;
            float t = 1e30f;
            if (hipEventRecord(e0, ctx->stream) != hipSuccess) failed = true;
            if (!failed) launch_stage(ctx, A, mp);
            if (!failed && (hipEventRecord(e1, ctx->stream) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
                            hipEventElapsedTime(&t, e0, e1) != hipSuccess))
                failed = true;
            return t;
        };
        // Candidates run from tall to short strips, the three-wave form first.
        // One warm-up launch, then one timed launch of each candidate; the
        // three fastest are timed twice more and keep their fastest launch
        // (the minimum is steadier than a sum against the device's noise).
        // Among those, in candidate order, a later one must be more than 3 %
        // faster to win (ties go to fewer warm-up rows and the three-wave form).
        std::vector<std::pair<int, float>> res;  // (code, ms) in candidate order
        {
            StageArgs A = A0;
            A.TI = guess;
            A.form = 0;
            launch_stage(ctx, A, mp);  // warm
        }
        // The four-wave form is timed at stage 0, which nearly fits its 128
        // VGPRs (4096 x 4096: 272 us against 261); the later stages spill there
        // (354 against 291 us at stage 1, 2.4 times as long at stage 3).  Strips
        // under 8 rows lose to the row form wherever the launch is small enough
        // to want them (601 x 333: 21 to 25 us against 10 to 13).
        std::vector<int> codes;
        for (int ti : cands) {
            if (ti < 8 || (ti > 8 && ti >= 2 * nx)) continue;  // a single strip either way
            codes.push_back(ti);
            if (A0.step == 0) codes.push_back(ti + W4_FORM);
        }
        if ((long)A0.nbx * nx <= (long)ROWS_PER_SIMD * 4 * ctx->n_cu)
            for (int ti : {12, 8, 4}) codes.push_back(ti + 2 * W4_FORM);
        for (int code : codes) {
            const float t = timed(code);
            if (failed) break;
            res.push_back({code, t});
        }
        if (!failed && !res.empty()) {
            std::vector<int> order(res.size());
            for (size_t k = 0; k < res.size(); k++) order[k] = (int)k;
            std::sort(order.begin(), order.end(), [&](int a, int b) { return res[a].second < res[b].second; });
            const size_t nfin = std::min<size_t>(3, order.size());
            std::vector<int> fin(order.begin(), order.begin() + nfin);
            for (int k : fin)
                for (int rep = 0; rep < 2 && !failed; rep++) res[k].second = std::min(res[k].second, timed(res[k].first));
            if (!failed) {
                std::sort(fin.begin(), fin.end());  // candidate order
                float best_ms = 1e30f;
                for (int k : fin)
                    if (res[k].second < 0.97f * best_ms) {
                        best_ms = res[k].second;
                        best = res[k].first;
                    }
            }
        }
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    tile_store(ctx, nx, np, best, (int)mp, A0.step);
    return best;
}

}  // namespace

extern "C" {

int vx_fct_stage_fused_available(void) { return 1; }

}  // extern "C"

// Checks and kernel arguments of one patch's fused stage.
static int stage_args(vx_ctx *ctx, const vx_patch *p, int step, double dt, const vx_fields *fl,
                      const double *fin, double *fout, bool mp, double f_scale, bool choose, StageArgs &A) {
    int rc = validate_patch(ctx, p);
    if (rc) return rc;
    if (step < 0 || step > 5 || !fl || !fl->E0 || !fl->a20)
        return fail(ctx, VX_EINVAL, "stage_fused: bad step %d or missing stage-0 fields", step);
    if ((rc = validate_span(ctx, p, fl->n_f))) return rc;
    if (!(p->left && p->right && p->down && p->up))
        return fail(ctx, VX_EINVAL, "stage_fused: patch must touch all four domain edges");
    if (fin == p->f[0] && step != 0)
        return fail(ctx, VX_EINVAL, "stage_fused: input aliases f^n after stage 0");
    if (fout == fin || fout == p->f[0])
        return fail(ctx, VX_EINVAL, "stage_fused: output must not alias the inputs");
    A.p = *p;
    A.fin = fin;
    A.fout = fout;
    A.E = fl->E;
    A.a2 = fl->a2;
    A.E0 = fl->E0;
    A.a20 = fl->a20;
    A.n_f = fl->n_f;
    A.step = step;
    A.ns = step + 1;
    for (int k = 0; k < 6; k++) A.a[k] = 0.0;
    for (int k = 0; k < A.ns; k++) A.a[k] = vx::rk_a[step][k] * dt;
    for (int k = 0; k < 6; k++) A.b5[k] = vx::rk_a[5][k] * dt;  // as stage 5 forms its a[k]
    A.aSum = A.a[0];
    for (int k = 1; k < A.ns; k++) A.aSum = A.aSum + A.a[k];
    A.nbx = (p->n_p + OUTW - 1) / OUTW;
    A.sinv = 1.0;
    A.eps32 = 0.0f;
    A.inv_rtb = 1.0 / (double)p->rtb;
    if (mp) {
        if (!(f_scale > 0.0) || !std::isfinite(f_scale))
            return fail(ctx, VX_EINVAL, "stage_fused_mp: f scale must be positive and finite");
        A.sinv = std::ldexp(1.0, -std::ilogb(f_scale));
        A.eps32 = (float)(1.0e-10 * A.sinv * A.sinv);
    }
    A.form = 0;
    A.TI = 0;
    if (!choose) return VX_OK;  // (batch_launch chooses for all of its items)
    const int choice = tile_rows(ctx, A, mp);
    A.TI = choice % W4_FORM;
    A.form = choice / W4_FORM;
    A.nstrip = (p->n_x + A.TI - 1) / A.TI;
    return VX_OK;
}

static int stage_fused(vx_ctx *ctx, const vx_patch *p, int step, double dt, const vx_fields *fl,
                       const double *fin, double *fout, bool mp, double f_scale) {
    StageArgs A;
    int rc = stage_args(ctx, p, step, dt, fl, fin, fout, mp, f_scale, true, A);
    if (rc) return rc;
    LaunchTimer lt(ctx, "k_stage");
    launch_stage(ctx, A, mp);
    return check_launch(ctx, "k_stage");
}

// Staging of batched launch arguments: device slots with pinned host mirrors;
// a slot is rewritten only after the copy that last used it has completed.
constexpr int BATCH_MAX = 64, BATCH_SLOTS = 8;
constexpr size_t BATCH_SLOT_BYTES = sizeof(StageArgs) * BATCH_MAX + sizeof(int) * (BATCH_MAX + 1) + 256;

struct BatchRing {
    char *dev = nullptr, *host = nullptr;
    hipEvent_t ev[BATCH_SLOTS] = {};
    bool pending[BATCH_SLOTS] = {};
    int next = 0;
};

static void batch_ring_free(void *r) {
    BatchRing *b = (BatchRing *)r;
    for (auto &e : b->ev)
        if (e) (void)hipEventDestroy(e);
    if (b->dev) (void)hipFree(b->dev);
    if (b->host) (void)hipHostFree(b->host);
    delete b;
}

// Strip height and kernel form of a batched launch, one for all items and by
// the launch's total size, so that no shape is timed on the serving path (an
// item alone would want short strips, which redo their warm-up rows in a
// launch that fills the device anyway).  Up to BATCH_ROWS rows a SIMD: the row
// form (measured, stages 0..5: twelve FP64 patches of 49 rows a SIMD 84 to 120
// us as strips, 96 to 122 as rows; four mixed ones of 24 rows 38 to 55 as
// strips, 34 to 61 as rows; a 1024 x 1024 patch of 18 rows 39 to 60 as strips,
// 31 to 45 as rows); above: the strip height of the least rounds x (rows + 6), a round being
// the resident wavefronts (three a SIMD) walking a strip each.  VX_TILE_ROWS pins it
// (strips have one form here, held to three waves per SIMD).
constexpr int BATCH_ROWS = 20;
static void batch_form(vx_ctx *ctx, std::vector<StageArgs> &A, int step, bool mp) {
    const double simds = 4.0 * ctx->n_cu;
    auto waves = [&](int ti) {
        double w = 0;
        for (const StageArgs &a : A) w += (double)a.nbx * ((a.p.n_x + ti - 1) / ti);
        return w;
    };
    int form = 2, ti = ROWS_MAX;
    if (const int pin = pinned_tile(step)) {
        form = pin / W4_FORM == 2 ? 2 : 0;
        ti = pin % W4_FORM;
    } else if (waves(1) > BATCH_ROWS * simds) {
        form = 0;
        double best = 1e300;
        for (int t = 96; t >= 8; t -= 4) {
            const double cost = std::max(1.0, waves(t) / (3 * simds)) * (t + 2 * HALO);
            if (cost < 0.99 * best) {
                best = cost;
                ti = t;
            }
        }
    }
    for (StageArgs &a : A) {
        a.form = form;
        a.TI = ti;
        a.nstrip = (a.p.n_x + ti - 1) / ti;
    }
    ctx->batch_tile[mp][step] = form * W4_FORM + ti;
}

static int batch_launch(vx_ctx *ctx, std::vector<StageArgs> &A, int step, bool mp) {
    if (A.empty()) return VX_OK;
    if (ctx->capturing) return fail(ctx, VX_EINVAL, "stage batch while a step graph is recorded");
    batch_form(ctx, A, step, mp);
    const bool rows = A[0].form == 2;
    if (!ctx->batch_ring) {
        BatchRing *b = new BatchRing;
        ctx->batch_ring = b;
        ctx->batch_ring_free = batch_ring_free;
        int rc = check_hip(ctx, hipMalloc((void **)&b->dev, BATCH_SLOT_BYTES * BATCH_SLOTS), "batch args");
        if (!rc) rc = check_hip(ctx, hipHostMalloc((void **)&b->host, BATCH_SLOT_BYTES * BATCH_SLOTS), "batch staging");
        for (auto &e : b->ev)
            if (!rc) rc = check_hip(ctx, hipEventCreateWithFlags(&e, hipEventDisableTiming), "batch event");
        if (rc) return rc;
    }
    BatchRing *b = (BatchRing *)ctx->batch_ring;
    const int k = b->next;
    b->next = (k + 1) % BATCH_SLOTS;
    if (b->pending[k]) {
        int rc = check_hip(ctx, hipEventSynchronize(b->ev[k]), "batch slot wait");
        if (rc) return rc;
    }
    const int n = (int)A.size();
    char *h = b->host + BATCH_SLOT_BYTES * k, *d = b->dev + BATCH_SLOT_BYTES * k;
    std::memcpy(h, A.data(), sizeof(StageArgs) * n);
    int *start = (int *)(h + sizeof(StageArgs) * BATCH_MAX);
    int total = 0;
    for (int q = 0; q < n; q++) {
        start[q] = total;
        total += A[q].nbx * (rows ? A[q].nstrip : (A[q].nstrip + 3) / 4);
    }
    start[n] = total;
    int rc = check_hip(ctx, hipMemcpyAsync(d, h, BATCH_SLOT_BYTES, hipMemcpyHostToDevice, ctx->stream), "batch upload");
    if (rc) return rc;
    rc = check_hip(ctx, hipEventRecord(b->ev[k], ctx->stream), "batch event record");
    b->pending[k] = rc == VX_OK;
    if (rc) return rc;
    const StageArgs *dA = (const StageArgs *)d;
    const int *dS = (const int *)(d + sizeof(StageArgs) * BATCH_MAX);
    const int wf = rows ? A[0].TI + 4 : 4;
    const size_t lds = rows ? sizeof(double) * 64 * RT_ARRAYS * wf : 0;
    dim3 grid((unsigned)total), block(64 * wf);
#define VX_BATCH(S)                                                                                   \
    if (mp && rows) k_stage_rows_batch<S, true><<<grid, block, lds, ctx->stream>>>(dA, dS, n);       \
    else if (rows) k_stage_rows_batch<S, false><<<grid, block, lds, ctx->stream>>>(dA, dS, n);       \
    else if (mp) k_stage_batch<S, true><<<grid, block, 0, ctx->stream>>>(dA, dS, n);                 \
    else k_stage_batch<S, false><<<grid, block, 0, ctx->stream>>>(dA, dS, n);
    switch (step) {
        case 0: VX_BATCH(0) break;
        case 1: VX_BATCH(1) break;
        case 2: VX_BATCH(2) break;
        case 3: VX_BATCH(3) break;
        case 4: VX_BATCH(4) break;
        default: VX_BATCH(5) break;
    }
#undef VX_BATCH
    return check_launch(ctx, "k_stage_batch");
}

extern "C" {

int vx_fct_stage_fused(vx_ctx *ctx, const vx_patch *p, int step, double dt, const vx_fields *fl,
                       const double *fin, double *fout) {
    return stage_fused(ctx, p, step, dt, fl, fin, fout, false, 0.0);
}

int vx_fct_stage_fused_mp(vx_ctx *ctx, const vx_patch *p, int step, double dt, const vx_fields *fl,
                          const double *fin, double *fout, double f_scale) {
    return stage_fused(ctx, p, step, dt, fl, fin, fout, true, f_scale);
}

int vx_fct_stage_fused_batch(vx_ctx *ctx, const vx_stage_item *items, int n, int step) {
    if (n < 0 || n > BATCH_MAX || (n > 0 && !items))
        return fail(ctx, VX_EINVAL, "stage batch: %d items (at most %d)", n, BATCH_MAX);
    std::vector<StageArgs> fp64, mixed;
    for (int q = 0; q < n; q++) {
        const vx_stage_item &it = items[q];
        StageArgs A;
        const bool mp = it.f_scale > 0.0;
        int rc = stage_args(ctx, &it.p, step, it.dt, &it.fl, it.fin, it.fout, mp, it.f_scale, false, A);
        if (rc) return rc;
        (mp ? mixed : fp64).push_back(A);
    }
    LaunchTimer lt(ctx, "k_stage");
    int rc = batch_launch(ctx, fp64, step, false);
    return rc ? rc : batch_launch(ctx, mixed, step, true);
}

static int tile_choice(vx_ctx *ctx, int32_t n_x, int32_t n_p, int step, int mixed) {
    for (auto &c : ctx->ti_cache)
        if (c[0] == n_x && c[1] == n_p && c[3] == (mixed ? 1 : 0) && c[4] == step) return c[2];
    return tile_lookup(ctx->device, n_x, n_p, mixed ? 1 : 0, step);
}

int vx_stage_tile_rows(vx_ctx *ctx, int32_t n_x, int32_t n_p, int step, int mixed) {
    return tile_choice(ctx, n_x, n_p, step, mixed) % W4_FORM;
}

int vx_stage_tile_waves(vx_ctx *ctx, int32_t n_x, int32_t n_p, int step, int mixed) {
    const int c = tile_choice(ctx, n_x, n_p, step, mixed);
    return c == 0 ? 0 : (c >= W4_FORM ? 4 : 3);
}

int vx_stage_tile_code(vx_ctx *ctx, int32_t n_x, int32_t n_p, int step, int mixed) {
    if (n_x == 0 && n_p == 0) return step >= 0 && step <= 5 ? ctx->batch_tile[mixed ? 1 : 0][step] : 0;
    return tile_choice(ctx, n_x, n_p, step, mixed);
}

}  // extern "C"
