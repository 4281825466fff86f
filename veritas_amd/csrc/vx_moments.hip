// p-moments: charge and current density (Rectangle::CalculateRhoAndJ,
// Rectangle.cpp:157-282) and their assembly on the finest grid
// (Level.cpp:19-62, Mesh.cpp:52-56, EMSolver.cpp:104-122).
//
// The reference sums over p sequentially (j = 0, 1, ..., n_p-1) for each x
// column and each finest sub-cell k.  To reproduce those bits one wavefront
// forms a column's summands, 64 consecutive p-cells in parallel (interpolants,
// gamma factors, logarithms), and another adds them in order from LDS, one lane
// per accumulation chain.
#include <algorithm>
#include <cstring>
#include <type_traits>
#include <vector>

#include "vx_dev.h"
#include "vx_internal.h"
#include "vx_math.h"

using namespace vxi;
using namespace vxd;

namespace {

constexpr int MAX_RTB = 4;  // coarsest level of a 3-level hierarchy at ratio 2
constexpr long TAB_CELLS = 1 << 20;  // a patch of more cells gets a logarithm table (and a tall one)
constexpr long BATCH_CELLS = 1 << 21;  // a patch of more cells has a launch (and a table) of its own
constexpr int TAB_KEY = 8;  // A^2, pmin, dp, p_pos, mc2inv, c1, c2, n_p

// Rectangle.cpp:76-89
__constant__ double kInterp[12] = {
    0.104166666666667, -0.708333333333334, 0.708333333333334, -0.104166666666667,
    0.117647058823529, 0.029411764705882,  0.029411764705882, 0.117647058823529,
    -0.083333333333333, 0.166666666666667, -0.166666666666667, 0.083333333333334};

// What the moments of one patch need
struct MomPatch {
    const double *f;
    const uint8_t *nested;
    double *chargeR, *currentR;
    int n_x, n_p, x_pos, p_pos, rtb, pitch;
    double dx, dp, pmin, q, mc2inv;
    double c1, c2, c3;    // m_inv*c_inv, 1/c1, 1/48
    double inv_rtb;       // 1.0 / relativeToBottom
    double dpq, jscale;   // dp*q and -q*q/mass
    double rel[3 * MAX_RTB];  // interpolatCoefsREL (Rectangle.cpp:103-110)
    // A patch that is the whole assembly by itself: the places of the assembled
    // charge, current and species' charge (null otherwise), each 0.0 + the patch's
    // (the assembly's sum, which makes -0.0 +0.0)
    double *charge, *J, *species;
};

struct MomArgs {
    MomPatch p;
    vx_fields fl;
    // Two tables of logarithm terms, each for one value a0 of A^2: table 0 for
    // the patch's first sub-column (every column when A^2 is uniform), table 1
    // for A^2 = 0 (the plasma ahead of a laser pulse).  Table q's entries t in
    // [0, n_p+2) (tab_entries) hold c2 log(h(t)/h(t-1)) with h(j) = Gamma(p_j, a0)
    // + c1 p_j; its head, at tab + q TAB_HEAD wherever the entries lie (so that a
    // table of another n_p is never taken for this one), holds what they were
    // formed from (a0 first, then the p grid and the constants) and at TAB_KEY 1
    // once built, so an unchanged table is not rebuilt.  A wavefront whose chains
    // all have A^2 == a0 of a table reads it (the same bits it would form itself);
    // the others form their logarithms per distinct A^2.
    const double *tab;
};

// Several patches in one launch: patch k's workgroups start at start[k].
constexpr int MOM_BATCH = 12;  // 3 KB of kernel arguments
struct MomBatch {
    vx_fields fl;
    int n, start[MOM_BATCH + 1];
    MomPatch p[MOM_BATCH];
};

// EMFieldSolver::GetCellAverageASquared (EMSolver.hpp:57-64)
__device__ __forceinline__ double cell_a2(const vx_fields &fl, long i) {
    i += fl.n_prepad;
    i = i > -1 ? i : 0;
    i = i < fl.n_e ? i : (fl.n_e - 1);
    double ay = fl.Ay1[i], az = fl.Az1[i];
    return (ay * ay) + (az * az);
}


constexpr int TAB_HEAD = 16;
__host__ __device__ inline long tab_entries(int q, int n_p) { return 2 * TAB_HEAD + q * ((long)n_p + 3); }

// Logarithm tables of one patch (see MomArgs::tab); workgroup q builds table q.
template <int RTB>
__global__ __launch_bounds__(1024) void k_moment_table(MomArgs A, double *tab) {
    const MomPatch &P = A.p;
    const int t = threadIdx.x;
    const double a0 = blockIdx.x == 0 ? P.q * P.q * cell_a2(A.fl, (long)P.x_pos * RTB) : 0.0;
    const double key[TAB_KEY] = {a0, P.pmin, P.dp, (double)P.p_pos, P.mc2inv, P.c1, P.c2, (double)P.n_p};
    double *kt = tab + blockIdx.x * TAB_HEAD, *entry = tab + tab_entries((int)blockIdx.x, P.n_p);
    bool hit = kt[TAB_KEY] == 1.0;
    for (int k = 0; k < TAB_KEY; k++) hit = hit && kt[k] == key[k];
    if (__syncthreads_or(hit ? 1 : 0) != 0) return;  // the same table is in place
    // (every thread read the same bits; the barrier also orders those reads
    // before the writes below)
    auto h = [&](int j) {
        double pm = momentum(P.pmin, P.dp, j, P.p_pos);
        return gamma_(pm, a0, P.mc2inv) + P.c1 * pm;
    };
    for (int e = t; e < P.n_p + 2; e += blockDim.x) entry[e] = P.c2 * vx_log(h(e) / h(e - 1));
    if (t < TAB_KEY) kt[t] = key[t];
    if (t == 0) kt[TAB_KEY] = 1.0;
}

// Compensated wavefront sum of the lanes' (value, error) pairs (mixed-precision
// form, where the reference's p order is not kept): a butterfly of error-free
// additions (TwoSum); every lane ends with the same sum s and error e.
__device__ __forceinline__ void wave_two_sum(double v, double ve, double &s, double &e) {
    s = v;
    e = ve;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const double so = __shfl_xor(s, off, 64), eo = __shfl_xor(e, off, 64);
        const double t = s + so, z = t - s;
        const double err = (s - (t - z)) + (so - z);
        e = (e + eo) + err;
        s = t;
    }
}

// (acc, cmp) += v with an error-free addition
__device__ __forceinline__ void add_two(double &acc, double &cmp, double v) {
    const double t = acc + v, z = t - acc;
    const double err = (acc - (t - z)) + (v - z);
    cmp = cmp + err;
    acc = t;
}

// A workgroup owns WCOL consecutive x-columns.  Producer wavefront c forms the
// summands of column c's RTB sub-columns (the reference's accumulation chains)
// for one 64-cell p-chunk at a time and puts them in LDS; the consumer
// wavefront adds each chunk in p order while the producers form the next, lane
// n the charge of chain n and lane 32 + n its current, all 2 WCOL RTB chains in
// lockstep.  A workgroup barrier per chunk hands the buffers over.  Skipped
// cells (nested, or past n_p) contribute -0.0, which is an exact identity for
// addition, so every chain performs the reference's additions in its order.
//
// A chunk's sub-cell values and logarithms are formed once, by the lane of their
// p-cell; those of p + 1 and p + 2 come from the next lanes by DPP rotations with
// the next chunk's first two lanes, so each iteration forms the next chunk's
// values.  The loads of the next WDEPTH chunks are in flight.
//
// Bound by the producers' VALU issue where the launch fills the device (at RTB
// 4 about 190 instructions per chunk; without a table each distinct A^2 adds a
// square root, two divisions and a logarithm, about 430 cycles), else by the
// consumer's dependent additions, about 0.3 us per chunk.  With 4 columns a
// workgroup's five wavefronts spread over a CU's SIMDs and small launches over
// more CUs.  Measured on an MI355X, us with the table's launch, 2 / 4 / 8
// columns: 8190 x 1024 at RTB 1 with a pulse 52.9 / 46.5 / 53.5 and without 46.9
// / 30.6 / 28.6, 8192 x 512 at RTB 4 39.3 / 42.1 / 40.3, 1000 x 500 at RTB 1 10.9
// / 9.8 / 11.4, 500 x 512 at RTB 4 with a pulse 20.5 / 20.9 / 27.1.  One
// wavefront per 4 sub-columns that adds its own chunk took 64.9, 35.4, 66.9, 27.1
// and 30.0; two of them, a producer and a consumer, 92.3, 34.8, 80.4, 22.4, 27.5.
constexpr int MCOL = 4, MCOL_TALL = 8;

// Whole-wavefront rotation by one lane (DPP wave_rol:1): lane l receives the
// value of lane (l + 1) mod 64.
__device__ __forceinline__ double rol1(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x134, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x134, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// Entries l + 1 and l + 2 (lane l's view) of the sequence cur[0..63],
// nxt[0], nxt[1] (this chunk's values, then the next chunk's first two).
__device__ __forceinline__ void next2_rot(int lane, double cur, double nxt, double &n1, double &n2) {
    n1 = rol1(lane == 0 ? nxt : cur);
    n2 = rol1(rol1(lane < 2 ? nxt : cur));
}

// vx_log(a / b) for the ratio of neighbouring h (close to 1): where every lane's
// ratio lies in (sqrt(1/2), sqrt(2)), vx_log's exponent is 0 and its mantissa the
// ratio, and the terms with the exponent add +0; both divisions then stay in the
// short form's range (a ratio formed outside it is not in that interval).
__device__ __forceinline__ double log_ratio(double a, double b) {
    const double x = div_refined(a, b, rcp_refined(b));
    if (__builtin_amdgcn_ballot_w64(!(x > 0.70710678118654757 && x <= 1.4142135623730951)) != 0) return vx_log(a / b);
    const double f = x - 1.0, d = 2.0 + f;
    const double s = div_refined(f, d, rcp_refined(d));
    const double z = s * s;
    const double R = vx_log_r(z);
    const double hfsq = 0.5 * f * f;
    return f - (hfsq - s * (hfsq + R));
}

__device__ __forceinline__ void put_charge(const MomPatch &P, long e, double v) {
    P.chargeR[e] = v;
    if (P.charge) P.charge[e] = P.species[e] = 0.0 + v;
}
__device__ __forceinline__ void put_current(const MomPatch &P, long e, double v) {
    P.currentR[e] = v;
    if (P.charge) P.J[e] = 0.0 + v;
}

// COMP (mixed-precision form): no consumer; each producer keeps its lanes'
// compensated (TwoSum) sums over the chunks and ends with one compensated
// reduction across its lanes.
// NEST: the patch has nested cells (their summands are -0.0).
// tabs: the patch's logarithm tables, or null; blk: the workgroup's number in
// the patch; lds: 2 x 2 x WCOL RTB rows of 65 (not used by COMP).
template <int RTB, int WCOL, bool COMP, bool NEST>
__device__ __forceinline__ void moments_columns(const MomPatch &P, const vx_fields &fl, const double *tabs, int blk,
                                                double *lds) {
    constexpr int NR = RTB == 1 ? 1 : 5;  // rows of f that a column's values read
    constexpr int WDEPTH = RTB == 1 ? 4 : 2;
    constexpr int NCH = WCOL * RTB;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63);
    const int i0 = blk * WCOL;
    // buffer, charge/current, chain, p-cell of the chunk (rows of 65: the
    // consumer's lanes read one row each, in different LDS banks)
    double(*T)[2][NCH][65] = reinterpret_cast<double(*)[2][NCH][65]>(lds);
    const int nchunk = (P.n_p + 63) / 64;
    if (wave < WCOL) {
        const int i = i0 + wave;
        const bool col_ok = i < P.n_x;
        const int ic = col_ok ? i : P.n_x - 1;
        // the sub-columns' A^2 and a logarithm table built for them, if there is one
        double asq[RTB];
#pragma unroll
        for (int s = 0; s < RTB; s++) asq[s] = P.q * P.q * cell_a2(fl, (long)(ic + P.x_pos) * RTB + s);
        const double *tab = nullptr;
        for (int q = 1; q >= 0 && tabs && !tab; q--) {
            const double *kt = tabs + q * TAB_HEAD;
            bool all = kt[TAB_KEY] != 0.0;
#pragma unroll
            for (int s = 0; s < RTB; s++) all = all && asq[s] == kt[0];
            if (all) tab = tabs + tab_entries(q, P.n_p);
        }
        // Chunk k (jb = 64 k) loads entry r = jb + l of two sequences: the
        // column's f from p = -1 (f at p-cell jb - 1 + l; rows ic - 2 .. ic + 2
        // for the interpolation) and the logarithm table (entry jb + l), with r
        // clamped to n_p + 2 (f at p-cell n_p + 1, past the table's last), and
        // the nested flag of p-cell jb + l, clamped to the last; those clamped
        // entries serve skipped cells only.  The chunk's address is scalar, the
        // lane adds a 32-bit offset.
        const double *row = P.f + pidx(P.pitch, RTB == 1 ? ic : ic - 2, -1);
        const uint8_t *nrow = NEST ? P.nested + pidx(P.pitch, ic, 0) : nullptr;
        auto h = [&](int m, double a2) {
            const double pm = momentum(P.pmin, P.dp, m, P.p_pos);
            return gamma_(pm, a2, P.mc2inv) + P.c1 * pm;
        };
        // sub-cell values of a p-cell from its rows (Rectangle.cpp:76-110)
        auto values = [&](const double *f, double *v) __attribute__((always_inline)) {
            if (RTB == 1) {
                v[0] = f[0];
                return;
            }
            const double f3 = f[NR / 2];
            const double f1 = f[0] - f3, f2 = f[NR > 1 ? 1 : 0] - f3, f4 = f[NR > 3 ? 3 : 0] - f3,
                         f5 = f[NR > 4 ? 4 : 0] - f3;
            const double a1 = kInterp[0] * f1 + kInterp[1] * f2 + kInterp[2] * f4 + kInterp[3] * f5;
            const double a2 = kInterp[4] * f1 + kInterp[5] * f2 + kInterp[6] * f4 + kInterp[7] * f5;
            const double a3 = kInterp[8] * f1 + kInterp[9] * f2 + kInterp[10] * f4 + kInterp[11] * f5;
            double te = 0.0;
#pragma unroll
            for (int s = 0; s < RTB; s++) {
                v[s] = P.rel[3 * s] * a1 + P.rel[3 * s + 1] * a2 + P.rel[3 * s + 2] * a3 + f3;
                te += v[s] + 0.0;  // the interpolant with a zero correction
            }
            const double corr = f3 - P.inv_rtb * te;
#pragma unroll
            for (int s = 0; s < RTB; s++) v[s] = v[s] + corr;
        };
        // The loop is specialised on the table case, so that no branch joins
        // the registers of the chunks in flight (a join makes the loads wait),
        // and its ring of chunks in flight is unrolled: slot d holds chunk
        // k0 + d in fixed registers and is reloaded with chunk k0 + d + WDEPTH
        // once its values are formed (a rotating copy would wait for the loads
        // in flight).  COMP with a table at RTB 1, a loop of few instructions, has no exit
        // inside it (the chunks past the last are skipped cells) and reloads a slot
        // behind the chunk's sums: 4096 x 4096 29.0 us against 32.6, 2048 x 4096 18.3
        // and 20.9.
        double aR[RTB], cR[RTB], aJ[RTB], cJ[RTB];  // COMP: the lanes' sums
#pragma unroll
        for (int s = 0; s < RTB; s++) aR[s] = cR[s] = aJ[s] = cJ[s] = 0.0;
        auto run = [&](auto tab_c) __attribute__((always_inline)) {
            constexpr bool TAB = decltype(tab_c)::value;
            constexpr int NL = TAB ? 1 : RTB;  // logarithm sequences
            constexpr bool WHOLE = COMP && TAB && RTB == 1;  // whole rounds of the ring, loads behind the sums
            double pv[WDEPTH][NR], pt[WDEPTH];
            int pn[WDEPTH];
            auto load = [&](int k, int d) __attribute__((always_inline)) {
                const int jl = min(64 * k, P.n_p + 2);
                const uint32_t vo = 8 * (uint32_t)min(lane, P.n_p + 2 - jl);
#pragma unroll
                for (int q = 0; q < NR; q++) pv[d][q] = *(const double *)((const char *)(row + (long)q * P.pitch + jl) + vo);
                if (TAB) pt[d] = *(const double *)((const char *)(tab + jl) + vo);
                if (NEST) {
                    const int jn = min(64 * k, P.n_p - 1);
                    pn[d] = (nrow + jn)[(uint32_t)min(lane, P.n_p - 1 - jn)];
                }
            };
            // the slots are loaded in the order they are used (the scheduling
            // barriers keep the compiler from reordering them), so that waiting
            // for slot d leaves the later slots' loads in flight
#pragma unroll
            for (int d = 0; d < WDEPTH; d++) {
                load(d, d);
                __builtin_amdgcn_sched_barrier(0);
            }
            // logarithm terms c2 log(h(m)/h(m-1)) of sub-column s at m = jb + l,
            // h(m - 1) from the lane below (lane 0: the last chunk's h(jb - 1))
            double hl[RTB];
            auto logs = [&](int jb, double *out) __attribute__((always_inline)) {
#pragma unroll
                for (int s = 0; s < RTB; s++) {
                    if (s > 0 && same_bits(asq[s], asq[s - 1])) {  // uniform
                        out[s] = out[s - 1];
                        hl[s] = hl[s - 1];
                        continue;
                    }
                    const double hm = h(jb + lane, asq[s]), hs = shup1(hm);
                    out[s] = P.c2 * log_ratio(hm, lane == 0 ? hl[s] : hs);
                    hl[s] = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(hm), 63),
                                             __builtin_amdgcn_readlane(__double2loint(hm), 63));
                }
            };
            double V[RTB], L[NL];
            values(pv[0], V);
            if (TAB) {
                L[0] = pt[0];
            } else {
#pragma unroll
                for (int s = 0; s < RTB; s++) hl[s] = h(-1, asq[s]);
                logs(0, L);
            }
            int nf = NEST ? pn[0] : 0;
            for (int k0 = 0; !WHOLE || k0 < nchunk; k0 += WDEPTH) {
#pragma unroll
                for (int d = 0; d < WDEPTH; d++) {
                    // chunk k, its values in V and L (the only branch leaves
                    // the loop, so the wait for each slot's loads counts only
                    // the slots loaded after it)
                    const int k = k0 + d, dn = (d + 1) % WDEPTH;  // dn: chunk k + 1
                    const int jb = 64 * k;
                    if (!WHOLE) {
                        load(k + WDEPTH, d);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    double Vn[RTB], Ln[NL];
                    values(pv[dn], Vn);
                    if (TAB) Ln[0] = pt[dn];
                    else logs(jb + 64, Ln);
                    const bool skip = (jb + lane >= P.n_p) | !col_ok | (nf != 0);
                    double gm, gp1;
#pragma unroll
                    for (int s = 0; s < RTB; s++) {
                        if (s < NL) next2_rot(lane, L[s], Ln[s], gm, gp1);
                        double t0, tp;
                        next2_rot(lane, V[s], Vn[s], t0, tp);
                        const double tm = V[s], gm1 = L[s < NL ? s : 0];
                        const double jv = t0 * gm + P.c3 * (gp1 - gm1) * (tp - tm);
                        const double tr = skip ? -0.0 : t0, tj = skip ? -0.0 : jv;
                        if (COMP) {
                            add_two(aR[s], cR[s], tr);
                            add_two(aJ[s], cJ[s], tj);
                        } else {
                            T[k & 1][0][wave * RTB + s][lane] = tr;
                            T[k & 1][1][wave * RTB + s][lane] = tj;
                        }
                    }
#pragma unroll
                    for (int s = 0; s < RTB; s++) V[s] = Vn[s];
#pragma unroll
                    for (int s = 0; s < NL; s++) L[s] = Ln[s];
                    if (NEST) nf = pn[dn];
                    if (WHOLE) load(k + WDEPTH, d);
                    __builtin_amdgcn_sched_barrier(0);
                    if (!COMP) __syncthreads();
                    if (!WHOLE && k + 1 == nchunk) return;
                }
            }
        };
        if (tab) run(std::true_type{});
        else run(std::false_type{});
        if (COMP) {
#pragma unroll
            for (int s = 0; s < RTB; s++) {
                double sr, er, sj, ej;
                wave_two_sum(aR[s], cR[s], sr, er);
                wave_two_sum(aJ[s], cJ[s], sj, ej);
                if (lane == 0 && col_ok) {
                    const long e = (long)i * RTB + s;
                    const double q = (sr + er) * P.dpq, J = (sj + ej) * P.jscale;
                    P.chargeR[e] = q;
                    P.currentR[e] = J;
                    if (P.charge) {
                        P.charge[e] = P.species[e] = 0.0 + q;
                        P.J[e] = 0.0 + J;
                    }
                }
            }
        }
    } else if (!COMP) {
        // consumer: chain (lane & 31) of charge (lanes < 32) or current; lanes
        // past the chains repeat chain 0 and are not stored
        // the dependent additions are the critical path of each chunk: the
        // consumer issues ahead of the producers that share its SIMD
        __builtin_amdgcn_s_setprio(3);
        const int c = lane & 31, ch = c < NCH ? c : 0;
        const int kind = lane >> 5;
        double acc = 0.0;
        for (int k = 0; k < nchunk; k++) {
            __syncthreads();  // chunk k is in its buffer
            const double *row = &T[k & 1][kind][ch][0];
#pragma unroll
            for (int e = 0; e < 64; e += 8) {
                const double v0 = row[e], v1 = row[e + 1], v2 = row[e + 2], v3 = row[e + 3];
                const double v4 = row[e + 4], v5 = row[e + 5], v6 = row[e + 6], v7 = row[e + 7];
                acc += v0; acc += v1; acc += v2; acc += v3; acc += v4; acc += v5; acc += v6; acc += v7;
            }
        }
        const int i = i0 + c / RTB;
        if (c < NCH && i < P.n_x) {
            const long e = (long)i * RTB + c % RTB;
            if (lane < 32) put_charge(P, e, acc * P.dpq);
            else put_current(P, e, acc * P.jscale);
        }
    }
}

template <int RTB, bool COMP, bool NEST, int WCOL = MCOL>
__global__ __launch_bounds__(64 * (WCOL + 1)) void k_moments(MomArgs A) {
    __shared__ double T[COMP ? 1 : 2 * 2 * WCOL * RTB * 65];
    moments_columns<RTB, WCOL, COMP, NEST>(A.p, A.fl, A.tab, (int)blockIdx.x, T);
}

// The patches of a hierarchy in one launch, without tables.  A patch's own launch
// leaves most of the chip idle at its end (and, for a coarse patch, throughout).
// Three patches of 1.27, 0.34 and 1.05 M cells on an MI355X: 43 us, apart 42 us and two
// checks of the tables, 4.5 us each; 22 steps of the laser run 40.9 -> 39.9 ms.
template <bool COMP>
__global__ __launch_bounds__(64 * (MCOL + 1)) void k_moments_batch(MomBatch A) {
    constexpr int WCOL = MCOL;
    __shared__ double T[COMP ? 1 : 2 * 2 * WCOL * MAX_RTB * 65];
    int k = 0;
    while (k + 1 < A.n && (int)blockIdx.x >= A.start[k + 1]) k++;
    const MomPatch P = A.p[k];
    const int blk = (int)blockIdx.x - A.start[k];
    switch (P.rtb * 2 + (P.nested ? 1 : 0)) {
        case 2: moments_columns<1, WCOL, COMP, false>(P, A.fl, nullptr, blk, T); break;
        case 3: moments_columns<1, WCOL, COMP, true>(P, A.fl, nullptr, blk, T); break;
        case 4: moments_columns<2, WCOL, COMP, false>(P, A.fl, nullptr, blk, T); break;
        case 5: moments_columns<2, WCOL, COMP, true>(P, A.fl, nullptr, blk, T); break;
        case 8: moments_columns<4, WCOL, COMP, false>(P, A.fl, nullptr, blk, T); break;
        default: moments_columns<4, WCOL, COMP, true>(P, A.fl, nullptr, blk, T);
    }
}

// Rectangle::CalculateEnergy (Rectangle.cpp:284-305) without its data race:
// chain (j, k) sums the p-sub-cell value k of every non-nested cell (i, j) in
// increasing i, then scales by dx (the reference's OpenMP loop adds to the same
// energyR entries from several threads; the oracle and this kernel use the
// sequential order).
template <int RTB>
__global__ __launch_bounds__(256) void k_energy(MomPatch P, double *energyR) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= P.n_p * RTB) return;
    const int j = e / RTB, k = e % RTB;
    const int pitch = P.pitch;
    const double *g = P.f;
    double acc = 0.0;
    for (int i = 0; i < P.n_x; i++) {
        if (P.nested && P.nested[pidx(pitch, i, j)]) continue;
        double f1 = g[pidx(pitch, i, j - 2)], f2 = g[pidx(pitch, i, j - 1)], f3 = g[pidx(pitch, i, j)];
        double f4 = g[pidx(pitch, i, j + 1)], f5 = g[pidx(pitch, i, j + 2)];
        f5 -= f3; f4 -= f3; f2 -= f3; f1 -= f3;
        double a1 = kInterp[0] * f1 + kInterp[1] * f2 + kInterp[2] * f4 + kInterp[3] * f5;
        double a2 = kInterp[4] * f1 + kInterp[5] * f2 + kInterp[6] * f4 + kInterp[7] * f5;
        double a3 = kInterp[8] * f1 + kInterp[9] * f2 + kInterp[10] * f4 + kInterp[11] * f5;
        acc += P.rel[3 * k] * a1 + P.rel[3 * k + 1] * a2 + P.rel[3 * k + 2] * a3 + f3;
    }
    energyR[(long)j * RTB + k] = acc * P.dx;
}

struct MomentSrc {
    const double *chargeR, *currentR;
    int start, count;  // finest-grid span [start, start + count)
};

// Assembly in the reference order: per species, levels finest first, one
// patch per finest index and level (patches of a level do not overlap).
__global__ void k_assemble(const MomentSrc *src, const int *level_start, int n_species,
                           int n_levels, int n_f, double *charge, double *J,
                           double *charges_species) {
    int x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= n_f) return;
    double jsum = 0.0;  // EMSolver::J, accumulated over species and levels
    double ch = 0.0;
    for (int s = 0; s < n_species; s++) {
        double cs_ = 0.0;  // charges[s][x]
        for (int l = 0; l < n_levels; l++) {
            double cl = 0.0, jl = 0.0;  // chargeL / currentL of level l
            int a = level_start[s * n_levels + l], b = level_start[s * n_levels + l + 1];
            for (int q = a; q < b; q++) {
                int off = x - src[q].start;
                if (off >= 0 && off < src[q].count) {
                    cl += src[q].chargeR[off];
                    jl += src[q].currentR[off];
                }
            }
            cs_ += cl;
            jsum += jl;
        }
        if (charges_species) charges_species[(long)s * n_f + x] = cs_;
        ch += cs_;
    }
    charge[x] = ch;
    J[x] = jsum;
}

MomPatch mom_patch(const vx_patch &p) {
    MomPatch M{p.f[1], p.nested, p.chargeR, p.currentR, p.n_x, p.n_p, p.x_pos, p.p_pos, p.rtb, p.pitch,
               p.dx, p.dp, p.pmin, p.q, p.mc2inv};
    double m_inv = 1 / p.m;
    M.c1 = m_inv * vx_c_inv;
    M.c2 = 1 / M.c1;
    M.c3 = 1 / 48.0;
    double rtb = (double)p.rtb;
    M.inv_rtb = 1.0 / rtb;
    M.dpq = p.dp * p.q;
    M.jscale = -p.q * p.q / p.m;
    for (int i = 0; i < std::min(p.rtb, MAX_RTB); i++) {  // Rectangle.cpp:103-110
        double tl = -0.5 + i / rtb;
        double tr = -0.5 + (i + 1.0) / rtb;
        M.rel[3 * i] = (tl + tr) * 0.5;
        M.rel[3 * i + 1] = (tl * tl + tl * tr + tr * tr) / 3.0 - (1.0 / 12);
        M.rel[3 * i + 2] = (tl * tl * tl + tl * tl * tr + tl * tr * tr + tr * tr * tr) * 0.25;
    }
    M.charge = M.J = M.species = nullptr;
    return M;
}

}  // namespace

extern "C" {

int vx_energy_patch(vx_ctx *ctx, const vx_patch *p, double *energyR) {
    int rc = validate_patch(ctx, p);
    if (rc) return rc;
    if (!energyR) return fail(ctx, VX_EINVAL, "energy: null output");
    const MomPatch A = mom_patch(*p);
    const unsigned nb = (unsigned)((p->n_p * p->rtb + 255) / 256);
    switch (p->rtb) {
        case 1: k_energy<1><<<nb, 256, 0, ctx->stream>>>(A, energyR); break;
        case 2: k_energy<2><<<nb, 256, 0, ctx->stream>>>(A, energyR); break;
        case 4: k_energy<4><<<nb, 256, 0, ctx->stream>>>(A, energyR); break;
        default: return fail(ctx, VX_ENOTSUP, "energy: relativeToBottom %d not in {1,2,4}", p->rtb);
    }
    return check_launch(ctx, "k_energy");
}

}  // extern "C"

static int moments_check(vx_ctx *ctx, const vx_patch *p, const vx_fields *fl) {
    int rc = validate_patch(ctx, p);
    if (rc) return rc;
    if (p->rtb > MAX_RTB) return fail(ctx, VX_ENOTSUP, "moments: relativeToBottom %d > %d", p->rtb, MAX_RTB);
    if (!fl) return fail(ctx, VX_EINVAL, "moments: null fields");
    if ((rc = validate_span(ctx, p, fl->n_f))) return rc;
    if (p->rtb != 1 && p->rtb != 2 && p->rtb != 4)
        return fail(ctx, VX_ENOTSUP, "moments: relativeToBottom %d not in {1,2,4}", p->rtb);
    return VX_OK;
}

// whole: where the patch's moments are the assembled ones, the places of the charge,
// the current and its species' charge.
static int moments_patch(vx_ctx *ctx, const vx_patch *p, const vx_fields *fl, bool comp,
                         double *const *whole = nullptr) {
    int rc = moments_check(ctx, p, fl);
    if (rc) return rc;
    MomArgs A{mom_patch(*p), *fl, nullptr};
    if (whole) {
        A.p.charge = whole[0];
        A.p.J = whole[1];
        A.p.species = whole[2];
        // (a patch without arrays of its own: written, then written again as assembled)
        if (!A.p.chargeR) A.p.chargeR = whole[0];
        if (!A.p.currentR) A.p.currentR = whole[1];
    }
    // The table saves each column its logarithms but costs a launch (3.1 us).
    // us with / without it: 1024 x 512 at rtb 1 8.3 / 7.0, 1024 x 1024 11.9 / 10.7,
    // 2048 x 1024 12.1 / 15.4; 2000 x 64 at rtb 4 7.8 / 6.1, 512 x 512 11.4 / 12.4,
    // 8000 x 256 27.8 / 33.7; columns with a pulse do not use it (500 x 512 at rtb
    // 4 21.1 / 19.1).  A wavefront that forms the terms for its workgroup's columns
    // instead: 9.2 at 1024 x 1024, but 52 at 4096 x 4096, 46 with the table.
    // In launches that do not fill the device a column's chain of chunks counts: any
    // up to 512 columns at rtb 1, of 1280 p-cells 12.4 / 11.8, 1536 13.6 / 13.7, 2048 16.2 / 17.4,
    // 4096 27.3 / 31.7; compensated, of 1024 8.7 / 9.5, 2048 10.6 / 15.8, 4096 15 / 28.
    // (They go without where a graph is recorded before there is a table.)
    size_t need = (size_t)tab_entries(2, p->n_p);
    const bool tall = p->rtb == 1 && p->n_p > (comp ? 1024 : 1536) &&
                      !(ctx->capturing && ctx->mom_table_n < need);
    if (tall || (long)p->n_x * p->n_p > TAB_CELLS) {
        if (ctx->mom_table_n < need) {
            if (ctx->capturing) return fail(ctx, VX_EINVAL, "moments: table growth while a step graph is recorded");
            // The outgrown table stays until the context ends: a graph recorded
            // with it writes and reads it when it is replayed.  Each table has at
            // least twice the entries of the one before, so that all of them
            // together are less than two of the largest.
            need = std::max(need, 2 * ctx->mom_table_n);
            double *table = nullptr;
            if (hipMalloc(&table, sizeof(double) * need) != hipSuccess)
                return fail(ctx, VX_ENOMEM, "moments: logarithm table");
            // no table in place yet (flag 0)
            if (hipMemsetAsync(table, 0, sizeof(double) * need, ctx->stream) != hipSuccess) {
                (void)hipFree(table);
                return fail(ctx, VX_EHIP, "moments: logarithm table clear");
            }
            if (ctx->mom_table) ctx->mom_old.push_back(ctx->mom_table);
            ctx->mom_table = table;
            ctx->mom_table_n = need;
        }
        A.tab = ctx->mom_table;
        switch (p->rtb) {
            case 1: k_moment_table<1><<<2, 1024, 0, ctx->stream>>>(A, ctx->mom_table); break;
            case 2: k_moment_table<2><<<2, 1024, 0, ctx->stream>>>(A, ctx->mom_table); break;
            default: k_moment_table<4><<<2, 1024, 0, ctx->stream>>>(A, ctx->mom_table);
        }
        if ((rc = check_launch(ctx, "k_moment_table"))) return rc;
    }
    LaunchTimer lt(ctx, "k_moments");
    // 8 columns a workgroup where both the columns are tall and the workgroups fill
    // the device: one consumer for more of them, and enough chunks for its start.  us,
    // 8 / 4 columns, without and with a pulse: 8190 x 1024 30.1 / 31.6, 53.5 / 46.5; 4096 x
    // 2048 27.2 / 27.1, 43.8 / 45.8; 4096 x 4096 34.2 / 40.7, 75.9 / 83.1; compensated 18.0 /
    // 22.6 and 29.0 / 30.3 without.  Where they do not: 1024 x 2048 with a pulse 26.5 / 20.2,
    // 64 x 4096 without a table 44.3 / 31.6.
    const bool wide = p->rtb == 1 && !p->nested && p->n_p >= 2048 && p->n_x >= MCOL_TALL * ctx->n_cu;
    const int WCOL = wide ? MCOL_TALL : MCOL;
    const dim3 g((unsigned)((p->n_x + WCOL - 1) / WCOL)), b(64 * (comp ? WCOL : WCOL + 1));
    if (wide) {
        if (comp) k_moments<1, true, false, MCOL_TALL><<<g, b, 0, ctx->stream>>>(A);
        else k_moments<1, false, false, MCOL_TALL><<<g, b, 0, ctx->stream>>>(A);
        return check_launch(ctx, "k_moments");
    }
    switch (p->rtb * 4 + (comp ? 2 : 0) + (p->nested ? 1 : 0)) {
        case 4: k_moments<1, false, false><<<g, b, 0, ctx->stream>>>(A); break;
        case 5: k_moments<1, false, true><<<g, b, 0, ctx->stream>>>(A); break;
        case 6: k_moments<1, true, false><<<g, b, 0, ctx->stream>>>(A); break;
        case 7: k_moments<1, true, true><<<g, b, 0, ctx->stream>>>(A); break;
        case 8: k_moments<2, false, false><<<g, b, 0, ctx->stream>>>(A); break;
        case 9: k_moments<2, false, true><<<g, b, 0, ctx->stream>>>(A); break;
        case 10: k_moments<2, true, false><<<g, b, 0, ctx->stream>>>(A); break;
        case 11: k_moments<2, true, true><<<g, b, 0, ctx->stream>>>(A); break;
        case 16: k_moments<4, false, false><<<g, b, 0, ctx->stream>>>(A); break;
        case 17: k_moments<4, false, true><<<g, b, 0, ctx->stream>>>(A); break;
        case 18: k_moments<4, true, false><<<g, b, 0, ctx->stream>>>(A); break;
        default: k_moments<4, true, true><<<g, b, 0, ctx->stream>>>(A);
    }
    return check_launch(ctx, "k_moments");
}

extern "C" {

int vx_moments_patch(vx_ctx *ctx, const vx_patch *p, const vx_fields *fl) {
    return moments_patch(ctx, p, fl, false);
}

int vx_moments_patch_compensated(vx_ctx *ctx, const vx_patch *p, const vx_fields *fl) {
    return moments_patch(ctx, p, fl, true);
}

int vx_moments_whole(vx_ctx *ctx, const vx_patch *p, const vx_fields *fl, int compensated, double *charge, double *J,
                     double *charges_species) {
    int rc = moments_check(ctx, p, fl);
    if (rc) return rc;
    if (!charge || !J || !charges_species) return fail(ctx, VX_EINVAL, "moments: null output");
    if (p->x_pos != 0 || p->n_x * p->rtb != fl->n_f)
        return fail(ctx, VX_EINVAL, "moments: the patch does not cover the %d finest cells", fl->n_f);
    double *const whole[] = {charge, J, charges_species};
    return moments_patch(ctx, p, fl, compensated != 0, whole);
}

int vx_moments_patches(vx_ctx *ctx, const vx_patch *patches, int32_t n, const vx_fields *fl, int compensated) {
    if (n < 0 || (n > 0 && !patches)) return fail(ctx, VX_EINVAL, "moments: bad patch list");
    int rc;
    for (int k = 0; k < n; k++)
        if ((rc = moments_check(ctx, patches + k, fl))) return rc;
    MomBatch B;
    B.n = 0;
    // the last patches first (a hierarchy lists its levels finest first, and a
    // coarse patch's workgroups run longest)
    for (int k = n; k-- > 0;) {
        const vx_patch &p = patches[k];
        const bool alone = n == 1 || (long)p.n_x * p.n_p > BATCH_CELLS;
        if (alone) {
            if ((rc = moments_patch(ctx, &p, fl, compensated != 0))) return rc;
        } else {
            if (B.n == 0) B.start[0] = 0;
            B.p[B.n++] = mom_patch(p);
            B.start[B.n] = B.start[B.n - 1] + (p.n_x + MCOL - 1) / MCOL;
        }
        if (B.n == MOM_BATCH || (k == 0 && B.n > 0)) {
            B.fl = *fl;
            LaunchTimer lt(ctx, "k_moments");
            if (compensated) k_moments_batch<true><<<(unsigned)B.start[B.n], 64 * MCOL, 0, ctx->stream>>>(B);
            else k_moments_batch<false><<<(unsigned)B.start[B.n], 64 * (MCOL + 1), 0, ctx->stream>>>(B);
            if ((rc = check_launch(ctx, "k_moments_batch"))) return rc;
            B.n = 0;
        }
    }
    return VX_OK;
}

int vx_moment_plan_create(vx_ctx *ctx, const vx_patch *patches, const vx_moment_layout *lay,
                          int32_t n_f, vx_moment_plan **out) {
    if (!out) return fail(ctx, VX_EINVAL, "null plan pointer");
    *out = nullptr;
    if (!lay || lay->n_species < 1 || lay->n_levels < 1 || n_f < 1)
        return fail(ctx, VX_EINVAL, "bad moment layout");
    if (ctx->capturing) return fail(ctx, VX_EINVAL, "moment plan while a step graph is recorded");
    int ngroups = lay->n_species * lay->n_levels;
    int npatch = lay->level_start[ngroups];
    std::vector<MomentSrc> src(npatch > 0 ? npatch : 1);
    for (int q = 0; q < npatch; q++) {
        src[q].chargeR = patches[q].chargeR;
        src[q].currentR = patches[q].currentR;
        src[q].start = patches[q].x_pos * patches[q].rtb;
        src[q].count = patches[q].n_x * patches[q].rtb;
    }
    size_t sb = sizeof(MomentSrc) * src.size();
    size_t bytes = sb + sizeof(int) * (ngroups + 1);
    vx_moment_plan *pl = new vx_moment_plan;
    pl->n_species = lay->n_species;
    pl->n_levels = lay->n_levels;
    pl->n_f = n_f;
    if (hipMalloc(&pl->tables, bytes) != hipSuccess) {
        delete pl;
        return fail(ctx, VX_ENOMEM, "moment plan tables");
    }
    std::vector<char> host(bytes);
    std::memcpy(host.data(), src.data(), sb);
    std::memcpy(host.data() + sb, lay->level_start, sizeof(int) * (ngroups + 1));
    hipError_t e = hipMemcpy(pl->tables, host.data(), bytes, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        (void)hipFree(pl->tables);
        delete pl;
        return fail(ctx, VX_EHIP, "moment plan copy: %s", hipGetErrorString(e));
    }
    pl->src_off = 0;
    pl->ls_off = sb;
    *out = pl;
    return VX_OK;
}

void vx_moment_plan_destroy(vx_moment_plan *pl) {
    if (!pl) return;
    (void)hipFree(pl->tables);
    delete pl;
}

int vx_moments_assemble(vx_ctx *ctx, const vx_moment_plan *pl, double *charge, double *J,
                        double *charges_species) {
    if (!pl) return fail(ctx, VX_EINVAL, "null moment plan");
    const MomentSrc *dsrc = (const MomentSrc *)((char *)pl->tables + pl->src_off);
    const int *dls = (const int *)((char *)pl->tables + pl->ls_off);
    k_assemble<<<(unsigned)((pl->n_f + 255) / 256), 256, 0, ctx->stream>>>(
        dsrc, dls, pl->n_species, pl->n_levels, pl->n_f, charge, J, charges_species);
    return check_launch(ctx, "k_assemble");
}

}  // extern "C"
