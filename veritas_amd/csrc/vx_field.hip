// 1-D field solver on the finest grid (EMFieldSolver, EMSolver.cpp).
//
// Poisson (EMSolver.cpp:28-88,156-192).  The reference factors the dense N x N
// matrix with LAPACK and solves it at every RK stage, O(N^2) per solve.  Here
// the same matrix is solved to near correct rounding in O(N) (one workgroup
// with the vector in registers up to N = 4096, a sequence of multi-workgroup
// launches above):
//   rows 1..N-1 of the matrix are the periodic 4th-order stencil
//   (w2, w1, w3, w1, w2) with column 0 removed, i.e. the periodic operator with
//   phi_0 pinned to 0; row 0 then gives phi_0.  The periodic operator factors
//   exactly as L4 = L2 * M with L2 = [-1, 2, -1] and M = [-1, 14, -1] / 12, so
//   an approximate solve is two prefix sums (L2^-1 on zero-mean data) and M^-1,
//   whose entries decay as (7 - 4 sqrt 3)^|k| (a 33-tap convolution, or two
//   first-order recurrences).
//   Two or three rounds of iterative refinement with a double-double residual of the
//   reference's own coefficients take the result to the correctly rounded
//   solution (the CPU oracle reaches the same point with a band LU).
//
// Transverse fields (EMSolver.cpp:194-338, 479-619): one thread per cell.
#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

#include "vx_dev.h"

#include "vx_internal.h"

using namespace vxi;
using namespace vxd;

namespace {

constexpr int NG = 17;    // convolution half-width + 1 for M^-1

struct PoissonArgs {
    vx_field_state fs;
    double w1, w2, w3;
    double g[NG];  // M^-1 coefficients, g[|k|]
    double rho, C;  // M^-1 = C (1 - rho S^-1)^-1 (1 - rho S)^-1
    double invN;
};


// DPP move of a double; lanes outside row_mask or without a source lane get 0
template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ double dpp_or_0(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROW_MASK, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROW_MASK, 0xf, true);
    return __hiloint2double(hi, lo);
}

// Inclusive scan over the wavefront's lanes: within rows of 16 by row shifts
// of 1, 2, 4, 8, then row 0's total into row 1 and row 2's into row 3
// (row_bcast:15), then rows 0-1's total into rows 2 and 3 (row_bcast:31).
__device__ __forceinline__ double wave_scan_dpp(double v) {
    v += dpp_or_0<0x111>(v);
    v += dpp_or_0<0x112>(v);
    v += dpp_or_0<0x114>(v);
    v += dpp_or_0<0x118>(v);
    v += dpp_or_0<0x142, 0xa>(v);
    v += dpp_or_0<0x143, 0xc>(v);
    return v;
}

__device__ __forceinline__ double lane63(double v) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                            __builtin_amdgcn_readlane(__double2loint(v), 63));
}

// sh + sl -= a xq, the product and sums error-free
__device__ __forceinline__ void dd_sub(double &sh, double &sl, double a, double xq) {
    const double p = a * xq;
    const double e = fma(a, xq, -p);
    const double tt = sh - p;
    const double bv = tt - sh;
    const double err = (sh - (tt - bv)) + (-p - bv);
    sl = sl + (err - e);
    sh = tt;
}

// ------------------------------------------------ multi-workgroup solve, 4096 < n_f <= PM_MAX
// Workgroup b owns the chunk of 64 MW consecutive entries from 64 MW b on,
// wavefront w of it the sub-chunk w of 64 entries.  One approximate solve of
// A c = v and the residual of the next round are one launch:
//   S_i = sum_{k<i} v'_k with v'_0 = -tail, tail = sum_{k>=1} v_k,
//   d0 = mean(S), D_i = d0 - S_i (D_0 = 0), y_i = sum_{k<=i} D_k,
//   c = M^-1 y - (M^-1 y)_0 with c_0 from row 0, x (+)= c, then either the
//   next residual r = b - A x (double-double) or phi, Ex0 and E.
// Both prefix sums at a chunk's first entry follow from two numbers per earlier
// chunk, the sum M of its v and the sum P of its local exclusive prefixes of v:
//   S = -tail + sum_q M_q,   sum_{i<start} S_i = sum_q (M_q (start - end_q) + P_q) - tail (start - 1)
// (and within a chunk the same over its sub-chunks), so the launch that forms v
// writes M and P (k_pm_rhs for the first solve) and the next one needs no launch
// in between.  The terms M (start - end) are up to n_f times what they sum to
// (v is a difference of differences), so M, P and these sums are held in
// double-double: in double, entries of phi that cancel lose their last bits.  Every
// wavefront forms a sub-chunk's y from those sums by the same operations,
// whichever workgroup it is in, so the y of a neighbour's sub-chunk, formed again
// for the reach of M^-1, has the owner's bits; so have the x on a 2-entry halo
// (for the residual and E stencils) and at the six entries around 0 (row 0 and
// Ex0).  x and r alternate between two buffers: a launch reads one and writes
// the other.
// Bound by launch latency and each launch's chain (sums, two scans,
// convolution, residual, sums), and by FP64 issue where a CU has many
// wavefronts: five more than the chunk's form y.  MW = 3 gives a SIMD two of the
// eight and 32768 entries 171 CUs; above PM_SMALL the sums over the chunks weigh
// more, and MW = 8 has fewer.  us on an MI355X at 8192, 32768 and 100000 entries: MW =
// 2 29, 33, 97; 3 28, 31, 65; 4 32, 34, 56; 8 39, 38, 44.  32768 entries took 77 us
// as 13 launches (the two scans and the convolution apart), 42 us as 5 with MW = 8 and
// each launch's reads one behind the other.
constexpr int PM_SMALL = 192 * 192;  // largest n_f with MW = 3: three chunks a lane
constexpr int PM_MAX = 512 * 256;      // largest n_f of this form: a chunk for every compute unit
__host__ __device__ constexpr int pm_mw(int n) { return n <= PM_SMALL ? 3 : 8; }
constexpr int SUB = 64;
constexpr int HALO = 2;
constexpr int CW = NG - 1 + HALO;  // y window margin: convolution reach + halo
constexpr int NSPEC = 6;           // entries N-3, N-2, N-1, 0, 1, 2
constexpr int YS = NSPEC + 2 * (NG - 1);  // y window of those entries

__host__ __device__ constexpr int pm_chunks(int n) { return (n + SUB * pm_mw(n) - 1) / (SUB * pm_mw(n)); }

// M and P of a chunk or sub-chunk, double-double
struct PmSum {
    double mh, ml, ph, pl;
};

// Work layout (doubles): b | xa | xb | ra | rb | Ex0 on entry | per parity: the chunks'
// sums, the sub-chunks'
struct PmWork {
    double *b, *xa, *xb, *ra, *rb, *ex0;
    PmSum *sums[2];
};
__host__ __device__ inline PmWork pm_work(double *w, int n) {
    const size_t N = n, ns = (size_t)pm_chunks(n) * (1 + pm_mw(n));
    PmWork W;
    W.b = w;
    W.xa = w + N;
    W.xb = w + 2 * N;
    W.ra = w + 3 * N;
    W.rb = w + 4 * N;
    W.ex0 = w + 5 * N;
    W.sums[0] = (PmSum *)(W.ex0 + 1);
    W.sums[1] = W.sums[0] + ns;
    return W;
}

struct PoissonMB {
    vx_field_state fs;
    double w1, w2, w3;
    double g[NG];
    double invN;
    int nb;
    PmWork W;
    const double *in;    // right-hand side of this solve (b, then residuals)
    const PmSum *sums;   // its M, P
    PmSum *sums_out;     // those of the next residual
    const double *x_in;  // x before this solve's correction
    double *x_out;       // x after it
    double *r_out;       // next residual
};

__device__ __forceinline__ int wrap(int u, int N) { return u < 0 ? u + N : (u >= N ? u - N : u); }

// (M^-1 y) at window position c: the periodic 33-tap convolution
__device__ __forceinline__ double conv_at(const double *w, int c, const double *g) {
    double s = g[0] * w[c];
    for (int k = 1; k < NG; k++) s += g[k] * (w[c + k] + w[c - k]);
    return s;
}

struct DD {
    double h, l;
};
__device__ __forceinline__ DD dd_add(DD a, DD b) {
    const double s = a.h + b.h, z = s - a.h;
    return {s, ((a.h - (s - z)) + (b.h - z)) + (a.l + b.l)};
}
__device__ __forceinline__ DD dd_neg(DD a) { return {-a.h, -a.l}; }
__device__ __forceinline__ DD dd_mul(DD a, double b) {
    const double p = a.h * b;
    return {p, __builtin_fma(a.h, b, -p) + a.l * b};
}
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ DD dd_step(DD v) {
    return dd_add(v, {dpp_or_0<CTRL, ROW_MASK>(v.h), dpp_or_0<CTRL, ROW_MASK>(v.l)});
}
// sum over the wavefront's lanes (wave_scan_dpp's steps), the same in every lane
__device__ __forceinline__ DD wave_dd_sum(DD v) {
    v = dd_step<0x111, 0xf>(v);
    v = dd_step<0x112, 0xf>(v);
    v = dd_step<0x114, 0xf>(v);
    v = dd_step<0x118, 0xf>(v);
    v = dd_step<0x142, 0xa>(v);
    v = dd_step<0x143, 0xc>(v);
    return {lane63(v.h), lane63(v.l)};
}

// sum over lanes 0..7, in lane 7 (wave_scan_dpp's first steps)
__device__ __forceinline__ DD row_dd_sum8(DD v) {
    v = dd_step<0x111, 0xf>(v);
    v = dd_step<0x112, 0xf>(v);
    return dd_step<0x114, 0xf>(v);
}

// M and P of a wavefront's 64 entries v (entry 0 and entries past N passed as
// 0) and of the workgroup's chunk of n_own entries, into out.  P is the sum of v_l
// (n - 1 - l), n the wavefront's entries below N.
template <int MW>
__device__ __forceinline__ void pm_store_sums(double v, int n_own, PmSum *out, int nb, PmSum *ms) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, blk = blockIdx.x;
    const int n = min(SUB, n_own - w * SUB);
    const DD m = wave_dd_sum({v, 0.0}), p = wave_dd_sum(dd_mul({v, 0.0}, (double)max(n - 1 - lane, 0)));
    if (lane == 0 && w < MW) {
        const PmSum q{m.h, m.l, p.h, p.l};
        ms[w] = q;
        out[nb + blk * MW + w] = q;
    }
    __syncthreads();
    if (w == 0) {  // lane k: sub-chunk k, moved to the chunk's end
        DD M{0.0, 0.0}, P{0.0, 0.0};
        if (lane < MW) {
            const int end = min((lane + 1) * SUB, n_own);
            M = {ms[lane].mh, ms[lane].ml};
            P = dd_add({ms[lane].ph, ms[lane].pl}, dd_mul(M, (double)(n_own - end)));
        }
        M = row_dd_sum8(M);
        P = row_dd_sum8(P);
        if (lane == 7) out[blk] = {M.h, M.l, P.h, P.l};
    }
}

// b = dx^2 eps0_inv (charge + neutral) (EMSolver.cpp:157-167), its sums over
// entries >= 1, and the entry value of Ex0
template <int MW>
__global__ __launch_bounds__(SUB *MW) void k_pm_rhs(PoissonMB P) {
    constexpr int CHUNK = SUB * MW;
    __shared__ PmSum ms[MW];
    const vx_field_state &F = P.fs;
    const int N = F.n_f, i = blockIdx.x * CHUNK + threadIdx.x;
    double v = 0.0;
    if (i < N) {
        v = vx_eps0_inv * (F.charge[i] + F.neutral[i]);
        v *= F.dx2;
        P.W.b[i] = v;
    }
    pm_store_sums<MW>(i >= 1 ? v : 0.0, min(CHUNK, N - (int)blockIdx.x * CHUNK), P.sums_out, P.nb, ms);
    if (i == 0) *P.W.ex0 = *F.Ex0;
}

// MODE 0: first solve (x = c); 1: refinement (x += c); both then form the next
// residual.  MODE 2: last refinement, writes phi (x_out), Ex0 and E.
template <int MODE, int MW>
__global__ __launch_bounds__(64 * (MW + 5)) void k_pm_solve(PoissonMB P) {
    constexpr int CHUNK = SUB * MW, MT = 64 * (MW + 5);
    __shared__ double yw[CHUNK + 2 * CW];
    __shared__ double ys[YS];
    __shared__ double xw[CHUNK + 2 * HALO];
    __shared__ double cs[NSPEC];
    __shared__ PmSum ms[MW];
    const vx_field_state &F = P.fs;
    const int N = F.n_f, blk = blockIdx.x, lo = blk * CHUNK, nb = P.nb;
    const int n_own = min(CHUNK, N - lo);
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // this thread's entry of x (chunk and halo) and b, loaded ahead of their use
    const int j = threadIdx.x, gi = wrap(lo - HALO + j, N);
    const bool own = j >= HALO && j < n_own + HALO, have = j < n_own + 2 * HALO;
    const double xo = MODE > 0 && have ? P.x_in[gi] : 0.0;
    const double bv = MODE < 2 && j < n_own ? P.W.b[lo + j] : 0.0;
    double ps[NSPEC], ex0 = 0.0;  // MODE 2: x around entry 0, then phi; Ex0 on entry
    if (MODE == 2) {
#pragma unroll
        for (int k = 0; k < NSPEC; k++) ps[k] = P.x_in[wrap(k - 3, N)];
        ex0 = *P.W.ex0;
    }
    const PmSum *C = P.sums, *U = C + nb;  // chunks, sub-chunks
    // (sum v, sum v (pos - 1 - i)) of item q that ends at `end`, seen from pos
    auto item = [](const PmSum &q, int pos, int end, DD &t, DD &g) {
        const DD m{q.mh, q.ml};
        t = dd_add(t, m);
        g = dd_add(g, dd_add(dd_mul(m, (double)(pos - end)), {q.ph, q.pl}));
    };
    // the wavefront's sub-chunk: the chunk's, the neighbours' and those around entry
    // 0 (the last one may be shorter than the window, hence the one before it too);
    // none for some (s < 0 or s >= ns)
    const int ns = (N + SUB - 1) / SUB, s0 = blk * MW;
    const int s = w < MW ? s0 + w : w == MW ? s0 - 1 : w == MW + 1 ? s0 + MW : w == MW + 2 ? 0 : ns - (w - MW - 2);
    const int b = s / MW, i0 = s * SUB, i = i0 + lane;
    const bool sub = s >= 0 && s < ns;
    // what the steps below read from memory, all in flight at once
    const double in = sub && i < N ? P.in[i] : 0.0, in0 = P.in[0];
    PmSum u{0.0, 0.0, 0.0, 0.0};
    if (sub && lane < s - b * MW) u = U[b * MW + lane];
    // tail and d0 over every chunk (t, g), S and the sum of D before the sub-chunk (a, h)
    DD t{0.0, 0.0}, g{0.0, 0.0}, a{0.0, 0.0}, h{0.0, 0.0};
    for (int q = lane; q < nb; q += 64) {
        const PmSum c = C[q];
        item(c, N, min((q + 1) * CHUNK, N), t, g);
        if (q < b) item(c, i0, (q + 1) * CHUNK, a, h);
    }
    item(u, i0, (b * MW + lane + 1) * SUB, a, h);
    const DD tail = wave_dd_sum(t);
    g = wave_dd_sum(g);
    a = wave_dd_sum(a);
    h = wave_dd_sum(h);
    g = dd_add(g, dd_mul(tail, -(double)(N - 1)));
    const double d0 = (g.h + g.l) * P.invN, tl = tail.h + tail.l;
    if (sub) {  // y, into the windows it reaches
        a = dd_add(a, dd_neg(tail));
        h = dd_add(h, dd_mul(tail, -(double)(i0 - 1)));
        h = dd_add(dd_mul({d0, 0.0}, (double)(i0 - 1)), dd_neg(h));
        // (entry 0: S = 0, D = 0)
        const double S = s == 0 ? 0.0 : a.h + a.l, Y = s == 0 ? 0.0 : h.h + h.l;
        const double v = i == 0 ? -tl : in;
        const double Si = S + dpp_or_0<0x138>(wave_scan_dpp(v));
        const double Di = (i == 0 || i >= N) ? 0.0 : d0 - Si;
        const double y = Y + wave_scan_dpp(Di);
        if (i < N) {
            for (int img = -N; img <= N; img += N) {
                const int p = i + img - lo + CW;
                if (p >= 0 && p < n_own + 2 * CW) yw[p] = y;
            }
            const int e = i < N - i ? i + 3 + NG - 1 : i - N + 3 + NG - 1;
            if (e >= 0 && e < YS) ys[e] = y;
        }
    }
    __syncthreads();
    // M^-1 y at this thread's entry, and (by the last wavefront) around entry 0
    const double my = have ? conv_at(yw, j + NG - 1, P.g) : 0.0;
    const int e0 = (int)threadIdx.x - (MT - 64);
    if (e0 >= 0 && e0 < NSPEC) cs[e0] = conv_at(ys, e0 + NG - 1, P.g);
    __syncthreads();
    const double cp0 = cs[3];  // (M^-1 y)_0
    // row 0 (the approximate solve's last step): c_0 from c_1, c_2, c_{N-2}, c_{N-1}
    const double c0 = in0 - (((P.w1 * (cs[4] - cp0) + P.w2 * (cs[5] - cp0)) + P.w2 * (cs[1] - cp0)) +
                             P.w1 * (cs[2] - cp0));
    // x on the chunk and its halo
    if (have) {
        const double c = gi == 0 ? c0 : my - cp0;
        const double xn = MODE == 0 ? c : xo + c;
        xw[j] = xn;
        if (own) P.x_out[gi] = xn;
    }
    __syncthreads();
    if (MODE < 2) {
        // r = b - A x in double-double, rounded once (term order as the oracle's)
        double r = 0.0;
        const int i = lo + j, c = j + HALO;
        if (j < n_own) {
            double sh = bv, sl = 0.0;
            auto sub = [&](double a, double xv) { dd_sub(sh, sl, a, xv); };
            if (i == 0) {
                sub(1.0, xw[c]); sub(P.w1, xw[c + 1]); sub(P.w2, xw[c + 2]); sub(P.w2, xw[c - 2]);
                sub(P.w1, xw[c - 1]);
            } else {
                const double cf[5] = {P.w2, P.w1, P.w3, P.w1, P.w2};
                for (int d = -2; d <= 2; d++) {
                    if (wrap(i + d, N) == 0) continue;
                    sub(cf[d + 2], xw[c + d]);
                }
            }
            r = sh + sl;
            P.r_out[i] = r;
        }
        pm_store_sums<MW>(i >= 1 ? r : 0.0, n_own, P.sums_out, nb, ms);
    } else {
        // EMSolver.cpp:191: Ex0 += -(E(-1) + E(0)) * 0.5 with the entry Ex0, from phi
        // at N-3..N-1, 0..2 (recomputed here with the owners' operations)
#pragma unroll
        for (int k = 0; k < NSPEC; k++) ps[k] = ps[k] + (k == 3 ? c0 : cs[k] - cp0);
        const double fc = F.field_coef;
        const double e_m1 = -fc * (8 * (ps[3] - ps[1]) - ps[4] + ps[0]) + ex0;
        const double e_0 = -fc * (8 * (ps[4] - ps[2]) - ps[5] + ps[1]) + ex0;
        const double ex0n = ex0 + -(e_m1 + e_0) * 0.5;
        if (blk == 0 && threadIdx.x == 0) *F.Ex0 = ex0n;
        const int c = j + HALO;
        if (j < n_own) F.E[lo + j] = -fc * (8 * (xw[c + 1] - xw[c - 1]) - xw[c + 2] + xw[c - 2]) + ex0n;
    }
}

// ------------------------------------------------ multi-workgroup solve, n_f > PM_MAX
// The same steps with the sums, the scans and the convolution in launches of their
// own, 13 in all; chunks of 1024 entries:
//   k_pl_scan_s  S and the chunks' sums of S;
//   k_pl_scan_y  d0, D and y;
//   k_pl_conv    c, x, then the next residual and the chunks' sums of it, or phi, Ex0
//                and E.
// A sum across workgroups is formed from per-chunk partials that every workgroup
// reads and adds in the same order, so all of them hold the same bits.  The form in
// five launches forms sums over all chunks in every wavefront and a sub-chunk's y
// up to three times, which costs more than the launches it saves once a compute unit
// has more than one chunk: us on an MI355X, 5 / 13 launches, 131072 entries 45 / 71,
// 200000 88 / 77, 1000000 711 / 167, 4000000 8500 / 640.
constexpr int PL_T = 256, PL_PER = 4, PL_CHUNK = PL_T * PL_PER;
__host__ __device__ constexpr int pl_chunks(int n) { return (n + PL_CHUNK - 1) / PL_CHUNK; }

// Work layout (doubles): b | xa | xb | ra | rb | S | y | Pa[nb] | Pb[nb] | Ex0 on entry
struct PlWork {
    double *b, *xa, *xb, *ra, *rb, *S, *y, *Pa, *Pb, *ex0;
};
__host__ __device__ inline PlWork pl_work(double *w, int n) {
    const size_t N = n;
    const int nb = pl_chunks(n);
    PlWork W;
    W.b = w;
    W.xa = w + N;
    W.xb = w + 2 * N;
    W.ra = w + 3 * N;
    W.rb = w + 4 * N;
    W.S = w + 5 * N;
    W.y = w + 6 * N;
    W.Pa = w + 7 * N;
    W.Pb = W.Pa + nb;
    W.ex0 = W.Pb + nb;
    return W;
}

struct PoissonLong {
    vx_field_state fs;
    double w1, w2, w3;
    double g[NG];
    double invN;
    int nb;
    PlWork W;
    const double *in;    // right-hand side of this solve (b, then residuals)
    const double *x_in;  // x before this solve's correction
    double *x_out;       // x after it
    double *r_out;       // next residual
};

__device__ __forceinline__ double wave_incl_scan(double v) {
    const int lane = threadIdx.x & 63;
    for (int off = 1; off < 64; off <<= 1) {
        double t = __shfl_up(v, off, 64);
        if (lane >= off) v += t;
    }
    return v;
}

__device__ __forceinline__ double wave_sum(double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// sum of v[lo..hi) in a fixed order; every lane of every wave gets the same bits
__device__ __forceinline__ double wave_range_sum(const double *v, int lo, int hi) {
    double s = 0.0;
    for (int k = lo + (threadIdx.x & 63); k < hi; k += 64) s += v[k];
    return wave_sum(s);
}

__device__ __forceinline__ double pl_sum(double v, double *lds) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    v = wave_sum(v);
    if (lane == 0) lds[w] = v;
    __syncthreads();
    double r = ((lds[0] + lds[1]) + lds[2]) + lds[3];
    __syncthreads();
    return r;
}

// exclusive prefix of the per-thread totals over the workgroup
__device__ __forceinline__ double pl_offset(double tot, double *lds) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    double inc = wave_incl_scan(tot);
    double exc = __shfl_up(inc, 1, 64);
    if (lane == 0) exc = 0.0;
    if (lane == 63) lds[w] = inc;
    __syncthreads();
    double off = 0.0;
    for (int k = 0; k < w; k++) off += lds[k];
    __syncthreads();
    return off + exc;
}

// b = dx^2 eps0_inv (charge + neutral) (EMSolver.cpp:157-167), its chunk sums
// over entries >= 1, and the entry value of Ex0
__global__ __launch_bounds__(PL_T) void k_pl_rhs(PoissonLong P) {
    __shared__ double lds[PL_T / 64];
    const vx_field_state &F = P.fs;
    const int N = F.n_f, base = blockIdx.x * PL_CHUNK + threadIdx.x * PL_PER;
    const double te = vx_eps0_inv;
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < PL_PER; k++) {
        const int i = base + k;
        if (i < N) {
            double v = te * (F.charge[i] + F.neutral[i]);
            v *= F.dx2;
            P.W.b[i] = v;
            if (i >= 1) s += v;
        }
    }
    const double tot = pl_sum(s, lds);
    if (threadIdx.x == 0) {
        P.W.Pa[blockIdx.x] = tot;
        if (blockIdx.x == 0) *P.W.ex0 = *F.Ex0;
    }
}

__global__ __launch_bounds__(PL_T) void k_pl_scan_s(PoissonLong P) {
    __shared__ double lds[PL_T / 64];
    const int N = P.fs.n_f, blk = blockIdx.x, base = blk * PL_CHUNK + threadIdx.x * PL_PER;
    const double tail = wave_range_sum(P.W.Pa, 0, P.nb);
    // S at the chunk's first entry: v'_0 = -tail plus the entries >= 1 before the chunk
    const double start = blk == 0 ? 0.0 : -tail + wave_range_sum(P.W.Pa, 0, blk);
    double e[PL_PER], tot = 0.0;
#pragma unroll
    for (int k = 0; k < PL_PER; k++) {
        const int i = base + k;
        e[k] = (i == 0) ? -tail : (i < N ? P.in[i] : 0.0);
        tot += e[k];
    }
    double run = start + pl_offset(tot, lds);
    double ssum = 0.0;
#pragma unroll
    for (int k = 0; k < PL_PER; k++) {
        const int i = base + k;
        if (i < N) {
            P.W.S[i] = run;
            ssum += run;
        }
        run += e[k];
    }
    const double t2 = pl_sum(ssum, lds);
    if (threadIdx.x == 0) P.W.Pb[blk] = t2;
}

__global__ __launch_bounds__(PL_T) void k_pl_scan_y(PoissonLong P) {
    __shared__ double lds[PL_T / 64];
    const int N = P.fs.n_f, blk = blockIdx.x, base = blk * PL_CHUNK + threadIdx.x * PL_PER;
    const double d0 = wave_range_sum(P.W.Pb, 0, P.nb) * P.invN;
    // sum of D over the earlier chunks: (entries - [chunk 0]) * d0 - (chunk sum of S)
    double sd = 0.0;
    for (int k = threadIdx.x & 63; k < blk; k += 64) {
        const int n = min(PL_CHUNK, N - k * PL_CHUNK) - (k == 0 ? 1 : 0);
        sd += (double)n * d0 - P.W.Pb[k];
    }
    const double offD = wave_sum(sd);
    double D[PL_PER], tot = 0.0;
#pragma unroll
    for (int k = 0; k < PL_PER; k++) {
        const int i = base + k;
        D[k] = (i == 0 || i >= N) ? 0.0 : d0 - P.W.S[i];
        tot += D[k];
    }
    double run = offD + pl_offset(tot, lds);
#pragma unroll
    for (int k = 0; k < PL_PER; k++) {
        const int i = base + k;
        run += D[k];
        if (i < N) P.W.y[i] = run;
    }
}

// MODE 0: first solve (x = c); 1: refinement (x += c); both then form the next
// residual.  MODE 2: last refinement, writes phi (x_out), Ex0 and E.
template <int MODE>
__global__ __launch_bounds__(PL_T) void k_pl_conv(PoissonLong P) {
    __shared__ double yw[PL_CHUNK + 2 * CW];
    __shared__ double ys[NSPEC + 2 * (NG - 1)];
    __shared__ double xw[PL_CHUNK + 2 * HALO];
    __shared__ double cs[NSPEC];
    __shared__ double lds[PL_T / 64];
    const vx_field_state &F = P.fs;
    const int N = F.n_f, blk = blockIdx.x, lo = blk * PL_CHUNK;
    const int n_own = min(PL_CHUNK, N - lo);
    const double *y = P.W.y;
    for (int j = threadIdx.x; j < n_own + 2 * CW; j += PL_T) yw[j] = y[wrap(lo - CW + j, N)];
    for (int j = threadIdx.x; j < NSPEC + 2 * (NG - 1); j += PL_T) ys[j] = y[wrap(-3 - (NG - 1) + j, N)];
    __syncthreads();
    if (threadIdx.x < NSPEC) cs[threadIdx.x] = conv_at(ys, threadIdx.x + NG - 1, P.g);
    __syncthreads();
    const double cp0 = cs[3];  // (M^-1 y)_0
    // row 0 (the approximate solve's last step): c_0 from c_1, c_2, c_{N-2}, c_{N-1}
    const double c0 = P.in[0] - (((P.w1 * (cs[4] - cp0) + P.w2 * (cs[5] - cp0)) + P.w2 * (cs[1] - cp0)) +
                                 P.w1 * (cs[2] - cp0));
    // x on the chunk and its halo
    for (int j = threadIdx.x; j < n_own + 2 * HALO; j += PL_T) {
        const int gi = wrap(lo - HALO + j, N);
        const double c = (gi == 0) ? c0 : conv_at(yw, j + NG - 1, P.g) - cp0;
        const double xn = MODE == 0 ? c : P.x_in[gi] + c;
        xw[j] = xn;
        if (j >= HALO && j < n_own + HALO) P.x_out[gi] = xn;
    }
    __syncthreads();
    if (MODE < 2) {
        // r = b - A x in double-double, rounded once (term order as the oracle's)
        double s = 0.0;
        for (int j = threadIdx.x; j < n_own; j += PL_T) {
            const int i = lo + j, c = j + HALO;
            double sh = P.W.b[i], sl = 0.0;
            auto sub = [&](double a, double xv) { dd_sub(sh, sl, a, xv); };
            if (i == 0) {
                sub(1.0, xw[c]); sub(P.w1, xw[c + 1]); sub(P.w2, xw[c + 2]); sub(P.w2, xw[c - 2]);
                sub(P.w1, xw[c - 1]);
            } else {
                const double cf[5] = {P.w2, P.w1, P.w3, P.w1, P.w2};
                for (int d = -2; d <= 2; d++) {
                    if (wrap(i + d, N) == 0) continue;
                    sub(cf[d + 2], xw[c + d]);
                }
            }
            const double r = sh + sl;
            P.r_out[i] = r;
            if (i >= 1) s += r;
        }
        const double tot = pl_sum(s, lds);
        if (threadIdx.x == 0) P.W.Pa[blk] = tot;
    } else {
        // EMSolver.cpp:191: Ex0 += -(E(-1) + E(0)) * 0.5 with the entry Ex0, from phi
        // at N-3..N-1, 0..2 (recomputed here with the owners' operations)
        double ps[NSPEC];
#pragma unroll
        for (int k = 0; k < NSPEC; k++) {
            const int gi = wrap(k - 3, N);
            ps[k] = P.x_in[gi] + (k == 3 ? c0 : cs[k] - cp0);
        }
        const double ex0 = *P.W.ex0, fc = F.field_coef;
        const double e_m1 = -fc * (8 * (ps[3] - ps[1]) - ps[4] + ps[0]) + ex0;
        const double e_0 = -fc * (8 * (ps[4] - ps[2]) - ps[5] + ps[1]) + ex0;
        const double ex0n = ex0 + -(e_m1 + e_0) * 0.5;
        if (blk == 0 && threadIdx.x == 0) *F.Ex0 = ex0n;
        for (int j = threadIdx.x; j < n_own; j += PL_T) {
            const int c = j + HALO;
            F.E[lo + j] = -fc * (8 * (xw[c + 1] - xw[c - 1]) - xw[c + 2] + xw[c - 2]) + ex0n;
        }
    }
}

// Single-workgroup variant for n_f <= SMALL_MAX: thread t owns the CH
// consecutive entries [t*CH, t*CH + CH) in registers; neighbours come from an
// LDS copy of the vector with a periodic halo of VH entries on either side, so
// no stencil or recurrence needs index wrapping.
//
// M^-1 = C (1 - rho S^-1)^-1 (1 - rho S)^-1 with C = 12 rho / (1 - rho^2), so
// (M^-1 y)_i = C (u_i + v_i - y_i) with the first-order recurrences
// u_i = y_i + rho u_{i-1} and v_i = y_i + rho v_{i+1}.  Each thread runs them
// over its entries after VH warm-up entries (rho^17 < 4e-20, the reach of the
// convolution the multi-workgroup variant uses).  The approximate solve only
// has to be accurate: the refinement rounds take x to the correctly rounded
// solution whatever the rounding inside it.
//
// Barriers: a workgroup scan exchanges the wavefront partials through LDS once
// (one barrier); every thread then forms the same sums of the partials itself.
// Consecutive exchanges alternate between two partial buffers, so a buffer is
// rewritten only after a later barrier has ordered every read of it.
//
// Rounds of refinement: one leaves a fraction q of the error, because of the
// prefix sums' rounding and because the factors are not quite those of the
// matrix, whose coefficients are rounded (w3 + 2 w1 + 2 w2 = 1.4e-16, not 0,
// against a smallest eigenvalue near (pi / n)^2).  Up to n_f = 4096 q is near
// 1e-9, so two rounds leave what a third one leaves, the rounded solution:
// against exact solutions of 127 smooth, rough, sparse and wide-ranging right-hand
// sides (8 to 4096 entries) the same entries, 1 in 30000, were an ulp off after
// either.  At 32768 entries two rounds leave 1 or 2 ulps where phi is near 0, so
// the multi-workgroup solve keeps three.
//
// Bound by the chain of scans, recurrences, residuals and barriers; from n_f =
// 2048 also by FP64 issue on the one CU.  Measured on an MI355X, us at n_f = 64,
// 512, 1024, 2048 and 4096: 10.1, 11.3, 12.9, 17.9 and 24.8 with eight wavefronts
// at every size, three rounds and the sums apart from the scans; 4.9, 7.1, 8.8,
// 12.0 and 17.4 as it is.
constexpr int PW1 = 8;               // most wavefronts of the single-workgroup solve
constexpr int SMALL_MAX = 4096;      // largest n_f it serves
constexpr int SOLVES = 3;            // the first and two rounds of refinement
constexpr int VH = NG - 1;           // periodic halo of the LDS copy

constexpr int VLEN = SMALL_MAX + 2 * VH + 8;  // positions of the LDS copy
constexpr int VDUMMY = VLEN - VH;             // at(VDUMMY): a slot past them, written only

struct SmallLds {
    // at(j) = vec[j mod N] for j in [-VH, N + VH); the 8 positions after that
    // are 0 (the last thread's backward recurrence may start there).  Position
    // p = VH + j is stored at p + p / 8: a thread reads 8 consecutive entries
    // per step of its loops, and the pad after every 8 puts the lanes of a
    // wavefront (9 doubles apart) in different LDS banks.
    double v[(VLEN + 1) + (VLEN + 1) / 8 + 1];
    double part[2][PW1];  // wavefront partials, alternating
    double edge[5];       // c at entries 0, 1, 2, N-2, N-1 (row 0 of the matrix)
    __device__ __forceinline__ double &at(int j) {
        const int p = VH + j;
        return v[p + (p >> 3)];
    }
};

// Workgroup exclusive scan of the per-thread totals in thread order, and their
// sum (the same bits in every thread).
template <int W>
__device__ __forceinline__ double block_excl_scan1(double tot, double (&part)[2][PW1], int &buf, double &sum) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const double inc = wave_scan_dpp(tot);
    const double exc = dpp_or_0<0x138>(inc);  // wave_shr:1: lane l - 1's inclusive sum, 0 at lane 0
    if (W == 1) {
        __syncthreads();
        sum = lane63(inc);
        return exc;
    }
    if (lane == 63) part[buf][w] = inc;
    __syncthreads();
    double off = 0.0, all = 0.0;
#pragma unroll
    for (int k = 0; k < W; k++) {
        if (k == w) off = all;
        all += part[buf][k];
    }
    buf ^= 1;
    sum = all;
    return off + exc;
}

// The thread's entries into the LDS copy, with their periodic images in the
// halo.  For N >= 2 VH an entry has at most one image (i + N for i < VH,
// i - N for i >= N - VH), stored without a branch (an entry without an image
// stores itself twice); below that (N >= 8) the images are looped over, a
// branch the whole workgroup takes alike.
template <int CH>
__device__ __forceinline__ void put_periodic(SmallLds &L, const double *val, int N, int base) {
    if (N >= 2 * VH) {
#pragma unroll
        for (int k = 0; k < CH; k++) {
            const int i = base + k;
            if (i < N) {
                const int q = i < VH ? i + N : (i >= N - VH ? i - N : i);
                L.at(i) = val[k];
                L.at(q) = val[k];
            }
        }
        return;
    }
#pragma unroll
    for (int k = 0; k < CH; k++) {
        const int i = base + k;
        if (i >= N) continue;
        L.at(i) = val[k];
        for (int q = i - N; q >= -VH; q -= N) L.at(q) = val[k];
        for (int q = i + N; q < N + VH; q += N) L.at(q) = val[k];
    }
}

// One approximate solve of A out = in: S_i = sum_{1<=k<i} in_k - tail (tail the
// sum over k >= 1, S_0 = 0), d0 = mean(S), y_i = sum_{1<=k<=i} (d0 - S_k) = i d0 -
// T_i with T the inclusive prefix of S, c = M^-1 y - (M^-1 y)_0, and c_0 from row
// 0 of the matrix.  Each prefix sum's exchange also gives the sum.
template <int CH, int W>
__device__ void approx_one(const PoissonArgs &P, const double *in, double *out, SmallLds &L, int &buf) {
    const int N = P.fs.n_f;
    const int base = threadIdx.x * CH;
    double rp[CH], tot = 0.0, tail, ssum;
#pragma unroll
    for (int k = 0; k < CH; k++) {
        rp[k] = base + k >= 1 && base + k < N ? in[k] : 0.0;
        tot += rp[k];
    }
    double run = block_excl_scan1<W>(tot, L.part, buf, tail);
    run -= tail;
    double y[CH];
    tot = 0.0;
#pragma unroll
    for (int k = 0; k < CH; k++) {
        if (base + k >= 1 && base + k < N) tot += run;
        y[k] = tot;
        run += rp[k];
    }
    run = block_excl_scan1<W>(tot, L.part, buf, ssum);
    const double d0 = ssum * P.invN;
#pragma unroll
    for (int k = 0; k < CH; k++) y[k] = (double)(base + k) * d0 - (run + y[k]);
    // (every thread's reads of L.v before this solve came before its first
    // barrier above)
    put_periodic<CH>(L, y, N, base);
    __syncthreads();
    double cp[CH];
    if (base < N) {
        const double rho = P.rho;
        double fw[CH], bw[CH];
        double u = L.at(base - VH);
#pragma unroll
        for (int m = 1; m < VH; m++) u = fma(rho, u, L.at(base - VH + m));
#pragma unroll
        for (int k = 0; k < CH; k++) {
            u = fma(rho, u, L.at(base + k));
            fw[k] = u;
        }
        double b = L.at(base + CH - 1 + VH);
#pragma unroll
        for (int m = VH - 1; m >= 1; m--) b = fma(rho, b, L.at(base + CH - 1 + m));
#pragma unroll
        for (int k = CH - 1; k >= 0; k--) {
            b = fma(rho, b, L.at(base + k));
            bw[k] = b;
        }
#pragma unroll
        for (int k = 0; k < CH; k++) cp[k] = base + k < N ? P.C * ((fw[k] + bw[k]) - y[k]) : 0.0;
    } else {
#pragma unroll
        for (int k = 0; k < CH; k++) cp[k] = 0.0;
    }
    // row 0 needs c at entries 0, 1, 2, N-2 and N-1 (N >= 8: distinct)
#pragma unroll
    for (int k = 0; k < CH; k++) {
        const int i = base + k;
        const int e = i < 3 ? i : (i == N - 2 ? 3 : (i == N - 1 ? 4 : -1));
        if (e >= 0) L.edge[e] = cp[k];
    }
    __syncthreads();
    const double c0 = L.edge[0];
#pragma unroll
    for (int k = 0; k < CH; k++) out[k] = (base + k > 0) ? cp[k] - c0 : cp[k];
    if (threadIdx.x == 0) {
        const double y1 = L.edge[1] - c0, y2 = L.edge[2] - c0, yn2 = L.edge[3] - c0, yn1 = L.edge[4] - c0;
        out[0] = in[0] - (((P.w1 * y1 + P.w2 * y2) + P.w2 * yn2) + P.w1 * yn1);
    }
}

// r = b - A x with a double-double accumulation of the reference's
// coefficients (rows 1..N-1: the periodic stencil without column 0; row 0:
// x_0 + w1 x_1 + w2 x_2 + w2 x_{N-2} + w1 x_{N-1})
template <int CH>
__device__ void residual_one(const PoissonArgs &P, const double *b, const double *x, double *r, SmallLds &L) {
    const int N = P.fs.n_f;
    const int base = threadIdx.x * CH;
    put_periodic<CH>(L, x, N, base);
    __syncthreads();
    // x at entries base - 2 .. base + CH + 1, read at once (inside the LDS
    // array for every thread; entries >= N are not used)
    double w[CH + 4];
#pragma unroll
    for (int m = 0; m < CH + 4; m++) w[m] = L.at(base - 2 + m);
    const double cf[5] = {P.w2, P.w1, P.w3, P.w1, P.w2};
#pragma unroll
    for (int k = 0; k < CH; k++) {
        const int i = base + k;
        // rows i >= 1: neighbours j = i + d in [-1, N + 1]; column 0 (j = 0 or
        // j = N) gets a zero coefficient, which changes neither sum
        double sh = b[k], sl = 0.0;
#pragma unroll
        for (int d = -2; d <= 2; d++) {
            const int j = i + d;
            dd_sub(sh, sl, (j == 0 || j == N) ? 0.0 : cf[d + 2], w[k + d + 2]);
        }
        r[k] = i < N ? sh + sl : 0.0;
    }
    if (base == 0) {  // row 0
        double sh = b[0], sl = 0.0;
        dd_sub(sh, sl, 1.0, L.at(0));
        dd_sub(sh, sl, P.w1, L.at(1));
        dd_sub(sh, sl, P.w2, L.at(2));
        dd_sub(sh, sl, P.w2, L.at(N - 2));
        dd_sub(sh, sl, P.w1, L.at(N - 1));
        r[0] = sh + sl;
    }
}

template <int CH, int W>
__global__ __launch_bounds__(64 * W) void k_poisson_one(PoissonArgs P) {
    const vx_field_state &F = P.fs;
    const int N = F.n_f;
    constexpr int PT1 = 64 * W;
    const int t = threadIdx.x, base = t * CH;
    __shared__ SmallLds L;
    int buf = 0;
    // the entries past the last image, where the last thread's backward
    // recurrence may start, hold 0 (never written again)
    if (t < 8) L.at(N + VH + t) = 0.0;
    double b[CH], x[CH], r[CH], c[CH];
    const double te = vx_eps0_inv;
    // the right-hand side formed at entries t + PT1 m (coalesced loads, at
    // clamped indices, all in flight at once) and handed to the owners of
    // consecutive entries through the LDS copy
    double chv[CH], nev[CH];
#pragma unroll
    for (int m = 0; m < CH; m++) {
        const int i = min(t + PT1 * m, N - 1);
        chv[m] = F.charge[i];
        nev[m] = F.neutral[i];
    }
    // the entry Ex0 (written back at the end) as a vector load behind them,
    // so that its latency overlaps theirs (a scalar load would be waited for
    // before them)
    const double ex0 = __builtin_bit_cast(
        double, __builtin_amdgcn_raw_buffer_load_b64(
                    __builtin_amdgcn_make_buffer_rsrc(F.Ex0, 0, 8, 0x00020000), 0, 0, 0));
#pragma unroll
    for (int m = 0; m < CH; m++) {
        const int i = t + PT1 * m;
        double v = te * (chv[m] + nev[m]);
        v *= F.dx2;
        L.at(i < N ? i : VDUMMY) = v;  // no branch around the loads' use
    }
    __syncthreads();
    // (these reads come before the first barrier of the first solve, which
    // writes the LDS copy only after it)
#pragma unroll
    for (int k = 0; k < CH; k++) {
        b[k] = base + k < N ? L.at(base + k) : 0.0;
        x[k] = 0.0;
    }
    // the approximate solve of b, then two rounds of refinement (residual r
    // of x, x += the approximate solve of r), as one loop: the kernel runs
    // once per field solve and its code is fetched cold, so one copy of each
    // step is fetched once and then reused
#pragma nounroll
    for (int it = 0; it < SOLVES; it++) {
        if (it > 0) {
            // the previous solve's last barrier ordered its reads of L.v
            residual_one<CH>(P, b, x, r, L);
        } else {
#pragma unroll
            for (int k = 0; k < CH; k++) r[k] = b[k];
        }
        // the first barrier of the solve below orders the residual's reads of
        // L.v before the solve writes it
        approx_one<CH, W>(P, r, c, L, buf);
#pragma unroll
        for (int k = 0; k < CH; k++) x[k] = it == 0 ? c[k] : x[k] + c[k];
    }
    // phi and E from the final potential (EMSolver.cpp:137-154, 191), stored
    // at entries t + PT1 m (coalesced) from the LDS copy: every thread's reads
    // of it in the last solve came before its final barrier
    put_periodic<CH>(L, x, N, base);
    __syncthreads();
    const double fc = F.field_coef;
    auto ef = [&](double e0, double pm2, double pm1, double pp1, double pp2) {
        return -fc * (8 * (pp1 - pm1) - pp2 + pm2) + e0;
    };
    const double e_m1 = ef(ex0, L.at(-3), L.at(-2), L.at(0), L.at(1)), e_0 = ef(ex0, L.at(-2), L.at(-1), L.at(1), L.at(2));
    const double ex0n = ex0 + -(e_m1 + e_0) * 0.5;
    if (t == 0) *F.Ex0 = ex0n;
#pragma unroll
    for (int m = 0; m < CH; m++) {
        const int i = t + PT1 * m;
        if (i < N) {
            F.phi[i] = L.at(i);
            F.E[i] = ef(ex0n, L.at(i - 2), L.at(i - 1), L.at(i + 1), L.at(i + 2));
        }
    }
}

// ---------------------------------------------------------------- Maxwell
struct MaxArgs {
    vx_field_state fs;
    int step;
    double by0, bz0;
    const double *drive;  // when set, by0 = drive[0] and bz0 = drive[1] in device memory
    double dx_inv;
    double a[6], b[6];
};

__device__ __forceinline__ int fidx(int ne, int i, int slot) { return slot * ne + i; }

// Above MX1 elements a field stage is two launches (three, with the faces apart, took 12.6 us at
// 4096 elements on an MI355X, these 8.9): the right-hand sides, which read
// slot 1 at the neighbouring elements and write slot step + 2, then the update
// of slot 1 and A^2 at the faces from it.  A face's four potentials are formed
// again from the update's inputs rather than read from slot 1, which the launch
// writes: those inputs (slots 0 and 2..step + 2) are not written by it.  At the
// last stage, whose update reads slot 1, the first launch forms the new value
// into slot 0 (which nothing reads any more) and the second copies it.

// EMSolver.cpp:479-553; blockIdx.y = 0: By, Ez, Az; 1: Bz, Ey, Ay (each set
// reads only itself)
__device__ __forceinline__ double maxwell_last(const double *y, int ne, int i, const double *b, double k5) {
    double t = y[fidx(ne, i, 1)] + b[0] * y[fidx(ne, i, 2)];
#pragma unroll
    for (int k = 1; k < 5; k++) t = t + b[k] * y[fidx(ne, i, k + 2)];
    return t + b[5] * k5;
}

// The right-hand sides of element i of a set (z: By, Ez, Az; else Bz, Ey, Ay)
__device__ __forceinline__ void maxwell_rhs(const MaxArgs &A, bool z, const double *B, const double *E, const double *V,
                                            int i, double &rB, double &rE, double &rV) {
    const vx_field_state &F = A.fs;
    const int ne = F.n_e, npre = F.n_prepad, N = F.n_f;
    const int i1 = fidx(ne, i, 1);
    const double dx_inv = A.dx_inv, db = z ? dx_inv : -dx_inv, de = z ? dx_inv : -dx_inv;
    rB = rE = rV = 0;
    if (i == 0) {
        const double b0 = z ? (A.drive ? A.drive[0] : A.by0) : (A.drive ? A.drive[1] : A.bz0);
        rB = db * (E[i1 + 1] - E[i1]);
        rE = de * (B[i1] - b0) * vx_eps0_inv * vx_mu_inv;
        rV = -E[i1];
    } else if (i < npre || (i >= npre + N && i < ne - 2)) {
        rB = db * (E[i1 + 1] - E[i1]);
        rE = de * (B[i1] - B[i1 - 1]) * vx_eps0_inv * vx_mu_inv;
        rV = -E[i1];
    } else if (i >= npre && i < npre + N) {
        const double c1 = -1.0 / 24;
        const double c2 = 9.0 / 8.0;
        const double Jc = F.J[i - npre];
        rB = db * (c1 * (E[i1 + 2] - E[i1 - 1]) + c2 * (E[i1 + 1] - E[i1]));
        rE = de * (c1 * (B[i1 + 1] - B[i1 - 2]) + c2 * (B[i1] - B[i1 - 1])) * vx_eps0_inv * vx_mu_inv -
             vx_eps0_inv * Jc * V[i1];
        rV = -E[i1];
    }
}

__global__ __launch_bounds__(256) void k_maxwell_rhs(MaxArgs A) {
    const vx_field_state &F = A.fs;
    const int ne = F.n_e;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ne) return;
    const bool z = blockIdx.y == 0;
    double *B = z ? F.By : F.Bz, *E = z ? F.Ez : F.Ey, *V = z ? F.Az : F.Ay;
    double rB, rE, rV;
    maxwell_rhs(A, z, B, E, V, i, rB, rE, rV);
    const int s = fidx(ne, i, A.step + 2);
    B[s] = rB;
    E[s] = rE;
    V[s] = rV;
    if (A.step == 5) {
        B[fidx(ne, i, 0)] = maxwell_last(B, ne, i, A.b, rB);
        E[fidx(ne, i, 0)] = maxwell_last(E, ne, i, A.b, rE);
        V[fidx(ne, i, 0)] = maxwell_last(V, ne, i, A.b, rV);
    }
}

// Slot 1 of element i after the stage's update (EMSolver.cpp:204-338)
__device__ __forceinline__ double maxwell_new(const double *y, const MaxArgs &A, int ne, int i) {
    if (A.step > 4) return y[fidx(ne, i, 0)];
    double t = y[fidx(ne, i, 0)] + A.a[0] * y[fidx(ne, i, 2)];
    for (int k = 1; k <= A.step; k++) t = t + A.a[k] * y[fidx(ne, i, k + 2)];
    return t;
}

// The update, one thread per element and field (blockIdx.y 0..3: By, Bz, Ey,
// Ez), and at blockIdx.y = 4 Ay, Az and A^2 at the faces (EMSolver.cpp:555-619;
// a_squared[n_f] is never written by the reference)
constexpr int MXT = 256;
__global__ __launch_bounds__(MXT) void k_maxwell_update(MaxArgs A) {
    const vx_field_state &F = A.fs;
    const int ne = F.n_e, e0 = blockIdx.x * MXT, i = e0 + (int)threadIdx.x;
    const int v = blockIdx.y;
    if (v < 4) {
        if (i >= ne) return;
        double *y = v == 0 ? F.By : v == 1 ? F.Bz : v == 2 ? F.Ey : F.Ez;
        y[fidx(ne, i, 1)] = maxwell_new(y, A, ne, i);
        return;
    }
    __shared__ double ay[MXT + 3], az[MXT + 3];  // elements e0 - 2 .. e0 + MXT
    for (int k = threadIdx.x; k < MXT + 3; k += MXT) {
        const int e = e0 - 2 + k;
        if (e < 0 || e >= ne) continue;
        const double y = maxwell_new(F.Ay, A, ne, e), z = maxwell_new(F.Az, A, ne, e);
        ay[k] = y;
        az[k] = z;
        if (k >= 2 && k < MXT + 2) {
            F.Ay[fidx(ne, e, 1)] = y;
            F.Az[fidx(ne, e, 1)] = z;
        }
    }
    __syncthreads();
    const int face = i - F.n_prepad, k = (int)threadIdx.x;
    if (face < 0 || face >= F.n_f) return;
    const double y = face_weno(ay[k], ay[k + 1], ay[k + 2], ay[k + 3]);
    const double z = face_weno(az[k], az[k + 1], az[k + 2], az[k + 3]);
    F.a2[face] = (y * y) + (z * z);
}

// The whole stage in one workgroup, for at most MX1 elements: a thread forms the
// right-hand sides and new values of an element of its set from slot 1, which is
// written only after a barrier has ordered every read of it, then A^2 at the
// faces from the new potentials in LDS.  Bound by launch latency: one launch for
// two.  us a stage on an MI355X, this / the two launches: 4.4 / 8.0 at 64 cells,
// 4.5 to 5.2 / 8.0 at 256, 4.7 to 6.1 / 8.2 at 508; two elements a thread took 6.0
// to 8.3 / 8.1 at 700, 7.1 to 10.6 / 8.1 at 1020.
constexpr int MX1 = 512;
__global__ __launch_bounds__(2 * MX1) void k_maxwell_one(MaxArgs A) {
    const vx_field_state &F = A.fs;
    const int ne = F.n_e;
    const bool z = threadIdx.x < MX1;  // uniform per wavefront
    const int i = (int)threadIdx.x & (MX1 - 1);
    double *B = z ? F.By : F.Bz, *E = z ? F.Ez : F.Ey, *V = z ? F.Az : F.Ay;
    __shared__ double pot[2][MX1];  // the new Ay, Az
    double nB, nE, nV;
    // slot 1 after the update, from the right-hand side and the slots before it
    auto fresh = [&](const double *y, double r) {
        if (A.step > 4) return maxwell_last(y, ne, i, A.b, r);
        double v = y[fidx(ne, i, 0)];
        for (int k = 0; k < A.step; k++) v = v + A.a[k] * y[fidx(ne, i, k + 2)];
        return v + A.a[A.step] * r;
    };
    if (i < ne) {
        double rB, rE, rV;
        maxwell_rhs(A, z, B, E, V, i, rB, rE, rV);
        nB = fresh(B, rB);
        nE = fresh(E, rE);
        nV = fresh(V, rV);
        const int s = fidx(ne, i, A.step + 2);
        B[s] = rB;
        E[s] = rE;
        V[s] = rV;
        pot[z][i] = nV;
    }
    __syncthreads();
    if (i < ne) {
        const int s = fidx(ne, i, 1);
        B[s] = nB;
        E[s] = nE;
        V[s] = nV;
        if (A.step > 4) {
            B[i] = nB;
            E[i] = nE;
            V[i] = nV;
        }
    }
    const int face = threadIdx.x;
    if (face >= F.n_f) return;
    const int e = face + F.n_prepad - 2;
    const double y = face_weno(pot[0][e], pot[0][e + 1], pot[0][e + 2], pot[0][e + 3]);
    const double v = face_weno(pot[1][e], pot[1][e + 1], pot[1][e + 2], pot[1][e + 3]);
    F.a2[face] = (y * y) + (v * v);
}

// a2_0 and E at the start of a step, in one launch
__global__ __launch_bounds__(256) void k_snapshot(vx_field_state F, double *E0, double *a20) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < F.n_f) E0[i] = F.E[i];
    if (i <= F.n_f) a20[i] = F.a2[i];
}

__global__ void k_neutralize(vx_field_state F) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= F.n_f) return;
    F.J[i] = 0.0;
    F.neutral[i] = -F.charge[i];
}

// ------------------------------------------------ fixed work array of vx_poisson_noalloc
// The multi-workgroup solve's work vector (pm_work layout) for n_f up to
// VX_POISSON_NOALLOC_MAX_NF: 3.67 MB that each GPU the library runs on holds
// until the process ends.  Host code never uses this name as an address: the
// device address comes from hipGetSymbolAddress, once per device, with that
// device current (scratch_address, at context creation).
__host__ __device__ constexpr size_t pm_work_elems(int n) { return 7 * (size_t)n + 2 * (((size_t)n + 1023) / 1024) + 1; }
constexpr size_t NOALLOC_WORK = pm_work_elems(VX_POISSON_NOALLOC_MAX_NF);
// pl_work's layout, whose size pm_work's 5 n + 1 doubles and 8 (1 + MW) per chunk of
// sums stay below for every n that they serve
constexpr bool pm_fits(int n) {
    return 5 * (size_t)n + 1 + (size_t)pm_chunks(n) * 2 * 4 * (1 + pm_mw(n)) <= pm_work_elems(n);
}
static_assert(pm_fits(4097) && pm_fits(PM_SMALL) && pm_fits(PM_SMALL + 1) && pm_fits(PM_MAX), "work array");
static_assert(2 * SUB > 2 * 4 * 2, "sums per sub-chunk (and its share of its chunk's) against 2 doubles per entry");
static __device__ __align__(256) double scratch[NOALLOC_WORK];
constexpr int MAX_DEVICES = 64;
static std::mutex scratch_mu;
static double *scratch_ptr[MAX_DEVICES] = {};

int validate_fs(vx_ctx *ctx, const vx_field_state *fs) {
    if (!fs) return fail(ctx, VX_EINVAL, "null field state");
    if (fs->n_f < 8 || fs->n_prepad < 2 || fs->n_postpad < 2 ||
        fs->n_e != fs->n_f + fs->n_prepad + fs->n_postpad)
        return fail(ctx, VX_EINVAL, "bad field sizes n_f=%d pre=%d post=%d n_e=%d", fs->n_f,
                    fs->n_prepad, fs->n_postpad, fs->n_e);
    return VX_OK;
}

}  // namespace

// Called by vx_ctx_create with ctx->device current: the device address of
// this GPU's fixed work array (looked up once per device), or a recorded error.
int vx_noalloc_scratch_init(vx_ctx *ctx) {
    std::lock_guard<std::mutex> lock(scratch_mu);
    if (ctx->device < 0 || ctx->device >= MAX_DEVICES) return VX_EINVAL;
    if (!scratch_ptr[ctx->device]) {
        void *p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            ctx->err = std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
            return VX_EHIP;
        }
        scratch_ptr[ctx->device] = (double *)p;
    }
    ctx->poisson_scratch = scratch_ptr[ctx->device];
    return VX_OK;
}

extern "C" {

size_t vx_field_work_elems(int32_t n_f) { return pm_work_elems(n_f); }

static int poisson_long(vx_ctx *ctx, const PoissonArgs &P, double *work) {
    PoissonLong M;
    M.fs = P.fs;
    M.w1 = P.w1;
    M.w2 = P.w2;
    M.w3 = P.w3;
    for (int k = 0; k < NG; k++) M.g[k] = P.g[k];
    M.invN = P.invN;
    M.nb = pl_chunks(P.fs.n_f);
    M.W = pl_work(work, P.fs.n_f);
    const PlWork &W = M.W;
    const unsigned nb = (unsigned)M.nb;
    k_pl_rhs<<<nb, PL_T, 0, ctx->stream>>>(M);
    // four approximate solves: of b (x = c), then of three residuals (x += c)
    const double *in[4] = {W.b, W.ra, W.rb, W.ra};
    double *r_out[4] = {W.ra, W.rb, W.ra, nullptr};
    const double *x_in[4] = {nullptr, W.xa, W.xb, W.xa};
    double *x_out[4] = {W.xa, W.xb, W.xa, P.fs.phi};
    for (int s = 0; s < 4; s++) {
        M.in = in[s];
        M.r_out = r_out[s];
        M.x_in = x_in[s];
        M.x_out = x_out[s];
        k_pl_scan_s<<<nb, PL_T, 0, ctx->stream>>>(M);
        k_pl_scan_y<<<nb, PL_T, 0, ctx->stream>>>(M);
        if (s == 0) k_pl_conv<0><<<nb, PL_T, 0, ctx->stream>>>(M);
        else if (s < 3) k_pl_conv<1><<<nb, PL_T, 0, ctx->stream>>>(M);
        else k_pl_conv<2><<<nb, PL_T, 0, ctx->stream>>>(M);
    }
    return check_launch(ctx, "k_poisson");
}

static int poisson(vx_ctx *ctx, const vx_field_state *fs, double *work) {
    int rc = validate_fs(ctx, fs);
    if (rc) return rc;
    PoissonArgs P;
    P.fs = *fs;
    P.w1 = -16.0 / 30.0 / 0.4;  // EMSolver.cpp:28
    P.w2 = 1.0 / 30.0 / 0.4;
    P.w3 = 1 / 0.4;
    double rho = 7.0 - std::sqrt(48.0);
    double C = 12.0 / (14.0 - 2.0 * rho);
    double pw = 1.0;
    for (int k = 0; k < NG; k++) {
        P.g[k] = C * pw;
        pw *= rho;
    }
    P.rho = rho;
    P.C = C;
    P.invN = 1.0 / fs->n_f;
    LaunchTimer lt(ctx, "k_poisson");
    if (fs->n_f <= SMALL_MAX) {
        const int n = fs->n_f;
        // entries a thread and wavefronts: the fewest wavefronts with an entry a
        // thread, then a wavefront per SIMD, then two (us, 2 x 4 / 1 x 8 at 512: 7.1
        // / 7.4; 4 x 4 / 2 x 8 at 1024: 8.7 / 9.1; 4 x 8 / 8 x 4 at 2048: 11.9 / 12.8)
        if (n <= 64) k_poisson_one<1, 1><<<1, 64, 0, ctx->stream>>>(P);
        else if (n <= 128) k_poisson_one<1, 2><<<1, 128, 0, ctx->stream>>>(P);
        else if (n <= 256) k_poisson_one<1, 4><<<1, 256, 0, ctx->stream>>>(P);
        else if (n <= 512) k_poisson_one<2, 4><<<1, 256, 0, ctx->stream>>>(P);
        else if (n <= 1024) k_poisson_one<4, 4><<<1, 256, 0, ctx->stream>>>(P);
        else if (n <= 2048) k_poisson_one<4, 8><<<1, 512, 0, ctx->stream>>>(P);
        else k_poisson_one<8, 8><<<1, 512, 0, ctx->stream>>>(P);
        return check_launch(ctx, "k_poisson");
    }
    if (!work) return fail(ctx, VX_EINVAL, "poisson: no work array for n_f = %d", fs->n_f);
    if (fs->n_f > PM_MAX) return poisson_long(ctx, P, work);
    PoissonMB M;
    M.fs = *fs;
    M.w1 = P.w1;
    M.w2 = P.w2;
    M.w3 = P.w3;
    for (int k = 0; k < NG; k++) M.g[k] = P.g[k];
    M.invN = P.invN;
    M.nb = pm_chunks(fs->n_f);
    M.W = pm_work(work, fs->n_f);
    const PmWork &W = M.W;
    const unsigned nb = (unsigned)M.nb;
    M.sums_out = W.sums[0];
    const bool small = pm_mw(fs->n_f) == 3;
    if (small) k_pm_rhs<3><<<nb, SUB * 3, 0, ctx->stream>>>(M);
    else k_pm_rhs<8><<<nb, SUB * 8, 0, ctx->stream>>>(M);
    // four approximate solves: of b (x = c), then of three residuals (x += c)
    const double *in[4] = {W.b, W.ra, W.rb, W.ra};
    double *r_out[4] = {W.ra, W.rb, W.ra, nullptr};
    const double *x_in[4] = {nullptr, W.xa, W.xb, W.xa};
    double *x_out[4] = {W.xa, W.xb, W.xa, fs->phi};
    for (int s = 0; s < 4; s++) {
        M.in = in[s];
        M.r_out = r_out[s];
        M.x_in = x_in[s];
        M.x_out = x_out[s];
        M.sums = W.sums[s & 1];
        M.sums_out = W.sums[~s & 1];
        if (small) {
            if (s == 0) k_pm_solve<0, 3><<<nb, 64 * 8, 0, ctx->stream>>>(M);
            else if (s < 3) k_pm_solve<1, 3><<<nb, 64 * 8, 0, ctx->stream>>>(M);
            else k_pm_solve<2, 3><<<nb, 64 * 8, 0, ctx->stream>>>(M);
        } else {
            if (s == 0) k_pm_solve<0, 8><<<nb, 64 * 13, 0, ctx->stream>>>(M);
            else if (s < 3) k_pm_solve<1, 8><<<nb, 64 * 13, 0, ctx->stream>>>(M);
            else k_pm_solve<2, 8><<<nb, 64 * 13, 0, ctx->stream>>>(M);
        }
    }
    return check_launch(ctx, "k_poisson");
}


int vx_poisson(vx_ctx *ctx, const vx_field_state *fs) { return poisson(ctx, fs, fs ? fs->work : nullptr); }

int vx_poisson_noalloc(vx_ctx *ctx, const vx_field_state *fs) {
    int rc = validate_fs(ctx, fs);
    if (rc) return rc;
    if (fs->n_f > VX_POISSON_NOALLOC_MAX_NF)
        return fail(ctx, VX_EINVAL, "vx_poisson_noalloc: n_f = %d exceeds its fixed work array (n_f <= %d)", fs->n_f,
                    VX_POISSON_NOALLOC_MAX_NF);
    if (!ctx->poisson_scratch) return fail(ctx, VX_EHIP, "vx_poisson_noalloc: no work array address on device %d", ctx->device);
    return poisson(ctx, fs, ctx->poisson_scratch);
}

}  // extern "C"

static int maxwell_stage(vx_ctx *ctx, const vx_field_state *fs, int step, double dt, double by0,
                         double bz0, const double *drive) {
    int rc = validate_fs(ctx, fs);
    if (rc) return rc;
    if (step < 0 || step > 5) return fail(ctx, VX_EINVAL, "maxwell: bad step %d", step);
    MaxArgs A;
    A.fs = *fs;
    A.step = step;
    A.by0 = by0;
    A.bz0 = bz0;
    A.drive = drive;
    A.dx_inv = 1 / fs->dx_f;
    for (int k = 0; k < 6; k++) A.a[k] = A.b[k] = 0.0;
    if (step <= 4) {
        for (int k = 0; k <= step; k++) A.a[k] = vx::rk_a[step][k] * dt;
    } else {
        double a[6];
        for (int k = 0; k < 5; k++) a[k] = vx::rk_a[4][k] * dt;
        a[5] = 0;
        for (int k = 0; k < 6; k++) A.b[k] = vx::rk_a[5][k] * dt - a[k];
    }
    if (fs->n_e <= MX1) {
        k_maxwell_one<<<1, 2 * MX1, 0, ctx->stream>>>(A);
        return check_launch(ctx, "k_maxwell_one");
    }
    unsigned g = (unsigned)((fs->n_e + MXT - 1) / MXT);
    k_maxwell_rhs<<<dim3(g, 2), MXT, 0, ctx->stream>>>(A);
    if ((rc = check_launch(ctx, "k_maxwell_rhs"))) return rc;
    k_maxwell_update<<<dim3(g, 5), MXT, 0, ctx->stream>>>(A);
    return check_launch(ctx, "k_maxwell_update");
}

extern "C" {

int vx_maxwell_stage(vx_ctx *ctx, const vx_field_state *fs, int step, double dt, double by0,
                     double bz0) {
    return maxwell_stage(ctx, fs, step, dt, by0, bz0, nullptr);
}

int vx_maxwell_stage_dev(vx_ctx *ctx, const vx_field_state *fs, int step, double dt,
                         const double *drive) {
    if (!drive) return fail(ctx, VX_EINVAL, "maxwell: null drive");
    return maxwell_stage(ctx, fs, step, dt, 0.0, 0.0, drive);
}

int vx_snapshot_fields(vx_ctx *ctx, const vx_field_state *fs, double *E0, double *a20) {
    int rc = validate_fs(ctx, fs);
    if (rc) return rc;
    if (!E0 || !a20) return fail(ctx, VX_EINVAL, "snapshot: null output");
    k_snapshot<<<(unsigned)((fs->n_f + 256) / 256), 256, 0, ctx->stream>>>(*fs, E0, a20);
    return check_launch(ctx, "k_snapshot");
}

int vx_neutralize(vx_ctx *ctx, const vx_field_state *fs) {
    int rc = validate_fs(ctx, fs);
    if (rc) return rc;
    k_neutralize<<<(unsigned)((fs->n_f + 255) / 256), 256, 0, ctx->stream>>>(*fs);
    return check_launch(ctx, "k_neutralize");
}

}  // extern "C"

// EMSolver.cpp:631-664 on the device: pc = max_i (the per-cell term), each term
// with the host code's operations; max is exact, so the order does not matter.
// One workgroup per CFL_CHUNK cells writes its maximum, and the host takes the
// maximum of at most CFL_WG of them.
constexpr int CFL_MAXSP = 8, CFL_CHUNK = 1024, CFL_WG = 64;
struct CflArgs {
    vx_field_state fs;
    int n_species;
    double aq[CFL_MAXSP], m[CFL_MAXSP], dps[CFL_MAXSP];  // |q_j|, m_j, 1 / dp_j
    double dpsMax;
};

__global__ __launch_bounds__(256) void k_cfl(CflArgs A, double *out) {
    const vx_field_state &F = A.fs;
    __shared__ double part[4];
    double pc = 0.0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < F.n_f; i += 256 * gridDim.x) {
        const double Azv = F.Az[i], Ayv = F.Ay[i];
        const double As = Ayv * Ayv + Azv * Azv;
        double temp = 0.0;
        for (int j = 0; j < A.n_species; j++) {
            const double v = A.aq[j] / A.m[j] / sqrt(1 + As / ((A.m[j] * vx_cs) * (A.m[j] * vx_cs))) * A.dps[j];
            temp = (temp < v) ? v : temp;
        }
        const double t = temp * fabs(Ayv * F.Bz[i] - Azv * F.By[i]) + A.dpsMax * fabs(F.E[i]);
        pc = (pc < t) ? t : pc;
    }
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(pc, off, 64);
        pc = (pc < o) ? o : pc;
    }
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = pc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = 0.0;
        for (int k = 0; k < 4; k++) r = (r < part[k]) ? part[k] : r;
        out[blockIdx.x] = r;
    }
}

// Launches k_cfl into `out` (device-visible, CFL_WG doubles); returns the number
// of maxima it writes.
static int cfl_launch(vx_ctx *ctx, const vx_field_state *fs, int n_species, const double *q, const double *m,
                      const double *dp_finest, double *out) {
    CflArgs A;
    A.fs = *fs;
    A.n_species = n_species;
    A.dpsMax = 0.0;
    for (int i = 0; i < n_species; i++) {  // EMSolver.cpp:637-642
        A.aq[i] = std::fabs(q[i]);
        A.m[i] = m[i];
        A.dps[i] = 1 / dp_finest[i];
        A.dpsMax = std::max(A.dpsMax, std::fabs(q[i]) * A.dps[i]);
    }
    const int n = std::min((fs->n_f + CFL_CHUNK - 1) / CFL_CHUNK, CFL_WG);
    k_cfl<<<n, 256, 0, ctx->stream>>>(A, out);
    return n;
}

static double cfl_bound(double c_dx, const double *host, int n) {
    double pc = 0.0;
    for (int k = 0; k < n; k++) pc = std::max(pc, host[k]);
    return 1.0 / std::max((c_dx + pc), 1e-40);
}

extern "C" {

int vx_cfl_bound_async(vx_ctx *ctx, const vx_field_state *fs, int n_species, const double *q, const double *m,
                       const double *dp_finest) {
    int rc = validate_fs(ctx, fs);
    if (rc) return rc;
    if (n_species < 1 || n_species > CFL_MAXSP) return fail(ctx, VX_EINVAL, "cfl: %d species", n_species);
    if (ctx->capturing) return fail(ctx, VX_EINVAL, "cfl bound while a step graph is recorded");
    if (!ctx->cfl_ev &&
        (rc = check_hip(ctx, hipEventCreateWithFlags(&ctx->cfl_ev, hipEventDisableTiming), "cfl event")))
        return rc;
    // the maxima go straight to pinned memory
    if (!ctx->cfl_host &&
        (rc = check_hip(ctx, hipHostMalloc((void **)&ctx->cfl_host, sizeof(double) * CFL_WG), "cfl pinned")))
        return rc;
    ctx->cfl_n = cfl_launch(ctx, fs, n_species, q, m, dp_finest, ctx->cfl_host);
    if ((rc = check_launch(ctx, "k_cfl"))) return rc;
    if ((rc = check_hip(ctx, hipEventRecord(ctx->cfl_ev, ctx->stream), "cfl event record"))) return rc;
    ctx->cfl_c_dx = vx_cs / fs->dx_f;
    ctx->cfl_pending = true;
    return VX_OK;
}

int vx_cfl_ready(vx_ctx *ctx, int *ready) {
    if (!ctx->cfl_pending || !ready) return fail(ctx, VX_EINVAL, "cfl: no bound pending");
    hipError_t e = hipEventQuery(ctx->cfl_ev);
    if (e == hipErrorNotReady) {
        *ready = 0;
        return VX_OK;
    }
    *ready = 1;
    return check_hip(ctx, e, "cfl query");
}

int vx_cfl_result(vx_ctx *ctx, double *out) {
    if (!ctx->cfl_pending || !out) return fail(ctx, VX_EINVAL, "cfl: no bound pending");
    int rc = check_hip(ctx, hipEventSynchronize(ctx->cfl_ev), "cfl wait");
    if (rc) return rc;
    ctx->cfl_pending = false;
    *out = cfl_bound(ctx->cfl_c_dx, ctx->cfl_host, ctx->cfl_n);
    return VX_OK;
}

// EMSolver.cpp:631-664 (the reference indexes the slot-0 fields without the
// n_prepad offset): the maxima on the device, straight into the context's pinned
// buffer if there is one, for the species the kernel holds and arrays that it may
// read, else on the host from downloaded arrays, whose copies refuse what is not the
// device's (five copies from pageable memory took 110 us at 64 cells, the launch and
// a wait 14).  The buffer serves the context's copies too: its mutex is held until
// the maxima are read.
int vx_cfl_bound(vx_ctx *ctx, const vx_field_state *fs, int n_species, const double *q,
                 const double *m, const double *dp_finest, double *out) {
    int rc = validate_fs(ctx, fs);
    if (rc) return rc;
    if (ctx->capturing) return fail(ctx, VX_EINVAL, "cfl bound while a step graph is being recorded");
    bool here = n_species >= 0 && n_species <= CFL_MAXSP;
    for (const double *a : {fs->Ay, fs->Az, fs->By, fs->Bz, fs->E}) here = here && vx_device_range(ctx, a, fs->n_f);
    if (here) {
        std::lock_guard<std::mutex> lock(ctx->stage_mu);
        if (vx_stage_init(ctx) == VX_OK) {
            const int n = cfl_launch(ctx, fs, n_species, q, m, dp_finest, ctx->stage);
            if ((rc = check_launch(ctx, "k_cfl")) || (rc = vx_sync(ctx))) return rc;
            *out = cfl_bound(vx_cs / fs->dx_f, ctx->stage, n);
            return VX_OK;
        }
    }
    int N = fs->n_f;
    std::vector<double> Ay(N), Az(N), By(N), Bz(N), E(N);
    if ((rc = vx_memcpy_d2h(ctx, Ay.data(), fs->Ay, sizeof(double) * N))) return rc;
    if ((rc = vx_memcpy_d2h(ctx, Az.data(), fs->Az, sizeof(double) * N))) return rc;
    if ((rc = vx_memcpy_d2h(ctx, By.data(), fs->By, sizeof(double) * N))) return rc;
    if ((rc = vx_memcpy_d2h(ctx, Bz.data(), fs->Bz, sizeof(double) * N))) return rc;
    if ((rc = vx_memcpy_d2h(ctx, E.data(), fs->E, sizeof(double) * N))) return rc;
    std::vector<double> dps(n_species);
    double dpsMax(0.0);
    for (int i = 0; i < n_species; i++) {
        dps[i] = 1 / dp_finest[i];
        dpsMax = std::max(dpsMax, std::fabs(q[i]) * dps[i]);
    }
    double pc(0.0);
    for (int i = 0; i < N; i++) {
        double Azv = Az[i], Ayv = Ay[i];
        double As = Ayv * Ayv + Azv * Azv;
        double temp(0.0);
        for (int j = 0; j < n_species; j++)
            temp = std::max(temp, std::fabs(q[j]) / m[j] / std::sqrt(1 + As / ((m[j] * vx_cs) * (m[j] * vx_cs))) * dps[j]);
        pc = std::max(pc, temp * std::fabs(Ayv * Bz[i] - Azv * By[i]) + dpsMax * std::fabs(E[i]));
    }
    *out = 1.0 / std::max((vx_cs / fs->dx_f + pc), 1e-40);
    return VX_OK;
}

}  // extern "C"
