// po_cheb_dev.hpp -- device bodies of the Chebyshev grid behind the node sums,
// shared by the single propagation (po_cheb.hip, po_ff.hip) and the batched
// sweep (sweep.hip): split reduction, coefficients, evaluation at the targets.
#pragma once

#include "po_common.hpp"

namespace pypo {

// Direction of a target as (a, b).
__device__ __forceinline__ void target_ab(const double *th, const double *ph, int t, double &a, double &b) {
    double sp, cp;
    sincos(ph[t], &sp, &cp);
    a = th[t] * cp;
    b = th[t] * sp;
}

// Box of the directions of one workgroup's share of the targets, in FP32 (the
// plan widens it by its rounding).  A direction that is not finite leaves NaN.
__device__ __forceinline__ void target_box(const ChebWs &w, int block, float *scratch) {
    float lo_a = INFINITY, lo_b = INFINITY, hi_a = -INFINITY, hi_b = -INFINITY, bad = 0.f;
#pragma unroll
    for (int j = 0; j < kChebBoxTargets / TILE; j++) {
        const int t = block * kChebBoxTargets + j * TILE + threadIdx.x;
        if (t >= w.n_tgt) break;
        double sp, cp;
        sincos(w.tgt_ph[t], &sp, &cp);
        const float a = (float)(w.tgt_th[t] * cp), b = (float)(w.tgt_th[t] * sp);
        lo_a = fminf(lo_a, a); hi_a = fmaxf(hi_a, a);
        lo_b = fminf(lo_b, b); hi_b = fmaxf(hi_b, b);
        if (!(fabsf(a) < 1e30f && fabsf(b) < 1e30f)) bad = 1.f;
    }
    lo_a = block_min(lo_a, scratch);
    lo_b = block_min(lo_b, scratch);
    hi_a = -block_min(-hi_a, scratch);
    hi_b = -block_min(-hi_b, scratch);
    bad = -block_min(-bad, scratch);
    if (threadIdx.x == 0) {
        float *o = w.tgt_box + 4 * block;
        o[0] = bad > 0.f ? __builtin_nanf("") : lo_a;
        o[1] = lo_b; o[2] = hi_a; o[3] = hi_b;
    }
}

// Box [min x, y, z, max x, y, z] of a tile's positions (this lane's: p), for the plan.
__device__ __forceinline__ void position_box(float *box, int tile, const double (&p)[3], bool valid, float *scratch) {
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const float x = (float)p[q];
        // a NaN would vanish in the minimum: it leaves an infinite box
        const bool nan = x != x;
        const float lo = block_min(valid ? (nan ? -INFINITY : x) : INFINITY, scratch);
        const float hi = -block_min(valid ? (nan ? -INFINITY : -x) : INFINITY, scratch);
        if (threadIdx.x == 0) {
            box[6 * tile + q] = lo;
            box[6 * tile + 3 + q] = hi;
        }
    }
}

// exp(j 2 pi c.(s r)) for r = (cp st, sp st, ct), s r rounded as the sums round
// it, and the product to twice FP64's precision: hundreds of revolutions that
// all sources of a target share, where the roundings of a sum over sources
// average out (1000 wavelengths of dish at f / D = 0.4, 700 from the
// origin: error of a far field 5.9e-13 with the plain product, 1.2e-14 with this).
__device__ __forceinline__ void centre_phase(const ChebPlan &pl, double s, double st, double ct, double sp, double cp,
                                             double &sn, double &cs) {
#pragma clang fp contract(off)
    const double u[3] = {cp * st * s, sp * st * s, ct * s};
    double rev = 0.0, lo = 0.0;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const double p = pl.c[q] * u[q], t = rev + p, v = t - rev;   // two-sum
        lo += ((rev - (t - v)) + (p - v)) + __builtin_fma(pl.c[q], u[q], -p);
        rev = t;
    }
    sincospi(2.0 * ((rev - __builtin_rint(rev)) + lo), &sn, &cs);
}

// cos(x) - 1 to full relative precision.
__device__ __forceinline__ double cos_less_one(double x) {
    const double s = sin(0.5 * x);
    return -2.0 * s * s;
}

// Split reduction of the node sums, times exp(j t k c.r): f[2a + part][node];
// one lane per node and complex component.  TURNED: sums of k_ff_fp64, whose
// sources carry the z part of that for r_z = 1.
template <bool TURNED>
__device__ __forceinline__ void cheb_reduce(const ChebWs &w, const double *__restrict__ partial, double rev_scale,
                                            int block, int blocks) {
    const ChebPlan &pl = *w.plan;
    const int comps = pl.has_m ? 6 : 3, n = pl.n, splits = pl.splits;
    for (int e = block * TILE + threadIdx.x; e < comps * n; e += blocks * TILE) {
        const int a = e / n, i = e - a * n;
        const double *p = partial + (size_t)(2 * a) * n + i;
        double re = 0.0, im = 0.0;
#pragma unroll 4
        for (int s = 0; s < splits; s++) {
            re += p[(size_t)s * 12 * n];
            im += p[(size_t)s * 12 * n + n];
        }
        double st, ct, sp, cp, sn, cs;
        sincos(w.th[i], &st, &ct);
        sincos(w.ph[i], &sp, &cp);
        if (TURNED) ct = cos_less_one(w.th[i]);
        centre_phase(pl, -rev_scale, st, ct, sp, cp, sn, cs);
        w.f[(size_t)(2 * a) * n + i] = re * cs - im * sn;
        w.f[(size_t)(2 * a + 1) * n + i] = re * sn + im * cs;
    }
}

// Whether target t stands where rows of `row` put it: its a against its row's
// first target and its b against the first row's, within the rounding of theta
// and phi.
__device__ __forceinline__ bool cheb_in_row(const ChebWs &w, int t, int row, double tol) {
    const int i = t / row, j = t - i * row;
    double a, b, a0, b0, x;
    target_ab(w.tgt_th, w.tgt_ph, t, a, b);
    target_ab(w.tgt_th, w.tgt_ph, i * row, a0, x);
    target_ab(w.tgt_th, w.tgt_ph, j, x, b0);
    return fabs(a - a0) <= tol && fabs(b - b0) <= tol;
}

// Checks the rows a plan supposes (pl.row) at every target.
__device__ __forceinline__ void cheb_check_rows(const ChebWs &w, int block, int blocks) {
    const ChebPlan &pl = *w.plan;
    if (!pl.row) return;
    bool bad = false;
    for (int t = block * TILE + threadIdx.x; t < w.n_tgt; t += blocks * TILE)
        bad |= !cheb_in_row(w, t, pl.row, pl.row_tol);
    if (bad) *w.not_rows = 1;
}

// Direction of node i.
__device__ __forceinline__ void cheb_node(const ChebPlan &pl, int i, double *th, double *ph) {
    const int ia = i / pl.nb, ib = i - ia * pl.nb;
    const double a = pl.a_mid + pl.a_half * cospi((2 * ia + 1) / (2.0 * pl.na));
    const double b = pl.b_mid + pl.b_half * cospi((2 * ib + 1) / (2.0 * pl.nb));
    th[i] = hypot(a, b);
    ph[i] = atan2(b, a);
}

// Chebyshev coefficients of the node values: a workgroup takes one row ka of
// one real component, transforms it along a (coalesced over ib), then along b.
// Where the targets form rows of equal a, it goes on to evaluate the row of
// coefficients at the b of every column: rows[ka][q][j].  2 n (na + nb) FMAs
// per component; latency-bound, some 10 us.
__device__ __forceinline__ void cheb_coef(const ChebWs &w, int block, int blocks) {
    __shared__ double ca[4 * kChebMaxAxis], cb[4 * kChebMaxAxis], g[kChebMaxAxis], c[kChebMaxAxis];
    const ChebPlan &pl = *w.plan;
    const int na = pl.na, nb = pl.nb, n = pl.n, tid = threadIdx.x;
    const bool rows = pl.row && !*w.not_rows;
    for (int j = tid; j < 4 * na; j += TILE) ca[j] = cospi(j / (2.0 * na));
    for (int j = tid; j < 4 * nb; j += TILE) cb[j] = cospi(j / (2.0 * nb));
    const int items = (pl.has_m ? 12 : 6) * na;
    for (int item = block; item < items; item += blocks) {
        const int q = item / na, ka = item - q * na;
        __syncthreads();
        if (tid < nb) {
            const double *f = w.f + (size_t)q * n + tid;
            double s = 0.0;
            int j = ka;                       // ka (2 m + 1) mod 4 na
#pragma unroll 4
            for (int m = 0; m < na; m++) {
                s = __builtin_fma(f[(size_t)m * nb], ca[j], s);
                j += 2 * ka;
                if (j >= 4 * na) j -= 4 * na;
            }
            g[tid] = s * (ka ? 2.0 : 1.0) / na;
        }
        __syncthreads();
        if (tid < nb) {
            double s = 0.0;
            int j = tid;
#pragma unroll 4
            for (int m = 0; m < nb; m++) {
                s = __builtin_fma(g[m], cb[j], s);
                j += 2 * tid;
                if (j >= 4 * nb) j -= 4 * nb;
            }
            s *= (tid ? 2.0 : 1.0) / nb;
            c[tid] = s;
            w.coef[((size_t)ka * nb + tid) * 12 + q] = s;
        }
        if (!rows) continue;
        __syncthreads();
        for (int j = tid; j < pl.row; j += TILE) {
            double a, b;
            target_ab(w.tgt_th, w.tgt_ph, j, a, b);
            const double y = fmin(1.0, fmax(-1.0, (b - pl.b_mid) / pl.b_half));
            double s = 0.0, u = 1.0, up = y;
            for (int l = 0; l < nb; l++) {
                s = __builtin_fma(u, c[l], s);
                const double un = __builtin_fma(2.0 * y, u, -up);
                up = u;
                u = un;
            }
            w.rows[((size_t)ka * 12 + q) * pl.row + j] = s;
        }
    }
}

// The series at the direction (a, b), rows [m0, m1) of its coefficients:
// S[q] += sum_ka T_ka(x) sum_kb T_kb(y) coef[ka][kb][q].  Coefficients are
// uniform over the wave (scalar loads); 13 FP64 FMAs per term (7 without
// magnetic currents).
template <bool HAS_M>
__device__ __forceinline__ void cheb_series(const ChebPlan &pl, const double *__restrict__ coef, double a, double b,
                                            int m0, int m1, double (&S)[12]) {
    constexpr int Q = HAS_M ? 12 : 6;
    const double x = fmin(1.0, fmax(-1.0, (a - pl.a_mid) / pl.a_half));
    const double y = fmin(1.0, fmax(-1.0, (b - pl.b_mid) / pl.b_half));
    const double angle = acos(x);
    double t0 = cos(m0 * angle), tp = cos((m0 - 1) * angle);   // T_m0(x), T_(m0-1)(x)
    for (int m = m0; m < m1; m++) {
        ConstDouble *c = const_space(coef) + (size_t)m * pl.nb * 12;
        double r[Q], u = 1.0, up = y;                          // T_0(y), T_(-1)(y) = T_1(y)
#pragma unroll
        for (int q = 0; q < Q; q++) r[q] = 0.0;
#pragma unroll 2
        for (int l = 0; l < pl.nb; l++) {
#pragma unroll
            for (int q = 0; q < Q; q++) r[q] = __builtin_fma(u, c[12 * l + q], r[q]);
            const double un = __builtin_fma(2.0 * y, u, -up);
            up = u;
            u = un;
        }
#pragma unroll
        for (int q = 0; q < Q; q++) S[q] = __builtin_fma(t0, r[q], S[q]);
        const double tn = __builtin_fma(2.0 * x, t0, -tp);
        tp = t0;
        t0 = tn;
    }
}

// Far field of the J and M sums S (S[2a], S[2a+1]: J_a, S[6+2a], S[7+2a]: M_a)
// at the direction r = (cp st, sp st, ct): E = -j pref [S_J - (S_J.r) r + t r x
// S_M], H = -j pref [S_M - (S_M.r) r - t r x S_J], written to out[q][t].
template <class Out>
__device__ __forceinline__ void ff_project(const double (&S)[12], double st, double ct, double sp, double cp,
                                           double tdir, double pref, const Out &out, int t) {
    const double r[3] = {cp * st, sp * st, ct};
    double jdr_re = 0, jdr_im = 0, mdr_re = 0, mdr_im = 0;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        jdr_re += S[2 * a] * r[a]; jdr_im += S[2 * a + 1] * r[a];
        mdr_re += S[6 + 2 * a] * r[a]; mdr_im += S[7 + 2 * a] * r[a];
    }
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const int b = (a + 1) % 3, c = (a + 2) % 3;
        // (r x V)_a = r_b V_c - r_c V_b
        const double rxm_re = r[b] * S[6 + 2 * c] - r[c] * S[6 + 2 * b];
        const double rxm_im = r[b] * S[7 + 2 * c] - r[c] * S[7 + 2 * b];
        const double rxj_re = r[b] * S[2 * c] - r[c] * S[2 * b];
        const double rxj_im = r[b] * S[2 * c + 1] - r[c] * S[2 * b + 1];
        const double e_re = S[2 * a] - r[a] * jdr_re + tdir * rxm_re;
        const double e_im = S[2 * a + 1] - r[a] * jdr_im + tdir * rxm_im;
        const double h_re = S[6 + 2 * a] - r[a] * mdr_re - tdir * rxj_re;
        const double h_im = S[7 + 2 * a] - r[a] * mdr_im - tdir * rxj_im;
        // multiply by -j*pref: (x + j y)(-j) = y - j x
        out.at(a)[t] = pref * e_im;
        out.at(3 + a)[t] = -pref * e_re;
        out.at(6 + a)[t] = pref * h_im;
        out.at(9 + a)[t] = -pref * h_re;
    }
}

// Far field at the targets from a plan that is on; the caller's grid has one
// workgroup per kChebEvalTargets targets.
//
// Targets in rows of equal a: a lane takes one column of two rows, S[q] =
// sum_ka T_ka(x) rows[ka][q][j] -- the two-dimensional series costs na terms a
// target instead of na nb (251 001 targets, 59 x 59 nodes: 540 -> 37 us).
// Any other order: 64 targets per workgroup, the four waves sharing the
// series' rows (31 313 targets would otherwise fill half of the chip's SIMDs
// with one wave each).
constexpr int kChebEvalTargets = 64;
constexpr int kChebEvalRows = 2;
template <class Out>
__device__ __forceinline__ void cheb_finish(const ChebWs &w, double rev_scale, double tdir, double pref,
                                            const Out &out, int block, int blocks) {
    __shared__ double sh[3][12][64];
    const ChebPlan &pl = *w.plan;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int Q = pl.has_m ? 12 : 6;
    if (pl.row && !*w.not_rows) {
        const int nx = w.n_tgt / pl.row, bj = (pl.row + 63) / 64, bi = (nx + 4 * kChebEvalRows - 1) / (4 * kChebEvalRows);
        for (int item = block; item < bi * bj; item += blocks) {
            const int j = item % bj * 64 + lane, i0 = (item / bj * 4 + wv) * kChebEvalRows;
            if (i0 >= nx || j >= pl.row) continue;
            double x[kChebEvalRows], t0[kChebEvalRows], tp[kChebEvalRows], S[kChebEvalRows][12];
#pragma unroll
            for (int r = 0; r < kChebEvalRows; r++) {
                double a, b;
                target_ab(w.tgt_th, w.tgt_ph, min(i0 + r, nx - 1) * pl.row, a, b);
                x[r] = fmin(1.0, fmax(-1.0, (a - pl.a_mid) / pl.a_half));
                t0[r] = 1.0;
                tp[r] = x[r];
#pragma unroll
                for (int q = 0; q < 12; q++) S[r][q] = 0.0;
            }
            const double *p = w.rows + j;
            const size_t n = pl.row;
            for (int m = 0; m < pl.na; m++, p += 12 * n) {
                double v[12];
#pragma unroll
                for (int q = 0; q < 12; q++) v[q] = q < 6 || Q == 12 ? p[q * n] : 0.0;
#pragma unroll
                for (int r = 0; r < kChebEvalRows; r++) {
#pragma unroll
                    for (int q = 0; q < 12; q++) S[r][q] = __builtin_fma(t0[r], v[q], S[r][q]);
                    const double tn = __builtin_fma(2.0 * x[r], t0[r], -tp[r]);
                    tp[r] = t0[r];
                    t0[r] = tn;
                }
            }
#pragma unroll
            for (int r = 0; r < kChebEvalRows; r++) {
                if (i0 + r >= nx) break;
                const int t = (i0 + r) * pl.row + j;
                double st, ct, sp, cp, sn, cs;
                sincos(w.tgt_th[t], &st, &ct);
                sincos(w.tgt_ph[t], &sp, &cp);
                centre_phase(pl, rev_scale, st, ct, sp, cp, sn, cs);
#pragma unroll
                for (int a = 0; a < 6; a++) {
                    const double re = S[r][2 * a], im = S[r][2 * a + 1];
                    S[r][2 * a] = re * cs - im * sn;
                    S[r][2 * a + 1] = re * sn + im * cs;
                }
                ff_project(S[r], st, ct, sp, cp, tdir, pref, out, t);
            }
        }
        return;
    }
    int t = block * kChebEvalTargets + lane;
    const bool valid = t < w.n_tgt;
    if (!valid) t = w.n_tgt - 1;
    double st, ct, sp, cp, sn, cs, S[12];
    sincos(w.tgt_th[t], &st, &ct);
    sincos(w.tgt_ph[t], &sp, &cp);
#pragma unroll
    for (int q = 0; q < 12; q++) S[q] = 0.0;
    const double a = w.tgt_th[t] * cp, b = w.tgt_th[t] * sp;
    const int m0 = wv * pl.na / 4, m1 = (wv + 1) * pl.na / 4;
    if (pl.has_m) cheb_series<true>(pl, w.coef, a, b, m0, m1, S);
    else cheb_series<false>(pl, w.coef, a, b, m0, m1, S);
    if (wv) {
#pragma unroll
        for (int q = 0; q < 12; q++) sh[wv - 1][q][lane] = S[q];
    }
    __syncthreads();
    if (wv || !valid) return;
    centre_phase(pl, rev_scale, st, ct, sp, cp, sn, cs);
#pragma unroll
    for (int c = 0; c < 6; c++) {
        const double re = S[2 * c] + sh[0][2 * c][lane] + sh[1][2 * c][lane] + sh[2][2 * c][lane];
        const double im = S[2 * c + 1] + sh[0][2 * c + 1][lane] + sh[1][2 * c + 1][lane] + sh[2][2 * c + 1][lane];
        S[2 * c] = re * cs - im * sn;
        S[2 * c + 1] = re * sn + im * cs;
    }
    ff_project(S, st, ct, sp, cp, tdir, pref, out, t);
}

}  // namespace pypo
