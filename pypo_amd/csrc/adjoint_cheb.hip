// adjoint_cheb.hip -- the adjoint on Chebyshev grids.
//
// Reverse sums.  B_i = sum_t A_t exp(j phi_ti) is the transpose of the far
// field's evaluation at the targets, phi_ti = -t k p_i.r(a_t, b_t): with the
// interpolant exp(-j t k (p_i - c).r(a, b)) = sum_n L_n(a, b) exp(-j t k (p_i -
// c).r_n) over the nodes of the plan (po_cheb.hpp; the dish points are its
// sources), the targets' amplitudes are gathered once,
//   A'_n = exp(j t k c.r_n) sum_t L_n(a_t, b_t) A_t exp(-j t k c.r_t),
// and the reverse kernels run over the nodes as their targets.  G_i's factor
// n_i.r(a, b) is part of the interpolated function (one more radian per radian
// in its rate), so that the same A' serve.  The sum with the Lagrange
// polynomials L goes through the Chebyshev moments of A, a (na x targets) by
// (targets x nb) product for each of the six real components.
//
// Currents.  H at the dish and its derivative along the normals come from the
// patches around the feed (po_near_cheb.hpp): one H-only sum at the nodes in
// place of the sum of H and dH at every dish point.  Errors of the node sums
// come back smooth over a patch and do not average out over the dish, so they
// are FP64 sums in mixed precision too (158 us).
//
// Measured on MI355X, 401^2 dish, 151^2 far field, 33^2 feed, mixed: reverse
// sums 1926 -> 740 us (503 of them the sums at the nodes, 157 the moments),
// currents 1356 -> 490 us (209 the series).  Gradient error against FP64 over
// fourteen problems of 327^2 to 426^2 dishes: rms 2.2e-7 -> 2.1e-7 of its norm.

#include "adjoint.hpp"
#include "po_cheb_dev.hpp"
#include "po_near_cheb_dev.hpp"

#include <algorithm>

namespace pypo {
namespace {

constexpr int kMomSplits = 64;     // target splits of the moments
constexpr int kMomT = 32;          // and targets per stage
// SIMD cycles a target takes for up to kMomTiles tiles of moments: 5.8 to 6.2 ns
// measured from 40 000 to 160 000 targets, 10 to 16 tiles.  A reverse sum over a
// 90^2 dish and 300^2 targets at 99 x 99 nodes, 521 us of moments, is slower than
// one over the targets (865 us of gradient against 702): the rule leaves it off.
constexpr double kMomCycles = 6.0e-9 * kSimdHz;

// Normal cone and position box per 256 dish points, then the targets' boxes.
__global__ __launch_bounds__(256) void k_adj_dish_meta(GridPtrs dish, int n, TileMeta *__restrict__ meta, ChebWs w) {
    __shared__ float scratch[4];
    if ((int)blockIdx.x >= n_tiles(n)) {
        target_box(w, blockIdx.x - n_tiles(n), scratch);
        return;
    }
    const int i = blockIdx.x * TILE + threadIdx.x;
    const bool valid = i < n;
    const int j = min(i, n - 1);
    const double p[3] = {dish.x[j], dish.y[j], dish.z[j]};
    const Cone c = block_cone((float)dish.nx[j], (float)dish.ny[j], (float)dish.nz[j], valid, scratch);
    if (threadIdx.x == 0) {
        TileMeta m{};
        m.ax = c.ax; m.ay = c.ay; m.az = c.az; m.cos_half = c.cos_half;
        meta[blockIdx.x] = m;
    }
    position_box(w.src_box, blockIdx.x, p, valid, scratch);
}

// Per target: arccos of its place along both axes, and A_t exp(-j t k c.r_t) (3
// complex), rows of n_tgt.  Apart from the moments, whose workgroups would form
// them ten times for eight lanes each (210 us with, 165 without).
__global__ __launch_bounds__(256) void k_adj_amplitudes(ChebWs w, Bundle12 e, const double *__restrict__ g,
                                                        double rev_scale, double pref, double *__restrict__ amp) {
    if (!w.plan->on) return;
    const ChebPlan &pl = *w.plan;
    const int t = blockIdx.x * 256 + threadIdx.x, n = w.n_tgt;
    if (t >= n) return;
    double st, ct, sp, cp, sn, cs;
    sincos(w.tgt_th[t], &st, &ct);
    sincos(w.tgt_ph[t], &sp, &cp);
    const double a = w.tgt_th[t] * cp, b = w.tgt_th[t] * sp;
    amp[t] = acos(fmin(1.0, fmax(-1.0, (a - pl.a_mid) / pl.a_half)));
    amp[(size_t)n + t] = acos(fmin(1.0, fmax(-1.0, (b - pl.b_mid) / pl.b_half)));
    centre_phase(pl, rev_scale, st, ct, sp, cp, sn, cs);
    const double s = 2.0 * g[t] * pref;      // A = 2 g (-j pref) conj(E)
#pragma unroll
    for (int p = 0; p < 3; p++) {
        const double re = -s * e.p[3 + p][t], im = -s * e.p[p][t];
        amp[(size_t)(2 + 2 * p) * n + t] = re * cs - im * sn;
        amp[(size_t)(3 + 2 * p) * n + t] = re * sn + im * cs;
    }
}

// moments[split][q][ka nb + kb] = sum over the split's targets of T_ka(x_t)
// T_kb(y_t) A_t exp(-j t k c.r_t).  A workgroup takes 64 x 16 moments: lane ka
// and four kb in registers, the polynomials of 32 targets staged in LDS.
__global__ __launch_bounds__(256) void k_adj_moments(ChebWs w, const double *__restrict__ amp,
                                                     double *__restrict__ moments) {
    if (!w.plan->on) return;
    const ChebPlan &pl = *w.plan;
    __shared__ double ta[kMomT][kMomA], tb[kMomT][kMomB], am[kMomT][6];
    const int na = pl.na, nb = pl.nb, tid = threadIdx.x, la = tid & 63, lb = (tid >> 6) * 4;
    const int ga = (na + kMomA - 1) / kMomA, gb = (nb + kMomB - 1) / kMomB;
    const int per = (w.n_tgt + kMomSplits - 1) / kMomSplits;
    const int t_begin = blockIdx.y * per, t_end = min(w.n_tgt, t_begin + per);
    for (int item = blockIdx.x; item < ga * gb; item += gridDim.x) {
        const int a0 = item % ga * kMomA, b0 = item / ga * kMomB;
        double acc[4][6];
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int q = 0; q < 6; q++) acc[j][q] = 0.0;
        for (int base = t_begin; base < t_end; base += kMomT) {
            __syncthreads();
            {   // eight lanes per target: its polynomials, and the amplitude
                const int r = tid >> 3, p = tid & 7, t = base + r;
                if (t < t_end) {
                    const double ax = amp[t], ay = amp[(size_t)w.n_tgt + t];
                    // T_{k + 8} = 2 T_8 T_k - T_{k - 8}
                    const double t8 = 2.0 * cos(8.0 * ax);
                    double u0 = cos((a0 + p - 8) * ax), u1 = cos((a0 + p) * ax);
#pragma unroll
                    for (int k = 0; k < kMomA; k += 8) {
                        ta[r][k + p] = u1;
                        const double u2 = __builtin_fma(t8, u1, -u0);
                        u0 = u1; u1 = u2;
                    }
                    for (int k = p; k < kMomB; k += 8) tb[r][k] = cos((b0 + k) * ay);
                    if (p < 6) am[r][p] = amp[(size_t)(2 + p) * w.n_tgt + t];
                } else {
                    for (int k = p; k < kMomA; k += 8) ta[r][k] = 0.0;
                    for (int k = p; k < kMomB; k += 8) tb[r][k] = 0.0;
                    if (p < 6) am[r][p] = 0.0;
                }
            }
            __syncthreads();
#pragma unroll 2
            for (int r = 0; r < kMomT; r++) {
                const double x = ta[r][la];
                double v[6];
#pragma unroll
                for (int q = 0; q < 6; q++) v[q] = am[r][q] * x;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const double y = tb[r][lb + j];
#pragma unroll
                    for (int q = 0; q < 6; q++) acc[j][q] = __builtin_fma(v[q], y, acc[j][q]);
                }
            }
        }
        if (a0 + la < na) {
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (b0 + lb + j < nb)
#pragma unroll
                    for (int q = 0; q < 6; q++)
                        moments[((size_t)blockIdx.y * 6 + q) * pl.n + (size_t)(a0 + la) * nb + b0 + lb + j] = acc[j][q];
        }
    }
}

__global__ __launch_bounds__(256) void k_adj_moment_sum(ChebWs w, const double *__restrict__ moments) {
    if (!w.plan->on) return;
    const int n = 6 * w.plan->n;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        double s = 0.0;
#pragma unroll 8
        for (int k = 0; k < kMomSplits; k++) s += moments[(size_t)k * n + i];
        w.f[i] = s;
    }
}

// f[q][ka][kb] -> coef[q][ia][ib] = sum_t L_ia L_ib A_t, with L_i(x) = sum_k (1 or
// 2) / n T_k(x_i) T_k(x): the transpose of cheb_coef, one (q, ia) a workgroup.
__global__ __launch_bounds__(256) void k_adj_gather(ChebWs w) {
    __shared__ double ca[4 * kChebMaxAxis], cb[4 * kChebMaxAxis], v[kChebMaxAxis];
    if (!w.plan->on) return;
    const ChebPlan &pl = *w.plan;
    const int na = pl.na, nb = pl.nb, n = pl.n, tid = threadIdx.x;
    for (int j = tid; j < 4 * na; j += 256) ca[j] = cospi(j / (2.0 * na));
    for (int j = tid; j < 4 * nb; j += 256) cb[j] = cospi(j / (2.0 * nb));
    for (int item = blockIdx.x; item < 6 * na; item += gridDim.x) {
        const int q = item / na, ia = item - q * na;
        __syncthreads();
        if (tid < nb) {
            const double *f = w.f + (size_t)q * n + tid;
            double s = 0.5 * f[0];
            int j = 0;                              // k (2 ia + 1) mod 4 na
            for (int k = 1; k < na; k++) {
                j += 2 * ia + 1;
                if (j >= 4 * na) j -= 4 * na;
                s = __builtin_fma(f[(size_t)k * nb], ca[j], s);
            }
            v[tid] = s * 2.0 / na;
        }
        __syncthreads();
        if (tid < nb) {
            double s = 0.5 * v[0];
            int j = 0;
            for (int k = 1; k < nb; k++) {
                j += 2 * tid + 1;
                if (j >= 4 * nb) j -= 4 * nb;
                s = __builtin_fma(v[k], cb[j], s);
            }
            w.coef[(size_t)q * n + (size_t)ia * nb + tid] = s * 2.0 / nb;
        }
    }
}

// Records of the nodes as the reverse sums' targets, rows alternately reversed
// so that consecutive ones are neighbours (the matrix kernel's follower phase).
template <class Rec>
__global__ __launch_bounds__(256) void k_adj_node_targets(ChebWs w, double rev_scale, Rec *__restrict__ out) {
    if (!w.plan->on) return;
    const ChebPlan &pl = *w.plan;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < pl.n; i += gridDim.x * 256) {
        double st, ct, sp, cp, sn, cs;
        sincos(w.th[i], &st, &ct);
        sincos(w.ph[i], &sp, &cp);
        const double r[3] = {cp * st, sp * st, ct};
        centre_phase(pl, -rev_scale, st, ct, sp, cp, sn, cs);
        Rec o{};
        o.ux = r[0] * rev_scale; o.uy = r[1] * rev_scale; o.uz = r[2] * rev_scale;
        o.rx = r[0]; o.ry = r[1]; o.rz = r[2];
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const double re = w.coef[(size_t)(2 * a) * pl.n + i], im = w.coef[(size_t)(2 * a + 1) * pl.n + i];
            o.a[2 * a] = re * cs - im * sn;
            o.a[2 * a + 1] = re * sn + im * cs;
        }
        out[packed_slot(i, pl.n, pl.na, pl.nb)] = o;
    }
}

// J and dJ at the dish points from the patches' series; rows of jd as
// k_adj_currents writes them.
__global__ __launch_bounds__(256) void k_adj_currents_series(NearWs w, GridPtrs dish, int n_dish, double rev_scale,
                                                             double pref, double *__restrict__ jd) {
    if (!w.plan->on) return;
    int i;
    const bool valid = near_eval_target(w, i);
    const double n[3] = {dish.nx[i], dish.ny[i], dish.nz[i]};
    double H[6], D[6];
    near_series_grad(w, rev_scale, i, n, H, D);
    if (threadIdx.x >= 64 || !valid) return;
    const double f = 2.0 * pref;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const int b = (a + 1) % 3, c = (a + 2) % 3;
        jd[(size_t)a * n_dish + i] = f * (n[b] * H[2 * c] - n[c] * H[2 * b]);
        jd[(size_t)(3 + a) * n_dish + i] = f * (n[b] * H[2 * c + 1] - n[c] * H[2 * b + 1]);
        jd[(size_t)(6 + a) * n_dish + i] = f * (n[b] * D[2 * c] - n[c] * D[2 * b]);
        jd[(size_t)(9 + a) * n_dish + i] = f * (n[b] * D[2 * c + 1] - n[c] * D[2 * b + 1]);
    }
}

size_t up256(size_t b) { return (b + 255) / 256 * 256; }

// Issue cycles of 64 pairs: reverse sums at 1.9e12 (matrix), 9.5e11 (vector) and
// 4.5e11 pairs/s (FP64), currents at 1.3e11 and 9.2e10.
double reverse_cycles(int precision) {
    return precision == PYPO_PREC_FP64 ? 350.0 : (ff_kernel() == PYPO_FF_MATRIX ? 82.0 : 165.0);
}
double currents_cycles(int precision) { return precision == PYPO_PREC_FP64 ? 1700.0 : 1218.0; }

double microseconds(double pairs, double cycles) { return pairs / 64 * cycles / kSimdHz * 1e6; }

}  // namespace

// Tried from 300 us of reverse sums; the passes around them are some 70 us, 15
// us where the plan stays off.
size_t adj_far_bytes(int precision, int n_dish, int n_tgt) {
    if (n_dish < 1024 || n_tgt < 1024 || microseconds((double)n_dish * n_tgt, reverse_cycles(precision)) < 300) return 0;
    const size_t cap = std::min(kChebMaxNodes, n_tgt);
    return up256(cheb_bytes(n_dish, n_tgt)) + up256((size_t)n_tiles(n_dish) * sizeof(TileMeta)) +
           up256(kMomSplits * 6 * cap * sizeof(double)) + up256((size_t)n_tgt * 8 * sizeof(double));
}

AdjFar adj_far_carve(void *base, int precision, int n_dish, const GridPtrs &ff, int n_tgt) {
    (void)precision;
    AdjFar f;
    char *b = (char *)base;
    f.w = cheb_carve(b, n_dish, ff, n_tgt);
    b += up256(cheb_bytes(n_dish, n_tgt));
    f.meta = (TileMeta *)b;
    b += up256((size_t)n_tiles(n_dish) * sizeof(TileMeta));
    f.moments = (double *)b;
    b += up256(kMomSplits * 6 * (size_t)std::min(kChebMaxNodes, n_tgt) * sizeof(double));
    f.amp = (double *)b;
    return f;
}

int launch_adj_far(int precision, const AdjFar &f, const GridPtrs &dish, int n_dish, const Bundle12 &E,
                   const double *g, double rev_scale, double pref, void *tg, hipStream_t st) {
    const ChebWs &w = f.w;
    hipLaunchKernelGGL(k_adj_dish_meta, dim3(n_tiles(n_dish) + w.boxes()), dim3(256), 0, st, dish, n_dish, f.meta, w);
    PYPO_CHECK_LAUNCH();
    // The FP64 node counts in mixed precision too: B_i is a sum of phases that
    // mostly cancel, and the interpolant's error is one of sum |A_t|.  No sum at
    // the nodes here: the plan's own splits are not used.
    const SumPlan p{1, (w.n_tgt + TILE - 1) / TILE, n_tiles(n_dish), TILE};
    int err = launch_cheb_plan(PYPO_PREC_FP64, p, f.meta, n_dish, rev_scale, partial_bytes(PYPO_MODE_FF, p, w.n_tgt),
                               {reverse_cycles(precision), 60.0, 1.0, kMomCycles}, w, st);
    if (err) return err;
    hipLaunchKernelGGL(k_adj_amplitudes, dim3((w.n_tgt + 255) / 256), dim3(256), 0, st, w, E, g, rev_scale, pref, f.amp);
    PYPO_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_adj_moments, dim3(kMomTiles, kMomSplits), dim3(256), 0, st, w, (const double *)f.amp, f.moments);
    PYPO_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_adj_moment_sum, dim3(256), dim3(256), 0, st, w, f.moments);
    PYPO_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_adj_gather, dim3(512), dim3(256), 0, st, w);
    PYPO_CHECK_LAUNCH();
    if (precision == PYPO_PREC_FP64)
        hipLaunchKernelGGL(k_adj_node_targets<TgtRec64>, dim3(64), dim3(256), 0, st, w, rev_scale, (TgtRec64 *)tg);
    else
        hipLaunchKernelGGL(k_adj_node_targets<TgtRec32>, dim3(64), dim3(256), 0, st, w, rev_scale, (TgtRec32 *)tg);
    PYPO_CHECK_LAUNCH();
    return 0;
}

// Tried from 800 us of the currents pass, 1 ms in FP64 (as in near_cheb_try):
// the FP64 sums at the nodes and the passes around them are some 250 us.
size_t adj_near_bytes(int precision, int n_feed, int n_dish) {
    const double us = microseconds((double)n_feed * n_dish, currents_cycles(precision));
    if (n_dish < 1024 || n_feed < 64 || us < (precision == PYPO_PREC_FP64 ? 1000 : 800)) return 0;
    return near_cheb_bytes(PYPO_MODE_JM, n_feed, n_dish);
}

int launch_adj_near(int precision, const NearWs &near, const void *feed64, int n_feed, const GridPtrs &dish,
                    int n_dish, double k, double tdir, double pref, double *partial, size_t partial_bytes, double *jd,
                    hipStream_t st) {
    NearWs w = near;
    w.nodes_only = true;
    const TileMeta *meta = (const TileMeta *)((const char *)feed64 + meta_offset(sizeof(SrcRec64), n_feed));
    // what the sums may launch; splits are grid.y, 65 536 at most, and a thousand
    // already fill the chip for one block of nodes
    const SumPlan p{1, std::min((n_dish + TILE - 1) / TILE, kNearMaxNodes / TILE), std::min(n_tiles(n_feed), 1024), TILE};
    const double carrier = tdir * k / kTwoPi;
    int err;
    if ((err = launch_near_cheb_plan(PYPO_MODE_JM, precision, PYPO_PREC_FP64, p, meta, n_feed, k, partial_bytes,
                                     currents_cycles(precision), w, st)) ||
        (err = launch_near_sum(PYPO_MODE_JM, PYPO_PREC_FP64, p, feed64, n_feed, dish, n_dish, k, tdir, partial, w,
                               st)) ||
        (err = launch_near_cheb_coef(PYPO_MODE_JM, partial, w, carrier, st)))
        return err;
    hipLaunchKernelGGL(k_adj_currents_series, dim3((n_dish + kNearEvalTargets - 1) / kNearEvalTargets), dim3(256), 0, st,
                       w, dish, n_dish, carrier, pref, jd);
    PYPO_CHECK_LAUNCH();
    return 0;
}

}  // namespace pypo
