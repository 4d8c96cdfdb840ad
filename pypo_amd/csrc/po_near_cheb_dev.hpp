// po_near_cheb_dev.hpp -- device parts of the near field's Chebyshev patches
// that the finish kernels (po_near.hip, po_scalar.hip) use: target coordinates,
// the carrier exp(j t k R), and the evaluation of a target's series.
#pragma once

#include "po_common.hpp"

namespace pypo {

// |p - c| as R + lo to twice FP64's precision: the carrier's phase k R of
// thousands of radians is taken out at the nodes and put back at the targets,
// and its rounding would be common to all sources of a target.
__device__ __forceinline__ void near_distance(const double *c, double px, double py, double pz, double (&u)[3],
                                              double &R, double &lo) {
    const double p[3] = {px, py, pz};
    double s = 0.0, r = 0.0;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const double d = p[q] - c[q];
        const double bb = p[q] - d;                                  // two-difference
        const double dl = (p[q] - (d + bb)) + (bb - c[q]);
        u[q] = d;
        const double sq = d * d;
        const double t = s + sq, tv = t - s;                         // two-sum
        r += (s - (t - tv)) + (sq - tv) + __builtin_fma(d, d, -sq) + 2.0 * d * dl;
        s = t;
    }
    R = sqrt(s);
    lo = (__builtin_fma(-R, R, s) + r) / (2.0 * R);
}

// exp(j 2 pi rev_scale (R + lo))
__device__ __forceinline__ void near_carrier(double rev_scale, double R, double lo, double &sn, double &cs) {
    const double rev = R * rev_scale;
    const double res = __builtin_fma(R, rev_scale, -rev) + lo * rev_scale;
    sincospi(2.0 * ((rev - __builtin_rint(rev)) + res), &sn, &cs);
}

// (a, b) of a direction in the plan's frame.
__device__ __forceinline__ void near_coords(const double (&e)[3][3], const double (&u)[3], double &a, double &b,
                                            double &theta) {
    double x[3];
#pragma unroll
    for (int q = 0; q < 3; q++) x[q] = e[q][0] * u[0] + e[q][1] * u[1] + e[q][2] * u[2];
    const double h = sqrt(x[0] * x[0] + x[1] * x[1]);
    theta = atan2(h, x[2]);
    const double f = h > 1e-200 ? theta / h : 0.0;
    a = x[0] * f;
    b = x[1] * f;
}

// Box of one workgroup's share of the targets, for the plan; a target that is
// not finite leaves NaN.
__device__ __forceinline__ void near_target_box(const NearWs &w, int block, float *scratch) {
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {INFINITY, INFINITY, INFINITY}, bad = 0.f;
    const double *p[3] = {w.tx, w.ty, w.tz};
#pragma unroll
    for (int j = 0; j < kNearBox / TILE; j++) {
        const int i = block * kNearBox + j * TILE + threadIdx.x;
        if (i >= w.n_tgt) break;
#pragma unroll
        for (int q = 0; q < 3; q++) {
            const float x = (float)p[q][i];
            lo[q] = fminf(lo[q], x);
            hi[q] = fminf(hi[q], -x);
            if (!(fabsf(x) < 1e30f)) bad = -1.f;
        }
    }
    bad = block_min(bad, scratch);
#pragma unroll
    for (int q = 0; q < 3; q++) {
        lo[q] = block_min(lo[q], scratch);
        hi[q] = -block_min(hi[q], scratch);
    }
    if (threadIdx.x == 0) {
        float *o = w.box + 6 * (size_t)(w.src_tiles() + block);
        for (int q = 0; q < 3; q++) { o[q] = lo[q]; o[3 + q] = hi[q]; }
        if (bad < 0.f) o[0] = __builtin_nanf("");
    }
}

// Patch of (a, b).
__device__ __forceinline__ int near_patch(const NearPlan &pl, double a, double b, int &ip, int &jp) {
    ip = min(pl.pa - 1, max(0, (int)((a - pl.a0) / pl.da)));
    jp = min(pl.pb - 1, max(0, (int)((b - pl.b0) / pl.db)));
    return ip * pl.pb + jp;
}

// The targets a near-field sum workgroup works on: the caller's, or the nodes
// of a plan that is on (then only the plan's first tblocks x splits workgroups
// have work; false: this one has none).  lit: no shadow test (at the nodes).
struct NearTargets {
    const double *x, *y, *z;
    int n, chunk, tb, sp;
    bool lit;
};
__device__ __forceinline__ bool near_targets(const NearWs &w, const double *x, const double *y, const double *z,
                                             int n_tgt, int chunk, NearTargets &o) {
    if (w.plan && w.plan->on) {
        const int lin = blockIdx.y * gridDim.x + blockIdx.x, nx = w.plan->tblocks, ny = w.plan->splits;
        if (lin >= nx * ny) return false;
        xcd_item(lin, nx, ny, o.tb, o.sp);
        o.x = w.x; o.y = w.y; o.z = w.z; o.n = w.plan->n; o.chunk = w.plan->chunk;
        o.lit = true;
        return true;
    }
    if (w.nodes_only) return false;
    xcd_item(o.tb, o.sp);
    o.x = x; o.y = y; o.z = z; o.n = n_tgt; o.chunk = chunk;
    o.lit = false;
    return true;
}

// Targets per workgroup of an evaluation: the four waves share the series'
// rows, so that a few ten thousand targets already fill the chip.
constexpr int kNearEvalTargets = 64;

// The target of this lane (every wave of the workgroup holds the same 64), and
// whether there is one.
__device__ __forceinline__ bool near_eval_target(const NearWs &w, int &t) {
    const int i = blockIdx.x * kNearEvalTargets + (threadIdx.x & 63);
    const int j = min(i, w.n_tgt - 1);
    t = w.plan->sorted ? w.perm[j] : j;
    return i < w.n_tgt;
}

// Field rows S[0..ROWS) at target t of a plan that is on, times exp(j t k R) /
// R; complete in wave 0 only.  Lanes of one patch go together: its coefficients
// are uniform then and come by scalar loads, ROWS + 1 FP64 FMAs a term, which
// is what bounds it once enough terms' loads are in flight: unrolled by 8, 4 and
// 3 instead of 2, scalar planes 157 -> 101 us, JM at 1 002 001 targets 250 -> 203,
// EHP at 640 800 380 -> 363 (more runs short of scalar registers or of terms).
template <int ROWS>
__device__ __forceinline__ void near_series(const NearWs &w, double rev_scale, int t, double (&S)[ROWS]) {
    constexpr int UNROLL = ROWS <= 2 ? 8 : (ROWS <= 6 ? 4 : 3);
    __shared__ double sh[3][ROWS][64];
    const NearPlan &pl = *w.plan;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double u[3], R, lo, a, b, theta;
    near_distance(pl.c, w.tx[t], w.ty[t], w.tz[t], u, R, lo);
    near_coords(pl.e, u, a, b, theta);
    const double s = 1.0 / R;
    int ip, jp;
    const int patch = near_patch(pl, a, b, ip, jp);
    const double x = fmin(1.0, fmax(-1.0, 2.0 * (a - pl.a0 - ip * pl.da) / pl.da - 1.0));
    const double y = fmin(1.0, fmax(-1.0, 2.0 * (b - pl.b0 - jp * pl.db) / pl.db - 1.0));
    const double z = fmin(1.0, fmax(-1.0, (s - pl.surface(a, b) - pl.s_mid) / pl.s_half));
#pragma unroll
    for (int q = 0; q < ROWS; q++) S[q] = 0.0;
    const int na = pl.na, nb = pl.nb, nr = pl.nr;
    const int m0 = wv * na / 4, m1 = (wv + 1) * na / 4;
    const double angle = acos(x);
    const double ts = cos(m0 * angle), tps = cos((m0 - 1) * angle);   // T_m0(x), T_(m0-1)(x)
    unsigned long long todo = ~0ull;
    while (todo) {
        const int pid = __builtin_amdgcn_readlane(patch, __builtin_ctzll(todo));
        const bool mine = patch == pid;
        todo &= ~__ballot(mine);
        if (mine) {
            double t0 = ts, tp = tps;
            for (int m = m0; m < m1; m++) {
                double v0 = 1.0, vp = z;
                for (int l = 0; l < nr; l++) {
                    // readfirstlane: uniform by construction, so that scalar loads are chosen
                    ConstDouble *c =
                        const_space(w.coef) + __builtin_amdgcn_readfirstlane(((pid * na + m) * nr + l) * nb * ROWS);
                    double r[ROWS], g = 1.0, gp = y;                      // T_0(y), T_(-1)(y) = T_1(y)
#pragma unroll
                    for (int q = 0; q < ROWS; q++) r[q] = 0.0;
#pragma unroll UNROLL
                    for (int i = 0; i < nb; i++) {
#pragma unroll
                        for (int q = 0; q < ROWS; q++) r[q] = __builtin_fma(g, c[ROWS * i + q], r[q]);
                        const double gn = __builtin_fma(2.0 * y, g, -gp);
                        gp = g;
                        g = gn;
                    }
                    const double f = t0 * v0;
#pragma unroll
                    for (int q = 0; q < ROWS; q++) S[q] = __builtin_fma(f, r[q], S[q]);
                    const double vn = __builtin_fma(2.0 * z, v0, -vp);
                    vp = v0;
                    v0 = vn;
                }
                const double tn = __builtin_fma(2.0 * x, t0, -tp);
                tp = t0;
                t0 = tn;
            }
        }
    }
    if (wv) {
#pragma unroll
        for (int q = 0; q < ROWS; q++) sh[wv - 1][q][lane] = S[q];
    }
    __syncthreads();
    if (wv) return;
    double sn, cs;
    near_carrier(rev_scale, R, lo, sn, cs);
    sn *= s;
    cs *= s;
#pragma unroll
    for (int q = 0; q < ROWS; q += 2) {
        const double re = S[q] + sh[0][q][lane] + sh[1][q][lane] + sh[2][q][lane];
        const double im = S[q + 1] + sh[0][q + 1][lane] + sh[1][q + 1][lane] + sh[2][q + 1][lane];
        S[q] = re * cs - im * sn;
        S[q + 1] = re * sn + im * cs;
    }
}

// The JM rows' series S (six rows) at target t with its directional derivative
// along n, both times the carrier: F = exp(j t k R) / R S(a, b, s) and
//   dF = exp(j t k R) / R [ (j t k - 1 / R) (n.R_hat) S + (n.grad) S ].
// The carrier's derivative is exact and k R times the rest, so the series'
// derivative matters at the 1e-3 level only.  Chebyshev derivatives by the
// differentiated recurrence T'_{i+1} = 2 T_i + 2 x T'_i - T'_{i-1}.  Complete in
// wave 0 only.
__device__ __forceinline__ void near_series_grad(const NearWs &w, double rev_scale, int t, const double (&n)[3],
                                                 double (&F)[6], double (&D)[6]) {
    constexpr int ROWS = 6;
    __shared__ double sh[3][2 * ROWS][64];
    const NearPlan &pl = *w.plan;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double u[3], R, lo, a, b, theta;
    near_distance(pl.c, w.tx[t], w.ty[t], w.tz[t], u, R, lo);
    near_coords(pl.e, u, a, b, theta);
    const double s = 1.0 / R;
    int ip, jp;
    const int patch = near_patch(pl, a, b, ip, jp);
    const double x = fmin(1.0, fmax(-1.0, 2.0 * (a - pl.a0 - ip * pl.da) / pl.da - 1.0));
    const double y = fmin(1.0, fmax(-1.0, 2.0 * (b - pl.b0 - jp * pl.db) / pl.db - 1.0));
    const double z = fmin(1.0, fmax(-1.0, (s - pl.surface(a, b) - pl.s_mid) / pl.s_half));
    // n.grad of x, y, z: in the frame, with (p, q) = sin(theta) (cos, sin)(phi)
    // the transverse direction cosines and c = cos(theta),
    //   a = f p, f = theta / sin(theta);   d p = (n_p - (n.R_hat) p) / R.
    double X[3], N[3];
#pragma unroll
    for (int q = 0; q < 3; q++) {
        X[q] = (pl.e[q][0] * u[0] + pl.e[q][1] * u[1] + pl.e[q][2] * u[2]) * s;
        N[q] = pl.e[q][0] * n[0] + pl.e[q][1] * n[1] + pl.e[q][2] * n[2];
    }
    const double nr = N[0] * X[0] + N[1] * X[1] + N[2] * X[2];
    const double h2 = X[0] * X[0] + X[1] * X[1], h = sqrt(h2);
    const double dp = (N[0] - nr * X[0]) * s, dq = (N[1] - nr * X[1]) * s, dc = (N[2] - nr * X[2]) * s;
    // theta = atan2(h, c): d theta = c dh - h dc; f = theta / h, d f = (d theta - f dh) / h
    const double f = h > 1e-9 ? theta / h : 1.0;
    const double dh = h > 1e-9 ? (X[0] * dp + X[1] * dq) / h : 0.0;
    const double df = h > 1e-4 ? (X[2] * dh - h * dc - f * dh) / h : 0.0;   // O(h) dh below
    const double ga = f * dp + df * X[0], gb = f * dq + df * X[1];
    const double dx = 2.0 * ga / pl.da, dy = 2.0 * gb / pl.db;
    const double sx = (a - pl.fa) * pl.ga, sy = (b - pl.fb) * pl.gb;
    const double dsurf = (pl.fit[1] + 2.0 * pl.fit[3] * sx + pl.fit[4] * sy) * pl.ga * ga +
                         (pl.fit[2] + 2.0 * pl.fit[5] * sy + pl.fit[4] * sx) * pl.gb * gb;
    const double dz = (-nr * s * s - dsurf) / pl.s_half;
#pragma unroll
    for (int q = 0; q < ROWS; q++) { F[q] = 0.0; D[q] = 0.0; }
    const int na = pl.na, nb = pl.nb, nz = pl.nr;
    const int m0 = wv * na / 4, m1 = (wv + 1) * na / 4;
    unsigned long long todo = ~0ull;
    while (todo) {
        const int pid = __builtin_amdgcn_readlane(patch, __builtin_ctzll(todo));
        const bool mine = patch == pid;
        todo &= ~__ballot(mine);
        if (mine) {
            double t0 = 1.0, tp = x, g0 = 0.0, gp = 1.0;   // T_0, T_{-1} = T_1; T'_0, T'_{-1} = T'_1
            for (int m = 0; m < m1; m++) {
                if (m >= m0) {
                    double v0 = 1.0, vp = z, e0 = 0.0, ep = 1.0;
                    for (int l = 0; l < nz; l++) {
                        ConstDouble *c =
                            const_space(w.coef) + __builtin_amdgcn_readfirstlane(((pid * na + m) * nz + l) * nb * ROWS);
                        double r[ROWS], rd[ROWS], k0 = 1.0, kp = y, j0 = 0.0, jp2 = 1.0;
#pragma unroll
                        for (int q = 0; q < ROWS; q++) { r[q] = 0.0; rd[q] = 0.0; }
#pragma unroll 4
                        for (int i = 0; i < nb; i++) {
#pragma unroll
                            for (int q = 0; q < ROWS; q++) {
                                r[q] = __builtin_fma(k0, c[ROWS * i + q], r[q]);
                                rd[q] = __builtin_fma(j0, c[ROWS * i + q], rd[q]);
                            }
                            const double jn = __builtin_fma(2.0 * y, j0, __builtin_fma(2.0, k0, -jp2));
                            const double kn = __builtin_fma(2.0 * y, k0, -kp);
                            jp2 = j0; j0 = jn;
                            kp = k0; k0 = kn;
                        }
                        const double c0 = t0 * v0, c1 = g0 * v0 * dx + t0 * e0 * dz, c2 = c0 * dy;
#pragma unroll
                        for (int q = 0; q < ROWS; q++) {
                            F[q] = __builtin_fma(c0, r[q], F[q]);
                            D[q] = __builtin_fma(c1, r[q], __builtin_fma(c2, rd[q], D[q]));
                        }
                        const double en = __builtin_fma(2.0 * z, e0, __builtin_fma(2.0, v0, -ep));
                        const double vn = __builtin_fma(2.0 * z, v0, -vp);
                        ep = e0; e0 = en;
                        vp = v0; v0 = vn;
                    }
                }
                const double gn = __builtin_fma(2.0 * x, g0, __builtin_fma(2.0, t0, -gp));
                const double tn = __builtin_fma(2.0 * x, t0, -tp);
                gp = g0; g0 = gn;
                tp = t0; t0 = tn;
            }
        }
    }
    if (wv) {
#pragma unroll
        for (int q = 0; q < ROWS; q++) { sh[wv - 1][q][lane] = F[q]; sh[wv - 1][ROWS + q][lane] = D[q]; }
    }
    __syncthreads();
    if (wv) return;
#pragma unroll
    for (int q = 0; q < ROWS; q++) {
        F[q] += sh[0][q][lane] + sh[1][q][lane] + sh[2][q][lane];
        D[q] += sh[0][ROWS + q][lane] + sh[1][ROWS + q][lane] + sh[2][ROWS + q][lane];
    }
    double sn, cs;
    near_carrier(rev_scale, R, lo, sn, cs);
    sn *= s;
    cs *= s;
    const double wr = -s * nr, wi = kTwoPi * rev_scale * nr;   // (j t k - 1 / R) n.R_hat
#pragma unroll
    for (int q = 0; q < ROWS; q += 2) {
        const double re = F[q], im = F[q + 1];
        const double dr = D[q] + wr * re - wi * im, di = D[q + 1] + wr * im + wi * re;
        F[q] = re * cs - im * sn;
        F[q + 1] = re * sn + im * cs;
        D[q] = dr * cs - di * sn;
        D[q + 1] = dr * sn + di * cs;
    }
}

}  // namespace pypo
