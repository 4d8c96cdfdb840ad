// po_near_cheb.hip -- the near field's Chebyshev patches (po_near_cheb.hpp):
// extents, frame, plan, split reduction of the node sums and their transform
// into coefficients.  The sums are the kernels of po_near.hip and po_scalar.hip;
// their finish kernels evaluate the series.

#include "po_near_cheb_dev.hpp"

#include <algorithm>

namespace pypo {
namespace {

constexpr float kNearCompact = 1.f / 3.f;   // largest rho / R of a plan that is on
constexpr float kNearWide = 1.5f;           // largest |a|, |b|

// Wave-wide minima of N values, step by step so that the exchanges of one step
// are in flight together.
template <int N>
__device__ __forceinline__ void wave_minima(float (&v)[N]) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        float x[N];
#pragma unroll
        for (int q = 0; q < N; q++) x[q] = __shfl_xor(v[q], o, 64);
#pragma unroll
        for (int q = 0; q < N; q++) v[q] = fminf(v[q], x[q]);
    }
}

// Middles and half extents of the N-dimensional boxes [b0, b1).
template <int N>
__device__ void near_extent(const float *box, int b0, int b1, float (*red)[9], double (&mid)[N], double (&half)[N],
                            bool &bad) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, waves = blockDim.x >> 6;
    float v[2 * N + 1];
#pragma unroll
    for (int q = 0; q <= 2 * N; q++) v[q] = q < 2 * N ? INFINITY : 0.f;
    for (int i = b0 + tid; i < b1; i += blockDim.x)
#pragma unroll
        for (int q = 0; q < 2 * N; q++) {
            const float x = q < N ? box[2 * N * i + q] : -box[2 * N * i + q];
            if (!(fabsf(x) < 1e30f)) v[2 * N] = -1.f;
            v[q] = fminf(v[q], x);
        }
    wave_minima(v);
    __syncthreads();
    if (lane == 0)
#pragma unroll
        for (int q = 0; q <= 2 * N; q++) red[wv][q] = v[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q <= 2 * N; q++)
        for (int i = 0; i < waves; i++) v[q] = fminf(v[q], red[i][q]);
    bad = v[2 * N] < 0.f;
#pragma unroll
    for (int q = 0; q < N; q++) {
        const double lo = v[q], hi = -(double)v[N + q];
        mid[q] = 0.5 * (lo + hi);
        half[q] = 0.5 * (hi - lo) + 2e-7 * fmax(fabs(lo), fabs(hi));   // widened by the FP32 rounding
    }
}

// Frame whose third axis points from the sources' centre to the targets'.
__device__ void near_frame(const double (&c)[3], const double (&tc)[3], double (&e)[3][3]) {
    double d[3] = {tc[0] - c[0], tc[1] - c[1], tc[2] - c[2]};
    const double n = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
    const double inv = n > 0.0 ? 1.0 / n : 0.0;
    for (int q = 0; q < 3; q++) d[q] *= inv;
    if (!(n > 0.0)) d[2] = 1.0;
    int m = 0;                                     // the axis least along d
    for (int q = 1; q < 3; q++)
        if (fabs(d[q]) < fabs(d[m])) m = q;
    double x[3];
    for (int q = 0; q < 3; q++) x[q] = (q == m ? 1.0 : 0.0) - d[m] * d[q];
    const double l = 1.0 / sqrt(x[0] * x[0] + x[1] * x[1] + x[2] * x[2]);
    for (int q = 0; q < 3; q++) { e[0][q] = x[q] * l; e[2][q] = d[q]; }
    e[1][0] = d[1] * e[0][2] - d[2] * e[0][1];
    e[1][1] = d[2] * e[0][0] - d[0] * e[0][2];
    e[1][2] = d[0] * e[0][1] - d[1] * e[0][0];
}

// Block-wide minima of N values; red: [4][N].
template <int N>
__device__ __forceinline__ void block_minima(float (&v)[N], float (*red)[9]) {
    static_assert(N <= 9, "rows of red");
    wave_minima(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int q = 0; q < N; q++) red[threadIdx.x >> 6][q] = v[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < N; q++) v[q] = fminf(fminf(red[0][q], red[1][q]), fminf(red[2][q], red[3][q]));
}

// A tile of sources that may not light all of the cone, or carries infinite currents.
__device__ __forceinline__ bool near_tile_off(const TileMeta &t, const Cone &cone) {
    return !(t.cmax < INFINITY) || cones_may_shadow(t.ax, t.ay, t.az, t.cos_half, cone);
}

__device__ __forceinline__ Cone near_cone(const double (&axis)[3], float theta, float near) {
    Cone cone;
    cone.ax = (float)axis[0]; cone.ay = (float)axis[1]; cone.az = (float)axis[2];
    const float ang = theta + asinf(near);   // widened by the sources' parallax
    cone.cos_half = ang < 1.57f ? cosf(ang) : -1.f;
    return cone;
}

constexpr int kNearSmall = 24;
struct NearIn {
    const TileMeta *meta;      // nullptr: scalar, no shadow test
    int n_tiles, n_src, n_tgt, slots, max_items, rows;
    long long max_partials;
    float kabs, q, p, log_eps;  // node count constants, ln(4 / eps)
    float dyadic;               // rate along s of the dyadic's 1 / (k R) and 1 / (k R)^2, 0: scalar
    float small[kNearSmall];    // small[n]: largest K for which n nodes do by the small-K bound
    float pair_cycles, direct_cycles, series_cycles, fixed_cycles, sort_cycles;   // sort_cycles: 0 where no sorting pass is launched
};

// Smallest n with 2 (K / 2)^n / n! <= eps (the remainder of the interpolant of
// a function of phase rate K), or the large-K rule.
__device__ float near_count(float K, const NearIn &in) {
    float n = ceilf(K + in.q * cbrtf(K) + in.p);
#pragma unroll
    for (int m = kNearSmall - 1; m >= 1; m--)
        if (K <= in.small[m]) n = fminf(n, (float)m);
    return n;
}

// Nodes along a direction axis of half-width h: see po_near_cheb.hpp.  x, y,
// z: half extents of the sources along the axis, the other one and e[2]; tilt:
// phase rate of the surface's slope.  Where the ellipse the large-K rule asks
// for is larger than `cap`, the bound 4 exp(rate(eta) eta) / (eta / h +
// sqrt((eta / h)^2 + 1))^n at the best eta within it.
__device__ float near_axis(const NearIn &in, float h, float x, float y, float z, float tilt, float lim, float lim_o,
                           float grow, float cap) {
    auto rate_at = [&](float eta) {
        const float ex = __expf(eta), ch = 0.5f * (ex + 1.f / ex);
        return ch * (grow * in.kabs * (x + y * fminf(1.f, (lim + eta) * lim_o * (1.f / 3.f)) + z * (lim + eta)) + tilt +
                     2.f);
    };
    float eta = 0.f, n = 1.f;
    for (int it = 0; it < 4; it++) {
        const float rate = rate_at(eta), K = rate * h * 1.00001f;
        n = near_count(K, in);
        eta = fminf(cap, sqrtf(fmaxf(0.f, n * n - K * K)) / fmaxf(rate, 1e-30f));
    }
    if (eta >= cap) {
        n = 1e6f;
        for (int i = 1; i <= 8; i++) {
            const float q = 0.125f * i * cap, r = q / h;
            n = fminf(n, ceilf((in.log_eps + rate_at(q) * q) / __logf(r + sqrtf(r * r + 1.f))));
        }
    }
    return n;
}

// Rates and radial nodes of a box: half widths and largest |a|, |b|, the
// sources' half extents along the frame and rho, the largest 1 / R, the half
// width in s and the surface's slope.
struct NearGeo {
    float ha, hb, la, lb, ex, ey, ez, grow, tilt, cap;
    int nr;
};
__device__ __forceinline__ NearGeo near_geo(const NearIn &in, float ha, float hb, float la, float lb,
                                            const float (&ext)[4], float r1, float hs, float slope) {
    NearGeo g{ha, hb, la, lb, ext[0], ext[1], ext[2]};
    const float rho = ext[3], near = rho * r1;
    g.grow = 1.f / (1.f - fminf(near, 0.5f));
    // radial phase and amplitude rates per unit of s: those that vanish with the
    // sources' extent, and with the dyadic's own
    const float smooth = 1.1f * g.grow * g.grow * in.kabs * 0.5f * rho * rho + 2.f * rho * g.grow;
    const float radial = smooth + in.dyadic;
    g.tilt = radial * slope;
    g.cap = fminf(1.5f, 0.8f * acoshf(1.f / near));
    // no further than four fifths of the way to the singularity at s = 1 / rho
    const float far = 1.f + fmaxf(0.f, (0.8f / rho - r1) / hs);
    const float least = ceilf(in.log_eps / __logf(far + sqrtf(far * far - 1.f)));
    // the dyadic is a polynomial of degree two in s: two more nodes always do
    g.nr = (int)fminf(fmaxf(near_count(smooth * hs, in), least) + 2.f, fmaxf(near_count(radial * hs, in), least));
    return g;
}

// The nodes of choice `at` of the patches (16 x 16), and the issue cycles of 64
// lanes of their sums and of the series at the targets (7 cycles an FMA with its
// scalar loads, measured) where a wave meets one patch; false: too many nodes.
__device__ __forceinline__ bool near_cost(const NearIn &in, const NearGeo &g, int at, float &na, float &nb, float &nodes,
                                          float &one) {
    const int pa = at / kNearMaxPatches + 1, pb = at % kNearMaxPatches + 1;
    na = near_axis(in, g.ha / pa, g.ex, g.ey, g.ez, g.tilt, g.la, g.lb, g.grow, g.cap);
    nb = near_axis(in, g.hb / pb, g.ey, g.ex, g.ez, g.tilt, g.lb, g.la, g.grow, g.cap);
    const float each = na * nb * g.nr, all = each * pa * pb;
    nodes = ceilf(all * (1.f / 256.f)) * 4.f * in.n_src * in.pair_cycles;
    one = in.n_tgt * (1.f / 64.f) * each * (in.rows + 1) * in.series_cycles;
    return na <= kNearMaxAxis && nb <= kNearMaxAxis && g.nr <= kNearMaxRadial && all <= kNearMaxNodes && all <= in.n_tgt;
}

// Whether that pays against the sums at the targets.
__device__ __forceinline__ bool near_pays(const NearIn &in, float cost) {
    return cost + in.fixed_cycles < 0.7f * (in.n_tgt * (1.f / 64.f) * (float)in.n_src * in.direct_cycles);
}

// One workgroup: the frame, and the quadratic surface through 256 of the
// targets (scattered over their order by the golden ratio).  Any coefficients
// are right, good ones make s small: a singular fit drops terms.  Where those
// targets alone already turn the plan off (too near, too wide, in shadow, too
// many nodes for their box), so would all of them: the kernels behind see that and return.
static_assert(kNearMaxPatches * kNearMaxPatches == 256, "one choice a lane");
__global__ __launch_bounds__(256) void k_near_frame(NearIn in, NearWs w) {
    __shared__ float red[4][9];
    __shared__ double sum[4][32], surface[6];
    double c[3], half[3], tc[3], th[3], e[3][3];
    bool bad, bad_t;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    if (tid == 0) w.plan->on = 0;
    const double g = tid * 0.6180339887498949;
    const int t = min(w.n_tgt - 1, (int)((g - floor(g)) * w.n_tgt));
    const double p[3] = {w.tx[t], w.ty[t], w.tz[t]};
    near_extent<3>(w.box, 0, w.src_tiles(), red, c, half, bad);
    near_extent<3>(w.box, w.src_tiles(), w.src_tiles() + w.tgt_blocks(), red, tc, th, bad_t);
    if (bad || bad_t) return;
    near_frame(c, tc, e);
    const double u[3] = {p[0] - c[0], p[1] - c[1], p[2] - c[2]};
    const double s = 1.0 / sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
    const double rho = sqrt(half[0] * half[0] + half[1] * half[1] + half[2] * half[2]);
    double a, b, theta;
    near_coords(e, u, a, b, theta);
    float v[6] = {(float)a, (float)b, -(float)a, -(float)b, -(float)theta, -(float)s};
    block_minima(v, red);
    const float la = v[0], lb = v[1], ha = -v[2], hb = -v[3], near = (float)rho * -v[5];
    bool off = !(near <= kNearCompact && fmaxf(fmaxf(-la, ha), fmaxf(-lb, hb)) <= kNearWide);
    if (in.meta && !off) {
        const Cone cone = near_cone(e[2], -v[4], near);
        for (int i = tid; i < in.n_tiles; i += 256) off |= near_tile_off(in.meta[i], cone);
    }
    if (__syncthreads_or(off)) return;
    const double fa = 0.5 * ((double)la + ha), fb = 0.5 * ((double)lb + hb);
    const double ga = 2.0 / fmax((double)ha - la, 1e-9), gb = 2.0 / fmax((double)hb - lb, 1e-9);
    const double x = (a - fa) * ga, y = (b - fb) * gb;
    const double f[7] = {1.0, x, y, x * x, x * y, y * y, s};
    // normal equations: the 27 products, summed over the workgroup
    double prod[27];
    int k = 0;
#pragma unroll
    for (int i = 0; i < 6; i++)
#pragma unroll
        for (int j = i; j < 7; j++, k++) prod[k] = f[i] * f[j];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        double x[27];
#pragma unroll
        for (int q = 0; q < 27; q++) x[q] = __shfl_xor(prod[q], o, 64);
#pragma unroll
        for (int q = 0; q < 27; q++) prod[q] += x[q];
    }
    if (lane == 0)
#pragma unroll
        for (int q = 0; q < 27; q++) sum[wv][q] = prod[q];
    __syncthreads();
    if (tid == 0) {
        double m[6][7];
        k = 0;
#pragma unroll
        for (int i = 0; i < 6; i++)
#pragma unroll
            for (int j = i; j < 7; j++, k++) {
                m[i][j] = sum[0][k] + sum[1][k] + sum[2][k] + sum[3][k];
                if (j < 6) m[j][i] = m[i][j];
            }
        // Gauss-Jordan with the diagonal as pivot (symmetric positive semi-definite)
        bool used[6];
#pragma unroll
        for (int p = 0; p < 6; p++) {
            used[p] = m[p][p] > 1e-9 * 256.0;
            if (!used[p]) continue;
            const double inv = 1.0 / m[p][p];
#pragma unroll
            for (int j = 0; j < 7; j++) m[p][j] *= inv;
#pragma unroll
            for (int i = 0; i < 6; i++) {
                if (i == p) continue;
                const double q = m[i][p];
#pragma unroll
                for (int j = 0; j < 7; j++) m[i][j] -= q * m[p][j];
            }
        }
#pragma unroll
        for (int q = 0; q < 6; q++) surface[q] = used[q] ? m[q][6] : 0.0;
    }
    __syncthreads();
    double ext[4];
    for (int q = 0; q < 3; q++)
        ext[q] = fabs(e[q][0]) * half[0] + fabs(e[q][1]) * half[1] + fabs(e[q][2]) * half[2];
    ext[3] = rho;
    {
        // the plan's cost for these targets alone, no slope, patches met one by one
        double res = s;
#pragma unroll
        for (int q = 0; q < 6; q++) res -= surface[q] * f[q];
        float r[4] = {(float)res, -(float)res, (float)s, -(float)s};
        block_minima(r, red);
        const float hs = fmaxf(fminf(-r[1] - r[0], -r[3] - r[2]) * 0.5f, -1e-7f * r[3]);
        const float ex[4] = {(float)ext[0], (float)ext[1], (float)ext[2], (float)ext[3]};
        const NearGeo geo = near_geo(in, fmaxf(0.5f * (ha - la), 1e-6f), fmaxf(0.5f * (hb - lb), 1e-6f), fmaxf(-la, ha),
                                     fmaxf(-lb, hb), ex, -r[3], hs, 0.f);
        float na, nb, nodes, one;
        const bool ok = near_cost(in, geo, tid, na, nb, nodes, one);
        if (!__syncthreads_or(ok && near_pays(in, nodes + one))) return;
    }
    if (tid) return;
    NearPlan &pl = *w.plan;
    pl.on = 1;
    for (int q = 0; q < 3; q++) {
        pl.c[q] = c[q];
        for (int r = 0; r < 3; r++) pl.e[q][r] = e[q][r];
    }
    for (int q = 0; q < 4; q++) pl.ext[q] = ext[q];
    for (int q = 0; q < 6; q++) pl.fit[q] = surface[q];
    pl.fa = fa; pl.fb = fb; pl.ga = ga; pl.gb = gb;
}

// One workgroup: decide, choose the patches, write the plan.  A kernel of its
// own: as the last workgroup of k_near_cones, behind a fence in each of them, it
// saved a launch but took 20 us more at 1 002 001 targets.
__global__ __launch_bounds__(1024) void k_near_plan(NearIn in, NearWs w) {
    __shared__ float red[16][9];
    __shared__ float spread[16][4];
    __shared__ unsigned short nodes_a[kNearMaxPatches * kNearMaxPatches], nodes_b[kNearMaxPatches * kNearMaxPatches];
    __shared__ NearPlan pl;
    __shared__ unsigned long long best;
    __shared__ int shadow;
    const int tid = threadIdx.x, lane = tid & 63;
    double mid[4], half[4];
    bool bad;
    if (!w.plan->on) return;
    if (tid == 0) {
        pl = *w.plan;
        best = ~0ull;
        shadow = 0;
    }
    float theta = 0.f, ea = 0.f, eb = 0.f, waves = 0.f;
    for (int i = tid; i < w.tgt_blocks(); i += 1024) {
        theta = fmaxf(theta, w.theta[4 * i]);
        ea += w.theta[4 * i + 1]; eb += w.theta[4 * i + 2]; waves += w.theta[4 * i + 3];
    }
    theta = -wave_min(-theta);
    ea = wave_sum(ea);
    eb = wave_sum(eb);
    waves = wave_sum(waves);
    if (lane == 0) {
        float *o = spread[tid >> 6];
        o[0] = theta; o[1] = ea; o[2] = eb; o[3] = waves;
    }
    near_extent<4>(w.cone, 0, w.tgt_blocks(), red, mid, half, bad);
    ea = eb = waves = 0.f;
    for (int i = 0; i < 16; i++) {
        theta = fmaxf(theta, spread[i][0]);
        ea += spread[i][1]; eb += spread[i][2]; waves += spread[i][3];
    }
    ea /= waves;
    eb /= waves;
    const float ex = (float)pl.ext[0], ey = (float)pl.ext[1], ez = (float)pl.ext[2], rho = (float)pl.ext[3];
    const float la = (float)(fabs(mid[0]) + half[0]), lb = (float)(fabs(mid[1]) + half[1]);
    // The surface over the whole box, node corners included: 1 / R between r0
    // and r1 there; a fit that would leave the range of the targets by a factor
    // of two is dropped.
    float r1 = (float)(mid[2] + half[2]), r0 = (float)(mid[2] - half[2]), slope = 0.f;
    bool fit;
    {
        const double xa = fabs((mid[0] - pl.fa) * pl.ga) + half[0] * pl.ga;
        const double xb = fabs((mid[1] - pl.fb) * pl.gb) + half[1] * pl.gb;
        const double *f = pl.fit;
        const double lin = fabs(f[1]) * xa + fabs(f[2]) * xb + fabs(f[4]) * xa * xb;
        const double lo = f[0] - lin + fmin(0.0, f[3]) * xa * xa + fmin(0.0, f[5]) * xb * xb + mid[3] - half[3];
        const double hi = f[0] + lin + fmax(0.0, f[3]) * xa * xa + fmax(0.0, f[5]) * xb * xb + mid[3] + half[3];
        fit = lo > 0.5 * r0 && hi < 2.0 * r1;
        if (fit) {
            r0 = fminf(r0, (float)lo);
            r1 = fmaxf(r1, (float)hi);
            slope = (float)fmax((fabs(f[1]) + 2.0 * fabs(f[3]) * xa + fabs(f[4]) * xb) * pl.ga,
                                (fabs(f[2]) + 2.0 * fabs(f[5]) * xb + fabs(f[4]) * xa) * pl.gb);
        }
    }
    const float near = rho * r1;
    bool on = !bad && la <= kNearWide && lb <= kNearWide && r0 > 0.f && near <= kNearCompact;
    if (on && in.meta) {
        // every source lights every target
        const Cone cone = near_cone(pl.e[2], theta, near);
        for (int i = tid; i < in.n_tiles; i += 1024)
            if (near_tile_off(in.meta[i], cone)) shadow = 1;
    }
    __syncthreads();
    on = on && !shadow;
    const float ha = fmaxf((float)half[0], 1e-6f), hb = fmaxf((float)half[1], 1e-6f);
    const float hs = fmaxf((float)half[fit ? 3 : 2], 1e-7f * r1);
    int nr = 0;
    if (on) {
        const float ext[4] = {ex, ey, ez, rho};
        const NearGeo geo = near_geo(in, ha, hb, la, lb, ext, r1, hs, slope);
        nr = geo.nr;
        if (tid < kNearMaxPatches * kNearMaxPatches) {
            float na, nb, nodes, one;
            const bool ok = near_cost(in, geo, tid, na, nb, nodes, one);
            nodes_a[tid] = (unsigned short)fminf(na, 1e4f);
            nodes_b[tid] = (unsigned short)fminf(nb, 1e4f);
            const int pa = tid / kNearMaxPatches + 1, pb = tid % kNearMaxPatches + 1;
            // a wave's targets meet several patches in grid order
            const float met = (1.f + ea * pa / (2.f * ha)) * (1.f + eb * pb / (2.f * hb));
            const float plain = one * (pa * pb > 1 ? met : 1.f);
            const float sorted = in.sort_cycles > 0.f ? one * 1.1f + in.sort_cycles : INFINITY;
            const float cost = nodes + fminf(plain, sorted);
            if (ok && near_pays(in, cost))
                atomicMin(&best, (unsigned long long)__float_as_uint(cost) << 32 | (sorted < plain ? 1u << 31 : 0u) |
                                     (unsigned)tid);
        }
    }
    __syncthreads();
    on = on && best != ~0ull;
    if (!on) {
        if (tid == 0) w.plan->on = 0;
        return;
    }
    const unsigned who = (unsigned)best;
    if (tid == 0) {
        const int chosen = who & 0xffff;
        pl.pa = chosen / kNearMaxPatches + 1;
        pl.pb = chosen % kNearMaxPatches + 1;
        pl.na = nodes_a[chosen];
        pl.nb = nodes_b[chosen];
        pl.nr = nr;
        pl.n = pl.pa * pl.pb * pl.na * pl.nb * nr;
        pl.on = 1;
        pl.sorted = who >> 31;
        pl.tblocks = (pl.n + TILE - 1) / TILE;
        pl.a0 = mid[0] - ha; pl.b0 = mid[1] - hb;
        pl.da = 2.0 * ha / pl.pa; pl.db = 2.0 * hb / pl.pb;
        if (!fit)
            for (int q = 0; q < 6; q++) pl.fit[q] = 0.0;
        pl.s_mid = mid[fit ? 3 : 2];
        pl.s_half = hs;
    }
    __syncthreads();   // every thread has read best
    if (tid == 0) best = ~0ull;
    __syncthreads();
    // Source splits of the node sums, as in the far field's plan.
    unsigned long long mine = ~0ull;
    for (int ct = tid + 1; ct <= in.n_tiles; ct += 1024) {
        const unsigned used = (in.n_tiles + ct - 1) / ct, items = used * pl.tblocks;
        if (items > (unsigned)in.max_items || used * (long long)in.rows * pl.n > in.max_partials) continue;
        const unsigned long long rounds = (items + in.slots - 1) / in.slots;
        mine = min(mine, rounds * (10ull * ct + 1) << 32 | (unsigned)ct);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) mine = min(mine, __shfl_xor(mine, o, 64));
    if (lane == 0) atomicMin(&best, mine);
    __syncthreads();
    const int ct = best == ~0ull ? in.n_tiles : (int)(best & 0xffffffffu);
    if (tid == 0) {
        pl.chunk = ct * TILE;
        pl.splits = (in.n_tiles + ct - 1) / ct;
        *w.plan = pl;
    }
}

// Box of kNearBox targets per workgroup in (a, b, 1/R, s), their largest
// theta, and how far a wave's 64 consecutive targets spread.
__global__ __launch_bounds__(256) void k_near_cones(NearWs w) {
    __shared__ float scratch[4];
    __shared__ float red[4][9];
    const NearPlan &pl = *w.plan;
    if (!pl.on) return;
    float v[9], ea = 0.f, eb = 0.f, waves = 0.f;
#pragma unroll
    for (int q = 0; q < 9; q++) v[q] = INFINITY;
#pragma unroll 1
    for (int j = 0; j < kNearBox / 256; j++) {
        const int t = blockIdx.x * kNearBox + j * 256 + threadIdx.x;
        if (__ballot(t < w.n_tgt) == 0ull) break;
        const int i = min(t, w.n_tgt - 1);
        const double u[3] = {w.tx[i] - pl.c[0], w.ty[i] - pl.c[1], w.tz[i] - pl.c[2]};
        const double r = 1.0 / sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
        double a, b, theta;
        near_coords(pl.e, u, a, b, theta);
        const float fa = (float)a, fb = (float)b, fr = (float)r, fs = (float)(r - pl.surface(a, b));
        v[0] = fminf(v[0], fa); v[4] = fminf(v[4], -fa);
        v[1] = fminf(v[1], fb); v[5] = fminf(v[5], -fb);
        v[2] = fminf(v[2], fr); v[6] = fminf(v[6], -fr);
        v[3] = fminf(v[3], fs); v[7] = fminf(v[7], -fs);
        v[8] = fminf(v[8], -(float)theta);
        ea -= wave_min(fa) + wave_min(-fa);
        eb -= wave_min(fb) + wave_min(-fb);
        waves += 1.f;
    }
    block_minima(v, red);
    const bool first = (threadIdx.x & 63) == 0;
    ea = block_sum(first ? ea : 0.f, scratch);
    eb = block_sum(first ? eb : 0.f, scratch);
    waves = block_sum(first ? waves : 0.f, scratch);
    if (threadIdx.x == 0) {
        for (int q = 0; q < 8; q++) w.cone[8 * blockIdx.x + q] = q < 4 ? v[q] : -v[q];
        float *o = w.theta + 4 * blockIdx.x;
        o[0] = -v[8]; o[1] = ea; o[2] = eb; o[3] = waves;
    }
}

__global__ __launch_bounds__(256) void k_near_nodes(NearWs w) {
    if (!w.plan->on) return;
    const NearPlan &pl = *w.plan;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < pl.n; i += gridDim.x * 256) {
        const int ib = i % pl.nb, ir = i / pl.nb % pl.nr, ia = i / (pl.nb * pl.nr) % pl.na;
        const int patch = i / (pl.nb * pl.nr * pl.na), ip = patch / pl.pb, jp = patch - ip * pl.pb;
        const double a = pl.a0 + pl.da * (ip + 0.5 + 0.5 * cospi((2 * ia + 1) / (2.0 * pl.na)));
        const double b = pl.b0 + pl.db * (jp + 0.5 + 0.5 * cospi((2 * ib + 1) / (2.0 * pl.nb)));
        const double R = 1.0 / (pl.surface(a, b) + pl.s_mid + pl.s_half * cospi((2 * ir + 1) / (2.0 * pl.nr)));
        const double th = hypot(a, b), f = th > 0.0 ? sin(th) / th : 1.0, x = R * a * f, y = R * b * f, z = R * cos(th);
        w.x[i] = pl.c[0] + x * pl.e[0][0] + y * pl.e[1][0] + z * pl.e[2][0];
        w.y[i] = pl.c[1] + x * pl.e[0][1] + y * pl.e[1][1] + z * pl.e[2][1];
        w.z[i] = pl.c[2] + x * pl.e[0][2] + y * pl.e[1][2] + z * pl.e[2][2];
    }
}

// ---- targets patch by patch: counts and ranks per bin, positions, order ----
__global__ __launch_bounds__(1024) void k_near_bin(NearWs w) {
    if (!w.plan->on || !w.plan->sorted) return;
    __shared__ int hist[kNearMaxPatches * kNearMaxPatches];
    const NearPlan &pl = *w.plan;
    if (threadIdx.x < kNearMaxPatches * kNearMaxPatches) hist[threadIdx.x] = 0;
    __syncthreads();
#pragma unroll 1
    for (int j = 0; j < kNearBin / 1024; j++) {
        const int t = blockIdx.x * kNearBin + j * 1024 + threadIdx.x;
        if (t >= w.n_tgt) break;
        const double u[3] = {w.tx[t] - pl.c[0], w.ty[t] - pl.c[1], w.tz[t] - pl.c[2]};
        double a, b, theta;
        near_coords(pl.e, u, a, b, theta);
        int ip, jp;
        const int p = near_patch(pl, a, b, ip, jp);
        w.slot[t] = (unsigned)p << 16 | (unsigned)atomicAdd(&hist[p], 1);
    }
    __syncthreads();
    if ((int)threadIdx.x < pl.pa * pl.pb) w.count[(size_t)threadIdx.x * w.bins() + blockIdx.x] = hist[threadIdx.x];
}

// Exclusive sums of the counts, patch after patch (one workgroup).
__global__ __launch_bounds__(1024) void k_near_scan(NearWs w) {
    if (!w.plan->on || !w.plan->sorted) return;
    __shared__ int part[16];
    const int n = w.plan->pa * w.plan->pb * w.bins(), tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    int base = 0;
    for (int i0 = 0; i0 < n; i0 += 4096) {
        int v[4], s = 0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int i = i0 + 4 * tid + q;
            v[q] = i < n ? w.count[i] : 0;
            s += v[q];
        }
        int x = s;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        __syncthreads();
        if (lane == 63) part[wv] = x;
        __syncthreads();
        int before = base, total = 0;
        for (int q = 0; q < 16; q++) {
            if (q < wv) before += part[q];
            total += part[q];
        }
        int at = before + x - s;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int i = i0 + 4 * tid + q;
            if (i < n) w.count[i] = at;
            at += v[q];
        }
        base += total;
    }
}

__global__ __launch_bounds__(256) void k_near_order(NearWs w) {
    if (!w.plan->on || !w.plan->sorted) return;
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= w.n_tgt) return;
    const unsigned s = w.slot[t];
    w.perm[w.count[(size_t)(s >> 16) * w.bins() + t / kNearBin] + (int)(s & 0xffff)] = t;
}

// Split reduction of the node sums, times R exp(-j t k R): f[row][node]; one
// lane per node and complex component.  row0: first row the sums write.
__global__ __launch_bounds__(256) void k_near_reduce(const double *__restrict__ partial, NearWs w, double rev_scale,
                                                     int stride, int row0, int rows) {
    if (!w.plan->on) return;
    const NearPlan &pl = *w.plan;
    const int n = pl.n, splits = pl.splits;
    for (int e = blockIdx.x * 256 + threadIdx.x; e < rows / 2 * n; e += gridDim.x * 256) {
        const int a = e / n, i = e - a * n;
        const double *p = partial + (size_t)(row0 + 2 * a) * n + i;
        double re = 0.0, im = 0.0;
#pragma unroll 4
        for (int s = 0; s < splits; s++) {
            re += p[(size_t)s * stride * n];
            im += p[(size_t)s * stride * n + n];
        }
        double u[3], R, lo, sn, cs;
        near_distance(pl.c, w.x[i], w.y[i], w.z[i], u, R, lo);
        near_carrier(-rev_scale, R, lo, sn, cs);
        sn *= R;
        cs *= R;
        w.f[(size_t)(2 * a) * n + i] = re * cs - im * sn;
        w.f[(size_t)(2 * a + 1) * n + i] = re * sn + im * cs;
    }
}

// Chebyshev coefficients: one row ka of one real component of a patch is
// transformed along a, then b, then s.  Rows of up to 64 (b, s) points go four
// to a workgroup, one per wave, larger ones take all of it (64 patches of 13 x
// 13 x 2: one row per workgroup left nine lanes in ten idle, 68 us).
__global__ __launch_bounds__(256) void k_near_coef(NearWs w, int rows) {
    constexpr int kPlane = kNearMaxAxis * kNearMaxRadial;
    __shared__ double ca[4 * kNearMaxAxis], cb[4 * kNearMaxAxis], cr[4 * kNearMaxRadial];
    __shared__ double gs[kPlane], hs[kPlane];
    if (!w.plan->on) return;
    const NearPlan &pl = *w.plan;
    const int na = pl.na, nb = pl.nb, nr = pl.nr, plane = nb * nr;
    for (int j = threadIdx.x; j < 4 * na; j += 256) ca[j] = cospi(j / (2.0 * na));
    for (int j = threadIdx.x; j < 4 * nb; j += 256) cb[j] = cospi(j / (2.0 * nb));
    for (int j = threadIdx.x; j < 4 * nr; j += 256) cr[j] = cospi(j / (2.0 * nr));
    const int size = plane <= 64 ? 64 : 256, groups = 256 / size;
    const int group = threadIdx.x / size, tid = threadIdx.x % size;
    double *g = gs + group * 64, *h = hs + group * 64;
    const int items = pl.pa * pl.pb * rows * na;
    for (int first = blockIdx.x * groups; first < items; first += gridDim.x * groups) {
        const int item = first + group, n = item < items ? plane : 0;
        const int ka = item % na, q = item / na % rows, patch = item / (na * rows);
        __syncthreads();
        for (int e = tid; e < n; e += size) {
            const double *f = w.f + (size_t)q * pl.n + (size_t)patch * na * plane + e;
            double s = 0.0;
            int j = ka;                        // ka (2 m + 1) mod 4 na
            for (int m = 0; m < na; m++) {
                s = __builtin_fma(f[(size_t)m * plane], ca[j], s);
                j += 2 * ka;
                if (j >= 4 * na) j -= 4 * na;
            }
            g[e] = s * (ka ? 2.0 : 1.0) / na;
        }
        __syncthreads();
        for (int e = tid; e < n; e += size) {
            const int ir = e / nb, kb = e - ir * nb;
            double s = 0.0;
            int j = kb;
            for (int m = 0; m < nb; m++) {
                s = __builtin_fma(g[ir * nb + m], cb[j], s);
                j += 2 * kb;
                if (j >= 4 * nb) j -= 4 * nb;
            }
            h[e] = s * (kb ? 2.0 : 1.0) / nb;
        }
        __syncthreads();
        for (int e = tid; e < n; e += size) {
            const int kr = e / nb, kb = e - kr * nb;
            double s = 0.0;
            int j = kr;
            for (int m = 0; m < nr; m++) {
                s = __builtin_fma(h[m * nb + kb], cr[j], s);
                j += 2 * kr;
                if (j >= 4 * nr) j -= 4 * nr;
            }
            w.coef[(((size_t)patch * na + ka) * plane + e) * rows + q] = s * (kr ? 2.0 : 1.0) / nr;
        }
    }
}

size_t up256(size_t b) { return (b + 255) / 256 * 256; }

int near_rows(int mode) { return mode == PYPO_MODE_SCALAR ? 2 : (mode == PYPO_MODE_JM ? 6 : 12); }

// Issue cycles of a SIMD for 64 pairs, from the rates the sums reach on MI355X
// (JM 5.2e11, other near modes 3.2e11, FP64 2.4e11 and 1.7e11, scalar 1.3e12 and 4.1e11
// pairs/s).
double pair_cycles(int mode, int precision) {
    if (mode == PYPO_MODE_SCALAR) return precision == PYPO_PREC_FP64 ? 384 : 121;
    if (precision == PYPO_PREC_FP64) return mode == PYPO_MODE_JM ? 650 : 900;
    return mode == PYPO_MODE_JM ? 300 : 490;
}

// Targets from which their order by patches is worth three more passes (some
// 15 us and 25 ns per thousand targets): 1 002 001 dish points of a JM, 13 x
// 13 x 3 nodes a patch and three patches a wave in grid order, 545 us.
constexpr int kNearSortTargets = 200000;

}  // namespace

// Tried where the sums at the targets take 300 us or more, 500 us with E: the
// passes around them are some 60 us where the plan is on.  Off, they are 5 to 15
// us where 256 targets show that (too near, too wide, in shadow: JM 745 -> 748 us,
// EH 1046 -> 1053, scalar 366 -> 381) and 22 where their box asks for too many
// nodes (JM 549 -> 571, scalar 352 -> 376; 45 without the early word).  From 1 ms only in
// FP64 (its node counts seldom pay below: 961 sources -> 90 300 targets stayed
// off), and for fewer sources than five times a patch's series costs at a
// target at the node counts that a wavelength across a patch takes, 13^2 x 2
// in three patches a wave.
bool near_cheb_try(int mode, int precision, int n_src, int n_tgt) {
    const double cycles = pair_cycles(mode, precision);
    const double us = (double)n_src * n_tgt / 64 * cycles / kSimdHz * 1e6;
    const double series = 13 * 13 * 2 * (near_rows(mode) + 1) * 7.0 * 3.0;
    const bool early = precision != PYPO_PREC_FP64 && n_src * cycles >= 5 * series;
    return mode != PYPO_MODE_FF && n_tgt >= 1024 && us >= (!early ? 1000 : near_rows(mode) == 12 ? 500 : 300);
}

size_t near_cheb_bytes(int mode, int n_src, int n_tgt) {
    const size_t cap = std::min(kNearMaxNodes, n_tgt);
    const size_t tb = (n_tgt + kNearBox - 1) / kNearBox;
    size_t b = 1024 + up256((n_tiles(n_src) + tb) * 6 * sizeof(float)) + up256(tb * 12 * sizeof(float)) +
               up256((3 + 2 * (size_t)near_rows(mode)) * cap * sizeof(double));
    if (n_tgt >= kNearSortTargets)
        b += up256((size_t)n_tgt * 8) +
             up256(((size_t)n_tgt + kNearBin - 1) / kNearBin * kNearMaxPatches * kNearMaxPatches * sizeof(int));
    return b;
}

NearWs near_cheb_carve(void *base, int mode, int n_src, const GridPtrs &ct, int n_tgt) {
    static_assert(sizeof(NearPlan) <= 1024, "room of the plan");
    const size_t cap = std::min(kNearMaxNodes, n_tgt);
    char *b = (char *)base;
    NearWs w;
    w.tx = ct.x; w.ty = ct.y; w.tz = ct.z;
    w.n_src = n_src; w.n_tgt = n_tgt;
    const size_t tb = w.tgt_blocks();
    w.plan = (NearPlan *)b;
    b += 1024;
    w.box = (float *)b;
    b += up256((w.src_tiles() + tb) * 6 * sizeof(float));
    w.cone = (float *)b;
    w.theta = w.cone + 8 * tb;
    b += up256(tb * 12 * sizeof(float));
    w.x = (double *)b;
    w.y = w.x + cap;
    w.z = w.y + cap;
    w.f = w.z + cap;
    w.coef = w.f + near_rows(mode) * cap;
    b += up256((3 + 2 * (size_t)near_rows(mode)) * cap * sizeof(double));
    if (n_tgt >= kNearSortTargets) {
        w.slot = (unsigned *)b;
        w.perm = (int *)b + n_tgt;
        b += up256((size_t)n_tgt * 8);
        w.count = (int *)b;
    }
    return w;
}

int launch_near_cheb_plan(int mode, int precision, int sums, const SumPlan &p, const TileMeta *meta, int n_src,
                          double kabs, size_t partial_bytes, double direct_cycles, const NearWs &w, hipStream_t st) {
    const bool f64 = precision == PYPO_PREC_FP64;
    NearIn in;
    in.meta = mode == PYPO_MODE_SCALAR ? nullptr : meta;
    in.n_tiles = n_tiles(n_src);
    in.n_src = n_src; in.n_tgt = w.n_tgt;
    in.slots = near_wgs_per_cu(mode, sums) * device_cus();
    in.max_items = (int)std::min((long long)p.tblocks * p.splits, (long long)(1 << 30));
    in.rows = near_rows(mode);
    in.max_partials = (long long)(partial_bytes / sizeof(double)) / (mode == PYPO_MODE_SCALAR ? 1 : 12 / in.rows);
    in.kabs = (float)kabs;
    const NodeRule &rule = f64 ? kNodesFp64 : kNodesMixed;
    in.q = (float)rule.q;
    in.p = (float)rule.p;
    in.log_eps = (float)rule.log_eps;
    for (int n = 1; n < kNearSmall; n++) {
        // 2 (K / 2)^n / n! = eps
        in.small[n] = 2.f * std::exp((std::lgamma(n + 1.f) + 0.693f - in.log_eps) / n);
    }
    in.small[0] = 0.f;
    in.dyadic = mode == PYPO_MODE_SCALAR ? 0.f : (float)(1.5 / kabs);
    in.pair_cycles = (float)pair_cycles(mode, sums);
    in.direct_cycles = direct_cycles > 0.0 ? (float)direct_cycles : in.pair_cycles;
    // a coefficient's share of a target's series, and with its gradient; the passes around them
    // (twice that and more where the targets' waves do not fill the chip)
    in.series_cycles = (w.nodes_only ? 18.f : 7.f) * std::max(1.f, 2048.f * 64 / w.n_tgt);
    in.fixed_cycles = (float)((w.nodes_only ? 90e-6 : 40e-6) * kSimdHz);
    in.sort_cycles = w.slot ? (float)((15e-6 + 25e-12 * w.n_tgt) * kSimdHz) : 0.f;
    hipLaunchKernelGGL(k_near_frame, dim3(1), dim3(256), 0, st, in, w);
    PYPO_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_near_cones, dim3(w.tgt_blocks()), dim3(256), 0, st, w);
    PYPO_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_near_plan, dim3(1), dim3(1024), 0, st, in, w);
    PYPO_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_near_nodes, dim3(64), dim3(256), 0, st, w);
    PYPO_CHECK_LAUNCH();
    if (w.slot) {
        hipLaunchKernelGGL(k_near_bin, dim3(w.bins()), dim3(1024), 0, st, w);
        PYPO_CHECK_LAUNCH();
        hipLaunchKernelGGL(k_near_scan, dim3(1), dim3(1024), 0, st, w);
        PYPO_CHECK_LAUNCH();
        hipLaunchKernelGGL(k_near_order, dim3((w.n_tgt + 255) / 256), dim3(256), 0, st, w);
        PYPO_CHECK_LAUNCH();
    }
    return 0;
}

int launch_near_cheb_coef(int mode, const double *partial, const NearWs &w, double rev_scale, hipStream_t st) {
    const int rows = near_rows(mode), stride = mode == PYPO_MODE_SCALAR ? 2 : 12;
    hipLaunchKernelGGL(k_near_reduce, dim3(512), dim3(256), 0, st, partial, w, rev_scale, stride, stride - rows, rows);
    PYPO_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_near_coef, dim3(1024), dim3(256), 0, st, w, rows);
    PYPO_CHECK_LAUNCH();
    return 0;
}

}  // namespace pypo
