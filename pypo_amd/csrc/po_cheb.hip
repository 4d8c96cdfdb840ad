// po_cheb.hip -- the Chebyshev grid of far-field directions: extents, plan,
// and the transform of the node sums into series coefficients.  po_cheb.hpp
// says what it is for; the sums themselves are the kernels of po_ff.hip and
// po_ff_mfma.hip, the series is evaluated by k_ff_finish.

#include "po_cheb_dev.hpp"

#include <algorithm>

namespace pypo {
namespace {

// Nodes along one axis of half-width h: the fixed point of the node count and
// the phase rate over its Bernstein ellipse (po_cheb.hpp).  x, y, z: half
// extents of the sources along the axis, along the other one and along z;
// lim, lim_o: largest |a| of the box along the axis and the other one; extra:
// rate of a factor beside the phase.
__device__ int cheb_nodes(float kabs, float h, float x, float y, float z, float lim, float lim_o, float q, float p,
                          float extra) {
    float eta = 0.f, n = 1.f;
    for (int it = 0; it < 4; it++) {
        const float e = __expf(eta), ch = 0.5f * (e + 1.f / e);
        const float rate =
            ch * (kabs * (x + y * fminf(1.f, (lim + eta) * lim_o * (1.f / 3.f)) + z * (lim + eta)) + extra);
        const float K = rate * h * 1.00001f;   // FP32 rounding
        n = ceilf(K + q * cbrtf(K) + p);
        eta = fminf(1.5f, sqrtf(fmaxf(0.f, n * n - K * K)) / fmaxf(rate, 1e-30f));
    }
    return (n > 0.f && n < 1e6f) ? (int)n : (1 << 20);
}

// Whether sums at n nodes and a series at every target cost less than sums at
// the targets, with room for the passes between (in units of a source-target
// pair of the sum).  eval: the series at one target in such units -- 13 (7
// without magnetic currents) FP64 FMAs of 4.8 issue cycles per 64 targets and
// term, against 59 cycles per 64 pairs of the matrix kernel, 80 of the vector
// kernel, 225 of the FP64 kernel (far_cycles; all measured on gfx950), or the
// adjoint's moments; fixed: the passes between.
__device__ bool cheb_pays(long long n, double eval, double n_src, double n_tgt, double lanes, double fixed) {
    const double nodes = ceil((double)n / lanes) * lanes, tgts = ceil(n_tgt / lanes) * lanes;
    return nodes * n_src + eval * n_tgt + fixed < 0.8 * tgts * n_src;
}

struct PlanIn {
    const TileMeta *meta;
    int n_tiles;
    int n_src, n_tgt, tpl, slots, max_items;   // max_items: workgroups launched for the sum
    long long max_partials;                    // doubles of the split partials
    double kabs, q, p, cycles, fixed, extra, moments;
};

// One workgroup: reduce the extents, decide, write the plan and (w.th not null)
// the nodes.
__global__ __launch_bounds__(1024) void k_cheb_plan(PlanIn in, ChebWs w) {
    __shared__ float red[16][10];
    __shared__ float ext[10];
    __shared__ int flags[2];       // some tile may be shadowed; some tile has M
    __shared__ ChebPlan pl;
    __shared__ unsigned long long best;
    __shared__ int row;            // first target whose a is not the first target's
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    // minima of (x, y, z, -x, -y, -z) and (a, b, -a, -b); NaN turns into "off"
    float v[10];
    bool bad = false;
#pragma unroll
    for (int q = 0; q < 10; q++) v[q] = INFINITY;
    for (int i = tid; i < in.n_tiles; i += 1024)
#pragma unroll
        for (int q = 0; q < 6; q++) {
            const float x = q < 3 ? w.src_box[6 * i + q] : -w.src_box[6 * i + q];
            bad |= !(fabsf(x) < 1e30f);
            v[q] = fminf(v[q], x);
        }
    for (int i = tid; i < w.boxes(); i += 1024)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float x = q < 2 ? w.tgt_box[4 * i + q] : -w.tgt_box[4 * i + q];
            bad |= !(fabsf(x) < 1e30f);
            v[6 + q] = fminf(v[6 + q], x);
        }
    if (tid < 2) flags[tid] = 0;
    if (tid == 0) { best = ~0ull; row = 1 << 30; }
#pragma unroll
    for (int q = 0; q < 10; q++) v[q] = wave_min(v[q]);
    if (lane == 0)
#pragma unroll
        for (int q = 0; q < 10; q++) red[wv][q] = v[q];
    bad = __syncthreads_or(bad);
    if (tid < 10) {
        float m = red[0][tid];
#pragma unroll
        for (int i = 1; i < 16; i++) m = fminf(m, red[i][tid]);
        ext[tid] = m;
    }
    __syncthreads();
    Cone cone;
    cone.ax = 0.f; cone.ay = 0.f; cone.az = 1.f; cone.cos_half = -1.f;
    {
        const double am = 0.5 * ((double)ext[6] - ext[8]), bm = 0.5 * ((double)ext[7] - ext[9]);
        // half-widths, widened by the FP32 rounding of the boxes
        const double ah = 0.5 * (-(double)ext[8] - ext[6]) + 2e-7 * fmax(fabs((double)ext[8]), fabs((double)ext[6]));
        const double bh = 0.5 * (-(double)ext[9] - ext[7]) + 2e-7 * fmax(fabs((double)ext[9]), fabs((double)ext[7]));
        const double t = hypot(am, bm), s = t > 0 ? sin(t) / t : 1.0, half = hypot(ah, bh);
        cone.ax = (float)(am * s); cone.ay = (float)(bm * s); cone.az = (float)cos(t);
        if (half < 1.5) cone.cos_half = (float)cos(half);   // r(a, b) moves no faster than (a, b)
        double c[3];
        float e[3];
        for (int q = 0; q < 3; q++) {
            const double lo = ext[q], hi = -(double)ext[3 + q];
            c[q] = 0.5 * (lo + hi);
            e[q] = (float)(0.5 * (hi - lo) + 2e-7 * fmax(fabs(lo), fabs(hi)));
        }
        const float la = (float)(fabs(am) + ah), lb = (float)(fabs(bm) + bh);
        if (wv == 0) {   // lane 0: along a, the others: along b
            const bool al = lane == 0;
            const int nl = cheb_nodes((float)in.kabs, (float)fmax(al ? ah : bh, 1e-12), al ? e[0] : e[1],
                                      al ? e[1] : e[0], e[2], al ? la : lb, al ? lb : la, (float)in.q, (float)in.p,
                                      (float)in.extra);
            const int na = __shfl(nl, 0, 64), nb = __shfl(nl, 1, 64);
            if (lane == 0) {
                pl.a_mid = am; pl.b_mid = bm;
                pl.a_half = fmax(ah, 1e-12); pl.b_half = fmax(bh, 1e-12);
                for (int q = 0; q < 3; q++) pl.c[q] = c[q];
                pl.na = na; pl.nb = nb;
                pl.on = !bad && la <= 1.5f && lb <= 1.5f && na <= kChebMaxAxis && nb <= kChebMaxAxis &&
                        na * nb <= kChebMaxNodes && na * nb <= in.n_tgt;
                pl.n = pl.on ? na * nb : 0;
            }
        }
    }
    {
        bool shadow = false, m = false;
        for (int i = tid; i < in.n_tiles; i += 1024) {
            const TileMeta t = in.meta[i];
            // infinite currents keep the sums' own infinities and NaN, target by target
            shadow |= !(t.cmax < INFINITY) || cones_may_shadow(t.ax, t.ay, t.az, t.cos_half, cone);
            m |= t.has_m != 0;
        }
        if (shadow) flags[0] = 1;
        if (m) flags[1] = 1;
    }
    __syncthreads();
    // Rows of equal a among the first targets; theta and phi of a generated
    // grid bring a and b back to a few ulp.  One LDS atomic per wave: a
    // thousand on one word would take microseconds.
    const double tol = 2e-15 * (fabs(pl.a_mid) + pl.a_half + fabs(pl.b_mid) + pl.b_half);
    if (pl.on && !flags[0] && in.moments == 0.0) {
        double a0, x;
        target_ab(w.tgt_th, w.tgt_ph, 0, a0, x);
        int first = 1 << 30;
        for (int t = 1 + tid; t <= min(kChebMaxRow, in.n_tgt - 1); t += 1024) {
            double a;
            target_ab(w.tgt_th, w.tgt_ph, t, a, x);
            if (fabs(a - a0) > tol) first = min(first, t);
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) first = min(first, __shfl_xor(first, o, 64));
        if (lane == 0) atomicMin(&row, first);
    }
    __syncthreads();
    // ... and 256 targets scattered over all of them (one wave a SIMD: sixteen waves'
    // sines took 6 us): the rule below counts on rows, and first targets in a row
    // say little of the others (a scan back and forth).
    bool rows = row >= 16 && row <= kChebMaxRow && in.n_tgt % row == 0 && pl.na * row <= min(kChebMaxRows, in.n_tgt);
    if (rows && tid < 256) {
        const double g = tid * 0.6180339887498949;
        rows = cheb_in_row(w, min(in.n_tgt - 1, (int)((g - floor(g)) * in.n_tgt)), row, tol);
    }
    rows = __syncthreads_and(rows);
    if (tid == 0) {
        pl.has_m = flags[1];
        pl.row_tol = tol;
        pl.row = rows ? row : 0;
        const double terms = pl.row ? pl.na : pl.n;
        const int tiles = ((pl.na + kMomA - 1) / kMomA) * ((pl.nb + kMomB - 1) / kMomB);
        const double eval = in.moments > 0.0 ? (tiles + kMomTiles - 1) / kMomTiles * in.moments * 64.0
                                             : terms * (flags[1] ? 13.0 : 7.0) * 4.8;
        pl.on = pl.on && !flags[0] &&
                cheb_pays(pl.n, eval / in.cycles, in.n_src, in.n_tgt, 256.0 * in.tpl, in.fixed);
        pl.tblocks = (pl.n + 256 * in.tpl - 1) / (256 * in.tpl);
    }
    __syncthreads();
    if (!pl.on) {
        if (tid == 0) *w.plan = pl;
        return;
    }
    // Source splits of the node sums: `ct` tiles per split, the count with the
    // fewest tile times over the rounds of concurrent workgroups, 0.3 tile
    // times of set-up per workgroup, within the partials and the workgroups
    // the launch has (one split of the targets' own plan always fits).
    unsigned long long mine = ~0ull;
    for (int ct = tid + 1; ct <= in.n_tiles; ct += 1024) {
        const unsigned used = (in.n_tiles + ct - 1) / ct, items = used * pl.tblocks;   // < 2^23 tiles x 128
        if (items > (unsigned)in.max_items || used * 12ll * pl.n > in.max_partials) continue;
        const unsigned long long rounds = (items + in.slots - 1) / in.slots;
        mine = min(mine, rounds * (10ull * ct + 3) << 32 | (unsigned)ct);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) mine = min(mine, __shfl_xor(mine, o, 64));
    if (lane == 0) atomicMin(&best, mine);
    __syncthreads();
    const int ct = best == ~0ull ? in.n_tiles : (int)(best & 0xffffffffu);
    if (tid == 0) {
        pl.chunk = ct * TILE;
        pl.splits = (in.n_tiles + ct - 1) / ct;
        *w.not_rows = 0;
        *w.plan = pl;
    }
    if (w.th)
        for (int i = tid; i < pl.n; i += 1024) cheb_node(pl, i, w.th, w.ph);
}

template <bool TURNED>
__global__ __launch_bounds__(256) void k_cheb_reduce(const double *__restrict__ partial, ChebWs w, double rev_scale) {
    if (!w.plan->on) return;
    cheb_reduce<TURNED>(w, partial, rev_scale, blockIdx.x, gridDim.x);
    cheb_check_rows(w, blockIdx.x, gridDim.x);
}

__global__ __launch_bounds__(256) void k_cheb_coef(ChebWs w) {
    if (w.plan->on) cheb_coef(w, blockIdx.x, gridDim.x);
}

static_assert(sizeof(ChebPlan) <= 192, "the plan and not_rows share 256 bytes");

size_t up256(size_t b) { return (b + 255) / 256 * 256; }

int node_cap(int n_tgt) { return std::min(kChebMaxNodes, n_tgt); }

}  // namespace

// Below about 6e8 pairs (2e8 in FP64) the sum itself takes under 250 us and
// the plan's passes would be felt where it then stays off.
bool cheb_try(int mode, int precision, int n_src, int n_tgt) {
    const double pairs = (double)n_src * n_tgt;
    return mode == PYPO_MODE_FF && n_tgt >= 1024 && n_src >= 1024 &&
           pairs >= (precision == PYPO_PREC_FP64 ? 2e8 : 6e8);
}

double far_cycles(int precision) {
    return precision == PYPO_PREC_FP64 ? 225.0 : (ff_kernel() == PYPO_FF_MATRIX ? 59.0 : 80.0);
}

size_t cheb_bytes(int n_src, int n_tgt) {
    const size_t cap = node_cap(n_tgt);
    const int boxes = (n_tgt + kChebBoxTargets - 1) / kChebBoxTargets;
    return 256 + up256((size_t)n_tiles(n_src) * 6 * sizeof(float)) + up256((size_t)boxes * 4 * sizeof(float)) +
           up256((26 * cap + 12 * (size_t)std::min(kChebMaxRows, n_tgt)) * sizeof(double));
}

ChebWs cheb_carve(void *base, int n_src, const GridPtrs &ct, int n_tgt) {
    const size_t cap = node_cap(n_tgt);
    char *b = (char *)base;
    ChebWs w;
    w.tgt_th = ct.x;
    w.tgt_ph = ct.y;
    w.n_tgt = n_tgt;
    w.plan = (ChebPlan *)b;
    w.not_rows = (int *)(b + 192);
    b += 256;
    w.src_box = (float *)b;
    b += up256((size_t)n_tiles(n_src) * 6 * sizeof(float));
    w.tgt_box = (float *)b;
    b += up256((size_t)w.boxes() * 4 * sizeof(float));
    w.th = (double *)b;
    w.ph = w.th + cap;
    w.f = w.ph + cap;
    w.coef = w.f + 12 * cap;
    w.rows = w.coef + 12 * cap;
    return w;
}

int launch_cheb_plan(int precision, const SumPlan &p, const TileMeta *meta, int n_src, double rev_scale,
                     size_t partial_bytes, const ChebCost &cost, const ChebWs &w, hipStream_t st) {
    const bool f64 = precision == PYPO_PREC_FP64;
    PlanIn in;
    in.meta = meta;
    in.n_tiles = n_tiles(n_src);
    in.n_src = n_src; in.n_tgt = w.n_tgt; in.tpl = p.tpl;
    in.slots = ff_wgs_per_cu(precision, p.tpl) * device_cus();
    in.max_items = (int)std::min((long long)p.tblocks * p.splits, (1LL << 30));
    in.max_partials = (long long)(partial_bytes / sizeof(double));
    in.kabs = std::fabs(rev_scale) * kTwoPi;
    const NodeRule &rule = f64 ? kNodesFp64 : kNodesMixed;
    in.q = rule.q;
    in.p = rule.p;
    in.cycles = cost.cycles;
    in.fixed = cost.fixed_us * 64.0 * kSimdHz * 1e-6 / cost.cycles;
    in.extra = cost.extra;
    in.moments = cost.moments;
    hipLaunchKernelGGL(k_cheb_plan, dim3(1), dim3(1024), 0, st, in, w);
    PYPO_CHECK_LAUNCH();
    return 0;
}

int launch_cheb_coef(int precision, const double *partial, const ChebWs &w, double rev_scale, hipStream_t st) {
    hipLaunchKernelGGL(precision == PYPO_PREC_FP64 ? k_cheb_reduce<true> : k_cheb_reduce<false>, dim3(512), dim3(256), 0,
                       st, partial, w, rev_scale);
    PYPO_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_cheb_coef, dim3(1024), dim3(256), 0, st, w);
    PYPO_CHECK_LAUNCH();
    return 0;
}

}  // namespace pypo
