// po_cheb.hpp -- far fields through a Chebyshev grid of directions.
//
// The source sums S_q(r) = sum_s C_q(s) exp(-j t k r_s.r) of the far field are
// band-limited functions of the direction: over a box of directions they
// carry no more detail than the extent of the sources in wavelengths allows,
// however finely the caller samples them.  With the coordinates
//   a = theta cos(phi),  b = theta sin(phi)      (AoE grids: azimuth, elevation)
// r(a, b) is an entire function, and so is, for the centre c of the sources,
//   f(a, b) = exp(j t k c.r) S_q(r(a, b)).
// Its interpolant at na x nb Chebyshev nodes of the box converges faster than
// any power once na, nb pass the largest phase rate of a source over the box,
//   K_a = k h_a max |(r_s - c).dr/da|      (h_a: half-width of the box)
// so the sums are taken at the nodes only, by the same kernels as the sums at
// the targets, and every target evaluates the Chebyshev series.
//
// Node count.  The interpolant of exp(j K x) at n Chebyshev nodes of [-1, 1]
// is off by at most 4 sum_{i >= n} |J_i(K)|; n = ceil(K + q K^(1/3) + p) keeps
// that below 1.6e-9 for kNodesMixed (mixed precision, whose FP32 sums are good
// to 1e-7) and below 1.5e-15 for kNodesFp64, for all K up to 160.
// The phase is not linear in a and b; what matters is its growth over the
// Bernstein ellipse of that convergence, imaginary extent eta = sqrt(n^2 -
// K^2) / (K / h), where |dr_x/da| <= cosh eta, |dr_y/da| <= |a b| / 3 cosh eta
// and |dr_z/da| <= (|a| + eta) cosh eta.  The plan iterates K with those
// bounds.  Over 250 random boxes (to 1.5 rad off axis) and source extents (to
// 1e4 rad), the worst error was 5.9e-11 mixed, 5.7e-12 FP64 (which phases of 1e4
// rad round to).
//
// When it is taken.  The decision needs the extents of the sources and of the
// directions, which live on the device, so it is made there: the pack
// pass reduces them beside its tile metadata (k_tile_meta), k_cheb_plan decides
// and writes a ChebPlan, and the kernels behind it read the plan.  No host synchronisation; a captured graph
// decides anew on every replay.  The plan is off, and the sums are taken at the
// targets as they come, when
//   * some tile of sources could be shadowed in part of the box (n.r of either
//     sign): the shadow test makes the sums discontinuous in r;
//   * an extent is not finite, a current infinite (one that is not a number
//     spoils every node, and so every target it would), or the box reaches beyond
//     1.5 rad;
//   * the nodes would cost more than the targets they stand for (the rule is at
//     cheb_pays).
//
// Far-field grids usually come as rows of equal a (an AoE grid's azimuth):
// the plan looks for the row length, the split reduction checks every target
// against it, and the series is then summed along b once per column.
//
// Measured on MI355X: 1 002 001 sources -> 251 001 targets over +-10.5 beam
// widths, 59 x 59 nodes, 91.6 -> 1.69 ms mixed (error against 64 bits 9.5e-8 ->
// 7.2e-8), of which the node sums 1.5 ms; 90 300 -> 40 401 in FP64 5.14 ->
// 0.72 ms; 89 999 -> 31 313 with J and M over +-15 beam widths 1.27 -> 0.385 ms.
// Where the plan stays off it costs some 15 us.
// The row form: the two-dimensional series took 540, 260 and 270 us of these,
// the rows 37, 31 and 44 us.
#pragma once

#include "common.hpp"

namespace pypo {

// Node counts of the far and the near grids: q and p of the rule, and ln(4 / eps).
struct NodeRule { double q, p, log_eps; };
constexpr NodeRule kNodesMixed{6.9, 3.05, 21.1}, kNodesFp64{8.9, 10.05, 34.8};

constexpr int kChebMaxNodes = 32768;    // na nb, also the workspace's size
constexpr int kChebMaxAxis = 224;       // na, nb
constexpr int kChebMaxRow = 2048;       // targets per row, and na times that, of the row form
constexpr int kChebMaxRows = 65536;
// The adjoint's moments of the targets (adjoint_cheb.hip): tiles of kMomA x kMomB
// moments, kMomTiles of them at a time.
constexpr int kMomA = 64, kMomB = 16, kMomTiles = 16;
constexpr int kChebBoxTargets = 1024;   // targets per workgroup that reduces their box

struct ChebPlan {
    int on;                // 0: the kernels work on the targets themselves
    int has_m;             // some source carries magnetic current
    int na, nb, n;         // nodes per axis, n = na nb; node i = ia nb + ib
    int tblocks, splits, chunk;   // launch plan of the sums at the nodes
    double a_mid, a_half, b_mid, b_half;
    double c[3];           // centre of the sources
    int row;               // targets per row of equal a, 0: no such rows
    double row_tol;        // and the rounding within which a and b may differ
};

// Workspace of one propagation, behind the split partials, and the targets.
struct ChebWs {
    ChebPlan *plan = nullptr;      // nullptr: not tried
    float *src_box = nullptr;      // [tile][6]: min x, y, z, max x, y, z
    float *tgt_box = nullptr;      // [block][4]: min a, b, max a, b (NaN: not finite)
    int *not_rows = nullptr;       // set where the targets do not form the plan's rows
    double *th = nullptr, *ph = nullptr;   // node directions
    double *f = nullptr;           // [12][n] sums at the nodes
    double *coef = nullptr;        // [na][nb][12] Chebyshev coefficients
    double *rows = nullptr;        // [na][12][row] the series along b at every column
    const double *tgt_th = nullptr, *tgt_ph = nullptr;   // the caller's targets
    int n_tgt = 0;
    __host__ __device__ int boxes() const { return (n_tgt + kChebBoxTargets - 1) / kChebBoxTargets; }
};

// Whether a propagation tries the Chebyshev grid at all (host rule on sizes),
// the bytes of its workspace, and the workspace at `base`.
bool cheb_try(int mode, int precision, int n_src, int n_tgt);
size_t cheb_bytes(int n_src, int n_tgt);
ChebWs cheb_carve(void *base, int n_src, const GridPtrs &ct, int n_tgt);

}  // namespace pypo
