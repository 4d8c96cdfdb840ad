// po_near_cheb.hpp -- near fields through Chebyshev patches around a compact
// source.
//
// Seen from the centre c of its sources, the field at p = c + R u (u a unit
// vector) is exp(j t k R) / R times a function of u and 1 / R that is as smooth
// as the extent of the sources allows: its phase moves by k |r_s - c| per
// radian of u and by k |r_s - c|^2 / 2 per unit of 1 / R.  With a frame whose
// third axis points at the targets, coordinates
//   (a, b) = theta (cos phi, sin phi) of u,   s = 1 / R - fit(a, b)
// the box of the targets in (a, b) is cut into pa x pb patches, the fields are
// summed at na x nb x nr Chebyshev nodes of every patch -- by the kernels that
// sum them at targets -- and every target evaluates its patch's series.  fit
// is the least-squares quadratic through a sample of the targets: they mostly
// lie on a smooth surface, and s then spans little (nr = 2 where 1 / R itself
// asks for 6 nodes).
// Node counts follow the phase rates over the Bernstein ellipses of the boxes,
// as for far fields (po_cheb.hpp), with
//   * 1 / (1 - rho / R_min) on the rates (rho: largest |r_s - c|) and 2 rad per
//     rad for the dyadic's R_hat R_hat;
//   * 1.5 / k per unit of s for the dyadic's 1 / (k R) and 1 / (k R)^2, which
//     stay where the sources shrink to a point: exp(1.5 x) dominates 1 + x + x^2
//     term by term.  Never more than two nodes beyond those of the rest, as
//     they are of degree two (worst error over sources of 2e-6 to 1 wavelength,
//     targets from 0.03 to 100, flat, dish-shaped or filling a volume: 1.6e-9 of
//     peak, FP64 4e-13; without it 5e-2 and 6e-6);
//   * an ellipse no larger than the singularity allows (a source point in
//     complex direction: cosh eta = R / rho; along s: s = 1 / rho);
//   * for small K the tighter 2 (K / 2)^n / n! <= eps.
//
// The node sums take no shadow test: the plan is on only where every source
// lights every target, and nodes of the box that no target is near may lie
// beyond a source's horizon, where the field has to continue smoothly.
//
// The plan is made on the device, like the far field's, and is off where
//   * R_min < 3 rho, the targets spread more than 1.5 rad around the axis, or
//     some pair may be in shadow;
//   * an extent is not finite or a current infinite (one that is not a number
//     spoils every node, and so every target it would);
//   * nodes and series would cost more than the sums at the targets.
//
// Targets of 200 000 points and more are evaluated in the order of their
// patches (a counting sort): in grid order a wave of a polar grid meets three.
//
// Measured on MI355X (node sums / series / whole call, before): JM 1089 ->
// 1 002 001 mixed 122 / 187 / 472 us (2 410), error against 64 bits 1.3e-7
// (4.8e-7); EHP 10 201 -> 640 800 491 / 322 / 950 us (20 150), 2.3e-8
// (3.2e-8); scalar 10 201 -> 160 801 133 / 93 / 304 us (1 253), 2.0e-7
// (2.2e-7).
#pragma once

#include "common.hpp"

namespace pypo {

constexpr int kNearMaxNodes = 65536;   // all patches together
constexpr int kNearMaxAxis = 96;       // na, nb
constexpr int kNearMaxRadial = 24;     // nr
constexpr int kNearMaxPatches = 16;    // per axis
constexpr int kNearBox = 1024;         // targets per workgroup of the box pass
constexpr int kNearBin = 4096;         // targets per workgroup that counts them by patch

struct NearPlan {
    int on;
    int pa, pb, na, nb, nr, n;         // n = pa pb na nb nr; node i = (((ipa pb + ipb) na + ia) nr + ir) nb + ib
    int tblocks, splits, chunk;        // launch plan of the sums at the nodes
    double a0, b0, da, db;             // box corner and patch widths
    double s_mid, s_half;
    double c[3], e[3][3];              // centre; frame, e[2] towards the targets
    double ext[4];                     // half extents of the sources along e, and rho
    double fit[6], fa, fb, ga, gb;     // fit[0..5] of 1, x, y, x^2, x y, y^2 at x = (a - fa) ga, y = (b - fb) gb
    int sorted;                        // targets go in the order of `perm`
    __host__ __device__ double surface(double a, double b) const {
        const double x = (a - fa) * ga, y = (b - fb) * gb;
        return fit[0] + x * (fit[1] + x * fit[3] + y * fit[4]) + y * (fit[2] + y * fit[5]);
    }
};

// Workspace of one propagation, behind the split partials, and its grids.
struct NearWs {
    NearPlan *plan = nullptr;          // nullptr: not tried
    float *box = nullptr;              // [source tile, then target block][6]: min x, y, z, max x, y, z (not finite: off)
    float *cone = nullptr;             // [target block][8]: min a, b, 1/R, s, max a, b, 1/R, s
    float *theta = nullptr;            // [target block][4]: largest theta, summed extents a, b of waves, waves
    double *x = nullptr, *y = nullptr, *z = nullptr;   // nodes
    double *f = nullptr;               // [rows][n] sums at the nodes
    double *coef = nullptr;            // [patch][na][nr][nb][rows] Chebyshev coefficients
    unsigned *slot = nullptr;          // [target]: patch << 16 | rank in its bin; nullptr: no sorting
    int *count = nullptr;              // [patch][bin]: counts, then first positions
    int *perm = nullptr;               // [n_tgt] targets patch by patch
    const double *tx = nullptr, *ty = nullptr, *tz = nullptr;   // targets
    int n_src = 0, n_tgt = 0;
    bool nodes_only = false;           // the sum kernel works on nodes or not at all
    __host__ __device__ int src_tiles() const { return (n_src + 255) / 256; }
    __host__ __device__ int tgt_blocks() const { return (n_tgt + kNearBox - 1) / kNearBox; }
    __host__ __device__ int bins() const { return (n_tgt + kNearBin - 1) / kNearBin; }
};

bool near_cheb_try(int mode, int precision, int n_src, int n_tgt);
size_t near_cheb_bytes(int mode, int n_src, int n_tgt);
NearWs near_cheb_carve(void *base, int mode, int n_src, const GridPtrs &ct, int n_tgt);

}  // namespace pypo
