// Error bounds of the 32-bit distance filter: what a value has to differ from
// zero by for its sign to be the 64-bit test's.  Values closer than that are
// decided by the 64-bit test.
#pragma once
#include <algorithm>
#include <cmath>

#include "../../include/nlhip.h"
#include "nlhip_internal.h"

namespace nlh {

constexpr float kFar32 = 1.0e18f;   // sentinel position: |p|^2 / 2 = 5e35, never a hit

// The distance that cutoff_sq, which decides, stands for (a caller fills both).
inline double search_radius(const nlh_geometry &g)
{
    return std::max(g.cutoff, std::sqrt(g.cutoff_sq));
}

// Bounds of the 32-bit distance filter (SysDev; tile_kernel in pairs.hip).
// With u = 2^-24, c the centre of a run of home cells, |p_i - c| <= H for
// its home atoms and |p_j - c| <= H + rc for any candidate within the cutoff,
// the computed 2 D = r^2 - rc^2 is off by at most
//   10 u ((2 H + rc)^2 + rc^2)   five fused multiply-adds over partial sums
//                                of at most (|p_i| + |p_j|)^2 + rc^2, doubled
//   7 u (H + rc)^2 + 4 u rc^2    |p_j - c|^2, |p_i - c|^2 - rc^2, rc^2 itself
//   7.2 u (P + 2 H + rc) rc      positions rounded to 32 bits, |p| <= P, then
//                                taken from c
//   1.6e-11 rc (|a1| + |a2| + |a3|)   the 64-bit roundings on both sides, for
//                                windings within +-511 (six times their bound)
// and by less than its distance from zero for candidates further away.  A
// quarter is added for what the line above leaves out (second-order terms).
inline void filter_bounds(SysDev &sd, const nlh_geometry &g)
{
    constexpr double u = 1.0 / (1 << 24);
    const double rc = search_radius(g);
    double step[3][3], len[3], sum = 0.0, P = rc;
    for (int k = 0; k < 3; ++k) {
        double l2 = 0.0;
        for (int m = 0; m < 3; ++m) {
            step[k][m] = g.cell[k + 3 * m] / (double)sd.n[k];   // a cell's edge along lattice vector k
            l2 += step[k][m] * step[k][m];
        }
        len[k] = std::sqrt(l2);
        sum += len[k] * sd.n[k];
        P += (sd.brick[k] / 2 + 2.5) * len[k];   // halo atom to an atom of the middle home cell
    }
    for (int m = 0; m < 3; ++m) step[0][m] *= sd.run;
    double diag2 = 0.0;   // the longest diagonal of a run of home cells
    for (int q = 0; q < 4; ++q) {
        double d2 = 0.0;
        for (int m = 0; m < 3; ++m) {
            const double d = step[0][m] + (q & 1 ? -1 : 1) * step[1][m] + (q & 2 ? -1 : 1) * step[2][m];
            d2 += d * d;
        }
        diag2 = std::max(diag2, d2);
    }
    const double H = 0.505 * std::sqrt(diag2) + 0.25 * rc;
    const double tol = 1.25 * u * (10 * ((2 * H + rc) * (2 * H + rc) + rc * rc) + 7 * (H + rc) * (H + rc) +
                                   4 * rc * rc + 7.2 * (P + 2 * H + rc) * rc) + 1.6e-11 * rc * sum;
    const bool ok = H < 1000 * rc && P < 1e6 * rc && rc > 1e-14 && rc < 1e9;
    sd.rc2half = (float)(0.5 * g.cutoff_sq);
    sd.tol = (float)(0.505 * tol);
    sd.tol64 = (float)(1.6e-11 * rc * sum);
    sd.h2half = (float)(0.499 * H * H);
    sd.pmax2 = ok ? (float)(0.999 * P * P) : -1.0f;
}

// The same for a system of a fused build (small_kernel), whose positions are
// kept in 32 bits from the system's centre, wrapped: with o the home cell's
// centre, A the longest cell shift of a candidate, O = (|a1| + |a2| + |a3|) / 2 and
// H as found for each group of home atoms, the positions' share is
//   u rc (8 H + 4 rc + 10 (A + O))
// (home atom u (|o| + 2 H); candidate u (2 (H + rc) + |s - o|) and, for s - o
// itself, u (4 A + 3 |o|)); with 2 H rc <= H^2 + rc^2 the sum of all terms is at
// most u (78 H^2 + 66 rc^2 + 10 (A + O) rc), of which the kernel adds the first;
// the 64-bit roundings' share is filter_bounds'.
inline void small_bounds(SysDev &sd, const nlh_geometry &g)
{
    constexpr double u = 1.0 / (1 << 24);
    const double rc = search_radius(g);
    double sum = 0.0, A = 0.0;
    for (int k = 0; k < 3; ++k) {
        double l2 = 0.0;
        for (int m = 0; m < 3; ++m) l2 += g.cell[k + 3 * m] * g.cell[k + 3 * m];
        const double len = std::sqrt(l2);
        sum += len;
        if (sd.pbc >> k & 1) A += len * ((sd.nxyz[k] + sd.n[k] - 1) / sd.n[k]);
    }
    sd.small_tol = (float)(0.505 * (1.25 * u * (66 * rc * rc + 10 * (A + 0.5 * sum) * rc) + 1.6e-11 * rc * sum));
    for (int k = 0; k < 9; ++k) sd.C32[k] = (float)sd.C[k];
}

// The filter's error bound (filter_bounds) for home atoms within H of their
// centre and brick atoms up to |p|^2 = far2 beyond the system's pmax2.
// Beyond any sane scale every value is decided by the 64-bit test.  (1,000 atoms
// centred on the corner of an open cell, count kernel: bricks with such atoms
// on the 64-bit per-wave path 684 us, with a bound of their own 68; 64-bit LDS
// path 235.)
__host__ __device__ inline float far_tol(const SysDev &sd, float H, float far2)
{
    const float P = __builtin_sqrtf(fmaxf(sd.pmax2, far2)), rc = __builtin_sqrtf(2.0f * sd.rc2half);
    const float a = 2.0f * H + rc, b = H + rc;
    const float e = 10.0f * (a * a + rc * rc) + 7.0f * b * b + 4.0f * rc * rc + 7.2f * (P + a) * rc;
    return H + P < 1.0e15f ? 0.505f * (1.25f / (1 << 24) * e + sd.tol64) : kFar32 * kFar32;
}

// The share of the home group's extent in the filter's error bound: times the
// largest |p_i|^2 / 2 of the group (see small_bounds for the rest).
constexpr float kSmallTol = 0.505f * 1.25f / (1 << 24) * 156.0f;
// ... and that of a centre beyond the system's cell: times its distance and the cutoff.
constexpr float kSmallTolFar = 0.505f * 1.25f / (1 << 24) * 10.0f;

}  // namespace nlh
