// The 32-bit distance filter of the pair search, emulated operation by
// operation beside the 64-bit test, for pairs near the cutoff and others:
// prints the pairs whose sign it would take although the 64-bit test differs,
// the largest error of a value near zero over its bound, and the share of pairs that
// the bound sends to the 64-bit test.  Built and run by tests/test_host_rules.py.
#include <cstdio>
#include <random>

#include "filter_bounds.h"

using namespace nlh;

namespace {

std::mt19937_64 rng(12345);
double uni() { return (double)(rng() >> 11) * 0x1p-53; }
double sym() { return 2.0 * uni() - 1.0; }
int pick(int lo, int hi) { return lo + (int)(rng() % (uint64_t)(hi - lo + 1)); }

struct Tally {
    long pairs = 0, wrong = 0, exact = 0;
    double worst = 0.0;   // largest error of a value over its bound, among those within four bounds of zero
    void add(float D, float tol, bool hit, long double truth)
    {
        ++pairs;
        if (std::fabs(D) < tol) ++exact;
        else if ((D < 0.0f) != hit) ++wrong;
        if (std::fabs(truth) < 4.0L * tol) worst = std::max(worst, (double)(std::fabs((long double)D - truth) / tol));
    }
};

struct V {
    double c[3];
};

// (C' S)_k in the library's order
V shift(const double *C, const int S[3])
{
    V r;
    for (int k = 0; k < 3; ++k)
        r.c[k] = (C[3 * k] * (double)S[0] + C[3 * k + 1] * (double)S[1]) + C[3 * k + 2] * (double)S[2];
    return r;
}

float dot3(float x, float y, float z, float a, float b, float c, float d)
{
    return std::fmaf(z, c, std::fmaf(y, b, std::fmaf(x, a, d)));
}

// D of a pair from 32-bit positions p_i, p_j relative to the same point and a centre
float filter(const float pi[3], const float pj[3], const float o[3], float rc2half, float &hq)
{
    float n[3], b[3];
    for (int k = 0; k < 3; ++k) {
        n[k] = o[k] - pi[k];
        b[k] = pj[k] - o[k];
    }
    hq = 0.5f * std::fmaf(n[2], n[2], std::fmaf(n[1], n[1], n[0] * n[0]));
    const float bq = 0.5f * std::fmaf(b[2], b[2], std::fmaf(b[1], b[1], b[0] * b[0]));
    return dot3(n[0], n[1], n[2], b[0], b[1], b[2], bq + (hq - rc2half));
}

void geometry(nlh_geometry &g, SysDev &sd, double scale, int brick)
{
    const double rc = scale * (2.0 + 6.0 * uni());
    g = nlh_geometry{};
    sd = SysDev{};
    g.cutoff = rc;
    g.cutoff_sq = rc * rc;
    const double skew = uni() < 0.5 ? 0.0 : 0.4;
    for (int k = 0; k < 3; ++k) {
        sd.n[k] = pick(1, 9);
        const double L = rc * (sd.n[k] + (sd.n[k] == 1 ? uni() : 0.3 * uni()));
        for (int m = 0; m < 3; ++m) g.cell[k + 3 * m] = L * (m == k ? 1.0 : skew * sym());
        sd.brick[k] = std::min(pick(1, brick), sd.n[k]);
        sd.nxyz[k] = 1;
    }
    for (int q = 0; q < 9; ++q) sd.C[q] = g.cell[q];
    sd.pbc = 7;
    sd.run = sd.brick[0] > 1 && uni() < 0.5 ? 2 : 1;
    sd.rc2 = g.cutoff_sq;
    filter_bounds(sd, g);
    small_bounds(sd, g);
}

// A pair a chosen distance apart: atom i at fractional f of the cell and winding
// wi, atom j moved by lattice vectors so that its own winding is wj; S between them.
struct Pair {
    V xi, xj;
    int S[3], wi[3], wj[3];
    double r2;
    bool hit;
    long double truth;   // (r^2 - rc^2) / 2
};

Pair make_pair(const SysDev &sd, double rc, int base, int spread, const double open[3])
{
    Pair p;
    const double kind = uni();
    const double rel = kind < 0.6 ? std::pow(10.0, -2.0 - 14.0 * uni()) * (uni() < 0.5 ? -1 : 1) : kind < 0.8 ? -uni() : uni();
    double d[3], l = 0.0;
    do {
        l = 0.0;
        for (double &x : d) {
            x = sym();
            l += x * x;
        }
    } while (l > 1.0 || l < 1e-3);
    for (int k = 0; k < 3; ++k) {
        p.wi[k] = base + pick(-spread, spread);
        p.wj[k] = base + pick(-spread, spread);
        p.S[k] = p.wi[k] - p.wj[k] + pick(-1, 1);
    }
    const double f[3] = {uni(), uni(), uni()};
    const V vi = shift(sd.C, p.wi), vs = shift(sd.C, p.S);
    for (int k = 0; k < 3; ++k) {
        const double u = (sd.C[3 * k] * f[0] + sd.C[3 * k + 1] * f[1]) + sd.C[3 * k + 2] * f[2];
        p.xi.c[k] = u + vi.c[k] + open[k];
        p.xj.c[k] = p.xi.c[k] + d[k] / std::sqrt(l) * rc * (1.0 + rel) - vs.c[k];
    }
    double R[3];
    long double t = 0.0L;
    for (int k = 0; k < 3; ++k) {
        R[k] = (p.xj.c[k] - p.xi.c[k]) + vs.c[k];
        long double q = (long double)p.xj.c[k] - p.xi.c[k];
        for (int m = 0; m < 3; ++m) q += (long double)sd.C[3 * k + m] * p.S[m];
        t += q * q;
    }
    p.r2 = (R[0] * R[0] + R[1] * R[1]) + R[2] * R[2];
    p.hit = p.r2 < sd.rc2;
    p.truth = (t - (long double)sd.rc2) / 2;
    return p;
}

// tile_kernel: positions from an origin atom of the brick, the run's centre or,
// far from it, the home atom
void tile_case(Tally &T, double scale, int base, int spread, double far)
{
    nlh_geometry g;
    SysDev sd;
    geometry(g, sd, scale, 4);
    if (sd.pmax2 < 0.0f) return;
    const double open[3] = {0.0, 0.0, far * g.cutoff * sym()};
    for (int rep = 0; rep < 40; ++rep) {
        const Pair p = make_pair(sd, g.cutoff, base, spread, open);
        // the origin atom: anywhere within the brick's halo around atom i, with a winding of its own
        int wo[3], to[3], ti[3], tj[3];
        V xo;
        for (int k = 0; k < 3; ++k) wo[k] = base + pick(-spread, spread);
        for (int k = 0; k < 3; ++k) {
            to[k] = -wo[k];
            ti[k] = -p.wi[k] - to[k];           // t' of atom i, in its home cell
            tj[k] = p.S[k] + ti[k];             // S = t'_j - t'_i
        }
        const V so = shift(sd.C, wo), si = shift(sd.C, p.wi);
        for (int k = 0; k < 3; ++k) {
            const double step = std::fabs(sd.C[3 * k]) / sd.n[0] + std::fabs(sd.C[3 * k + 1]) / sd.n[1] + std::fabs(sd.C[3 * k + 2]) / sd.n[2];
            xo.c[k] = (p.xi.c[k] - si.c[k]) + so.c[k] + 1.2 * step * sym();
        }
        const V ci = shift(sd.C, ti), cj = shift(sd.C, tj);
        float fi[3], fj[3], o[3];
        float far2 = 0.0f;
        for (int k = 0; k < 3; ++k) {
            fi[k] = (float)((p.xi.c[k] - xo.c[k]) + ci.c[k]);
            fj[k] = (float)((p.xj.c[k] - xo.c[k]) + cj.c[k]);
            o[k] = fi[k] + (float)(0.4 * g.cutoff * sym()) + (float)(open[k] != 0.0 ? -open[k] : 0.0);
        }
        for (const float *f : {fi, fj}) {
            const float f2 = f[0] * f[0] + f[1] * f[1] + f[2] * f[2];
            if (!(f2 <= sd.pmax2)) far2 = std::max(far2, f2);
        }
        float hq, D = filter(fi, fj, o, sd.rc2half, hq), tol = sd.tol;
        if (!(hq <= sd.h2half) || far2 != 0.0f) {
            if (hq > 32.0f * sd.rc2half) D = filter(fi, fj, fi, sd.rc2half, hq);
            tol = far_tol(sd, std::sqrt(2.0f * hq), far2);
        }
        T.add(D, tol, p.hit, p.truth);
    }
}

// small_kernel: wrapped positions from the system's centre, candidates shifted
void small_case(Tally &T, double scale, int base, int spread, double far)
{
    nlh_geometry g;
    SysDev sd;
    geometry(g, sd, scale, 4);
    if (sd.pmax2 < 0.0f) return;
    const double open[3] = {0.0, 0.0, far * g.cutoff * sym()};
    for (int rep = 0; rep < 40; ++rep) {
        const Pair p = make_pair(sd, g.cutoff, base, spread, open);
        float q[2][3], o[3];
        const Pair &r = p;
        for (int a = 0; a < 2; ++a) {
            const V &x = a ? r.xj : r.xi;
            const V w = shift(sd.C, a ? r.wj : r.wi);
            for (int k = 0; k < 3; ++k) {
                double u = x.c[k] - 0.5 * (sd.C[3 * k] + sd.C[3 * k + 1] + sd.C[3 * k + 2]);
                u -= w.c[k];
                q[a][k] = (float)u;
            }
        }
        int s[3];
        for (int k = 0; k < 3; ++k) s[k] = p.S[k] - p.wi[k] + p.wj[k];
        for (int k = 0; k < 3; ++k) o[k] = q[0][k] + (float)(0.4 * g.cutoff * sym()) + (float)(open[k] != 0.0 ? -open[k] : 0.0);
        float hq, so = 0.0f;
        const auto run = [&](const float *c) {
            float n[3], b[3];
            for (int k = 0; k < 3; ++k) {
                const float v = std::fmaf(sd.C32[3 * k], (float)s[0],
                                          std::fmaf(sd.C32[3 * k + 1], (float)s[1], std::fmaf(sd.C32[3 * k + 2], (float)s[2], -c[k])));
                n[k] = c[k] - q[0][k];
                b[k] = q[1][k] + v;
            }
            hq = 0.5f * std::fmaf(n[2], n[2], std::fmaf(n[1], n[1], n[0] * n[0]));
            const float bq = 0.5f * std::fmaf(b[2], b[2], std::fmaf(b[1], b[1], b[0] * b[0]));
            return dot3(n[0], n[1], n[2], b[0], b[1], b[2], bq + (hq - sd.rc2half));
        };
        float D = run(o);
        if (hq > 32.0f * sd.rc2half) {
            const float c[3] = {q[0][0], q[0][1], q[0][2]};
            D = run(c);
            so = std::sqrt(2.0f * sd.rc2half * (c[0] * c[0] + c[1] * c[1] + c[2] * c[2]));
        }
        const float tol = hq + so < 1.0e30f ? std::fmaf(so, kSmallTolFar, std::fmaf(hq, kSmallTol, sd.small_tol)) : kFar32 * kFar32;
        T.add(D, tol, p.hit, p.truth);
    }
}

}  // namespace

int main()
{
    Tally tile, small;
    for (int c = 0; c < 20000; ++c) {
        const double scale = c % 4 == 0 ? std::pow(10.0, -10.0 + 16.0 * uni()) : 1.0;
        const int base = c % 3 == 0 ? pick(-250, 250) : 0, spread = c % 5 == 0 ? 250 : (c % 5 == 1 ? 3 : 0);
        const double far = c % 7 == 0 ? std::pow(10.0, 6.0 * uni()) : 0.0;
        tile_case(tile, scale, base, spread, far);
        small_case(small, scale, base, spread / 2, far);
    }
    for (const Tally *t : {&tile, &small})
        std::printf("%ld %ld %.4f %.4f\n", t->pairs, t->wrong, t->worst, (double)t->exact / t->pairs);
    return 0;
}
