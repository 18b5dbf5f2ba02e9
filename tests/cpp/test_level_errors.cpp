// Host-side check of the far-field levels' accuracy: two spheres at the
// separation where a level starts, traction of a random density of one on the
// other, fine grids against the level.  A level may be no further off than the
// Gauss-Legendre grid of its order, and its quadrature weights are positive.
#include "common.hpp"

#include <cmath>
#include <cstdio>
#include <random>

using namespace sphstk;
typedef std::vector<double> Vec;

static void rotate(const double *q, double s, const double *v, double *o) {
    const double w = q[0], x = s * q[1], y = s * q[2], z = s * q[3];
    const double tx = 2 * (y * v[2] - z * v[1]), ty = 2 * (z * v[0] - x * v[2]), tz = 2 * (x * v[1] - y * v[0]);
    o[0] = v[0] + w * tx + y * tz - z * ty;
    o[1] = v[1] + w * ty + z * tx - x * tz;
    o[2] = v[2] + w * tz + x * ty - y * tx;
}
static Vec rotated(const double *q, double s, const Vec &f) {
    Vec o(f.size());
    for (size_t i = 0; i < f.size(); i += 3) rotate(q, s, &f[i], &o[i]);
    return o;
}
static Vec times(const Vec &m, const Vec &x, size_t rows) {
    Vec y(rows, 0.0);
    for (size_t c = 0; c < x.size(); c++)
        for (size_t r = 0; r < rows; r++) y[r] += m[c * rows + r] * x[c];
    return y;
}
// traction (without its factor) at the points of T, radius Rt at `cen`, of the lab-frame density f on S, radius 1
static Vec pair_sum(const ShTables &S, const ShTables &T, const double *qs, const double *qt, double Rt,
                    const double *cen, const Vec &f) {
    const Vec src = rotated(qs, 1.0, S.eta), nrm = rotated(qt, 1.0, T.eta);
    Vec out(3 * T.npts, 0.0);
    for (int j = 0; j < T.npts; j++)
        for (int i = 0; i < S.npts; i++) {
            double d[3], df = 0, dn = 0, r2 = 0;
            for (int k = 0; k < 3; k++) {
                d[k] = cen[k] + Rt * nrm[3 * j + k] - src[3 * i + k];
                df += d[k] * f[3 * i + k], dn += d[k] * nrm[3 * j + k], r2 += d[k] * d[k];
            }
            const double g = S.w[i] * df * dn / (r2 * r2 * std::sqrt(r2));
            for (int k = 0; k < 3; k++) out[3 * j + k] += g * d[k];
        }
    return out;
}

int main() {
    // order of the spheres, order of the level, separation where it starts (in R_s + R_t), R_t
    struct Case {
        int p, q;
        double sep, Rt;
    };
    const Case cases[] = {
        {8, 5, 2.0, 1.0},  {8, 5, 2.0, 3.0},  {12, 4, 3.0, 1.0},   {12, 3, 5.0, 1.0},   {12, 2, 8.0, 1.0},
        {10, 6, 3.0, 1.0}, {12, 7, 3.0, 1.0}, {14, 8, 3.0, 1.0},   {16, 9, 3.0, 1.0},   {18, 10, 3.0, 0.4},
        {20, 11, 3.0, 1.0}, {12, 5, 6.0, 1.0}, {16, 6, 6.0, 1.0},  {12, 4, 9.0, 1.0},   {12, 3, 16.0, 1.0},
        {12, 10, 4.8, 1.0}, {12, 9, 5.8, 1.0}, {12, 8, 7.35, 1.0}, {12, 7, 10.05, 1.0}, {12, 6, 15.1, 1.0},
        {12, 5, 23.0, 1.0}, {12, 10, 1.5, 1.0}, {12, 10, 1.5, 3.0}, {11, 10, 1.5, 1.0}};
    int fails = 0;
    for (int q = 1; q <= 12; q++)
        for (double w : level_tables(q).w)
            if (!(w > 0.0)) {
                std::printf("order %d: weight %.3e FAIL\n", q, w);
                fails++;
                break;
            }
    for (const Case &c : cases) {
        const ShTables &F = sh_tables(c.p);
        const ShTables *grid[2] = {&sh_tables(c.q), &level_tables(c.q)};
        const Resample *mat[2] = {&resample_tables(c.p, c.q), &level_resample(c.p, c.q)};
        std::mt19937 rng(7);
        std::normal_distribution<double> nd;
        double err[2] = {0.0, 0.0};
        for (int it = 0; it < 12; it++) {
            double qs[4], qt[4], cen[3], ns = 0, nt = 0, nc = 0;
            for (int k = 0; k < 4; k++) ns += (qs[k] = nd(rng)) * qs[k], nt += (qt[k] = nd(rng)) * qt[k];
            for (int k = 0; k < 3; k++) nc += (cen[k] = nd(rng)) * cen[k];
            for (int k = 0; k < 4; k++) qs[k] /= std::sqrt(ns), qt[k] /= std::sqrt(nt);
            for (int k = 0; k < 3; k++) cen[k] *= c.sep * (1.0 + c.Rt) / std::sqrt(nc);
            Vec f(3 * F.npts);
            for (double &v : f) v = nd(rng);
            f = times(F.synth, times(F.anal, f, 6 * F.Q), 3 * F.npts);
            const Vec exact = pair_sum(F, F, qs, qt, c.Rt, cen, rotated(qs, 1.0, f));
            for (int g = 0; g < 2; g++) {
                const Vec d = times(mat[g]->down, f, 3 * grid[g]->npts);
                const Vec l = pair_sum(*grid[g], *grid[g], qs, qt, c.Rt, cen, rotated(qs, 1.0, d));
                const Vec u = rotated(qt, 1.0, times(mat[g]->up, rotated(qt, -1.0, l), 3 * F.npts));
                for (size_t i = 0; i < u.size(); i++) err[g] += (u[i] - exact[i]) * (u[i] - exact[i]);
            }
        }
        const double ratio = std::sqrt(err[1] / err[0]);
        std::printf("p=%d, level of order %d from %.2f, radii 1:%.1f: error %.4f of the Gauss-Legendre grid's %s\n", c.p,
                    c.q, c.sep, c.Rt, ratio, ratio <= 1.0 ? "ok" : "FAIL");
        fails += !(ratio <= 1.0);
    }
    return fails ? 1 : 0;
}
