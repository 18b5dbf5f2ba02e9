// Host-side check of centre_pair (common.hpp): at the smallest distance that it
// admits for a pair of orders and radii, the closed forms at the sphere centres
// give what the sums over the grids give, up to the rounding of those sums.
#include "common.hpp"

#include <cmath>
#include <cstdio>
#include <random>

using namespace sphstk;

namespace {
std::mt19937 rng(5);
std::normal_distribution<double> nd;
void random3(double *v) {
    for (int k = 0; k < 3; k++) v[k] = nd(rng);
}
double dot(const double *a, const double *b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }
void cross(const double *a, const double *b, double *o) {
    o[0] = a[1] * b[2] - a[2] * b[1], o[1] = a[2] * b[0] - a[0] * b[2], o[2] = a[0] * b[1] - a[1] * b[0];
}

// largest difference of the closed-form traction of a rigid-body density on a
// sphere of radius rs and order ps from its grid sum, on a sphere of radius rt
// at distance d, relative to the largest traction there
double traction_error(double d, double rs, int ps, double rt) {
    const ShTables &S = sh_tables(ps), &T = sh_tables(8);
    double worst = 0.0;
    for (int it = 0; it < 8; it++) {
        double F[3], Tq[3], u[3];
        random3(F), random3(Tq), random3(u);
        const double len = std::sqrt(dot(u, u));
        double err = 0.0, size = 0.0;
        for (int j = 0; j < T.npts; j++) {
            const double *n = &T.eta[3 * j];
            double x[3], g[3] = {0, 0, 0}, c[3], q[3];
            for (int k = 0; k < 3; k++) x[k] = d * u[k] / len + rt * n[k];
            for (int i = 0; i < S.npts; i++) {
                const double *e = &S.eta[3 * i];
                double te[3], r[3], f[3];
                cross(Tq, e, te);
                for (int k = 0; k < 3; k++) {
                    r[k] = x[k] - rs * e[k];
                    f[k] = S.w[i] * (F[k] / (4 * kPi) + 3 * te[k] / (8 * kPi * rs));
                }
                const double w = -3 / (4 * kPi) * dot(r, f) * dot(r, n) * std::pow(dot(r, r), -2.5);
                for (int k = 0; k < 3; k++) g[k] += w * r[k];
            }
            const double r2 = dot(x, x), i5 = std::pow(r2, -2.5), rn = dot(x, n), rF = dot(x, F), Fn = dot(F, n);
            cross(Tq, x, q);
            const double qn = dot(q, n);
            for (int k = 0; k < 3; k++) {
                c[k] = -3 / (4 * kPi) * x[k] * rF * rn * i5 +
                       rs * rs / (12 * kPi) * (-3 * (F[k] * rn + x[k] * Fn + n[k] * rF) + 15 * rF * rn * x[k] / r2) * i5 -
                       3 / (8 * kPi) * (q[k] * rn + x[k] * qn) * i5;
                err = std::fmax(err, std::fabs(c[k] - g[k]));
                size = std::fmax(size, std::fabs(c[k]));
            }
        }
        worst = std::fmax(worst, err / size);
    }
    return worst;
}

// the same for the rigid-body averages, over a sphere of radius rt and order pt,
// of the flow of point forces at distance d - rs from its centre (Faxen's laws)
double average_error(double d, double rs, double rt, int pt) {
    const ShTables &T = sh_tables(pt);
    double worst = 0.0;
    for (int it = 0; it < 40; it++) {
        double f[3], u[3], y[3], v[3] = {0, 0, 0}, o[3] = {0, 0, 0}, fy[3];
        random3(f), random3(u);
        const double len = std::sqrt(dot(u, u));
        for (int k = 0; k < 3; k++) y[k] = -(d - rs) * u[k] / len; // from the point force to the centre
        for (int j = 0; j < T.npts; j++) {
            double x[3], g[3], ng[3];
            for (int k = 0; k < 3; k++) x[k] = y[k] + rt * T.eta[3 * j + k];
            const double r2 = dot(x, x), r = std::sqrt(r2), fx = dot(f, x);
            for (int k = 0; k < 3; k++) g[k] = f[k] / r + x[k] * fx / (r2 * r);
            cross(&T.eta[3 * j], g, ng);
            for (int k = 0; k < 3; k++) v[k] += T.w[j] * g[k] / (4 * kPi), o[k] += 3 * T.w[j] * ng[k] / (8 * kPi * rt);
        }
        const double r2 = dot(y, y), r = std::sqrt(r2), fd = dot(f, y);
        cross(f, y, fy);
        for (int k = 0; k < 3; k++) {
            const double V = f[k] / r + y[k] * fd / (r2 * r) + rt * rt / 6 * (2 * f[k] / (r2 * r) - 6 * y[k] * fd / (r2 * r2 * r));
            worst = std::fmax(worst, std::fabs(V - v[k]) * r / std::sqrt(dot(f, f)));
            worst = std::fmax(worst, std::fabs(fy[k] / (r2 * r) - o[k]) * r2 / std::sqrt(dot(f, f)));
        }
    }
    return worst;
}
} // namespace

int main() {
    int fails = 0;
    for (int p : {6, 8, 10, 11, 12, 14, 16, 20})
        for (double rt : {1.0, 0.33, 3.0}) {
            const double rs = 1.0;
            double lo = 1.5 * (rs + rt), hi = 4.0 * (rs + rt);
            if (!centre_pair(hi, rs, p, rt, p)) {
                std::printf("p=%d: not admitted at 4 radius sums FAIL\n", p);
                fails++;
                continue;
            }
            for (int k = 0; k < 60; k++) {
                const double mid = 0.5 * (lo + hi);
                (centre_pair(mid, rs, p, rt, p) ? hi : lo) = mid;
            }
            const double et = traction_error(hi, rs, p, rt), ea = average_error(hi, rs, rt, p);
            // below 4 radius sums: what the predicate allows, 5e-15, and the rounding of up
            // to 882 products that partly cancel (each at most 1.1e-16 of five times the sum,
            // adding up like a random walk: 1.7e-14)
            const bool closer = hi < 3.999 * (rs + rt);
            const bool ok = !closer || (et < 2.2e-14 && ea < 2.2e-14);
            std::printf("p=%d radii 1:%.2f from %.3f radius sums: traction %.1e averages %.1e %s\n", p, rt,
                        hi / (rs + rt), et, ea, ok ? "ok" : "FAIL");
            fails += !ok;
            // unequal orders: the lower one decides
            const bool mixed = centre_pair(hi * 0.999, rs, p, rt, 20) && centre_pair(hi * 0.999, rs, 20, rt, p);
            if (mixed) {
                std::printf("p=%d radii 1:%.2f: admitted by the other sphere's order alone FAIL\n", p, rt);
                fails++;
            }
        }
    return fails ? 1 : 0;
}
