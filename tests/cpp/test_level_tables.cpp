// Host-side check of the level grids (shtables.cpp): every rule integrates
// products of degree 2q exactly, its analysis and synthesis are a projection of
// degree q, and resampling to and from it reproduces fields of degree q.
#include "common.hpp"

#include <cmath>
#include <cstdio>

using namespace sphstk;

int main() {
    int fails = 0;
    for (int q = 1; q <= 12; q++) {
        const ShTables &t = level_tables(q);
        const int Q6 = 6 * t.Q, n3 = 3 * t.npts;
        double area = 0.0, sq = 0.0, worst = 0.0;
        for (int i = 0; i < t.npts; i++) {
            area += t.w[i];
            const double *e = &t.eta[3 * i];
            sq = std::fmax(sq, std::fabs(e[0] * e[0] + e[1] * e[1] + e[2] * e[2] - 1.0));
        }
        // analysis of each basis field gives that coefficient alone (scaled by
        // the coefficients' very different sizes: compare grid values)
        for (int c = 0; c < Q6; c++) {
            std::vector<double> f(&t.synth[(size_t)c * n3], &t.synth[(size_t)c * n3] + n3), k(Q6, 0.0), g(n3, 0.0);
            double size = 0.0;
            for (double v : f) size = std::fmax(size, std::fabs(v));
            if (size < 1e-12) continue; // (degree 0 has no tangential part)
            for (int i = 0; i < n3; i++)
                for (int r = 0; r < Q6; r++) k[r] += t.anal[(size_t)i * Q6 + r] * f[i];
            for (int r = 0; r < Q6; r++)
                for (int i = 0; i < n3; i++) g[i] += t.synth[(size_t)r * n3 + i] * k[r];
            for (int i = 0; i < n3; i++) worst = std::fmax(worst, std::fabs(g[i] - f[i]) / size);
        }
        double turn = 0.0;
        for (int p : {q, q + 2, 16}) {
            if (p < q) continue;
            // level -> fine -> level is the identity on fields of degree q
            const Resample &rs = level_resample(p, q);
            for (int c = 0; c < Q6; c += 5) {
                const double *f = &t.synth[(size_t)c * n3];
                double size = 0.0;
                for (int i = 0; i < n3; i++) size = std::fmax(size, std::fabs(f[i]));
                if (size < 1e-12) continue; // (degree 0 has no tangential part)
                std::vector<double> u(3 * rs.n, 0.0), d(n3, 0.0);
                for (int i = 0; i < n3; i++)
                    for (int r = 0; r < 3 * rs.n; r++) u[r] += rs.up[(size_t)i * 3 * rs.n + r] * f[i];
                for (int i = 0; i < 3 * rs.n; i++)
                    for (int r = 0; r < n3; r++) d[r] += rs.down[(size_t)i * n3 + r] * u[i];
                for (int i = 0; i < n3; i++) turn = std::fmax(turn, std::fabs(d[i] - f[i]) / size);
            }
        }
        const bool ok = std::fabs(area - 4.0 * kPi) < 1e-13 && sq < 1e-14 && worst < 1e-12 && turn < 1e-11 &&
                        (q > 10 || t.npts < grid_points(q));
        std::printf("q=%d: %d points, area %.1e, projection %.1e, resampling %.1e %s\n", q, t.npts,
                    std::fabs(area - 4.0 * kPi), worst, turn, ok ? "ok" : "FAIL");
        fails += !ok;
    }
    return fails ? 1 : 0;
}
