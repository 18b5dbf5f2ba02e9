// Host-side spherical-harmonic set-up: Gauss-Legendre rule, the per-order unit
// grid of Sphere/Shexp.cpp:206-271 (poles dropped as in
// BIE/SphereSTKSHOperator.cpp:103-121) and the analysis matrix that maps
// body-frame grid values to vector-SH coefficients (the role of SCTL
// Grid2VecSHC behind Shexp::calcSpectralCoeff, Sphere/Shexp.cpp:408-447).
//
// Basis (per degree n<=p, order 0<=m<=n; m<0 implied by conjugation):
//   y_nm = D_n^m on the unit sphere, D_n^m = (d/dx + i d/dy)^m (d/dz)^(n-m) (1/r)
//   e_r = y r,  e_s = grad_s y,  e_t = r x grad_s y,
// with |y_nm|^2 integrating to 4 pi (n-m)!(n+m)!/(2n+1) and |e_s|^2, |e_t|^2 to
// n(n+1) times that.  The analysis is the orthogonal projection in the grid's
// quadrature inner product, which is exact for vector-SH degree <= p.
#include "common.hpp"
#include "pool.hpp"

#include <algorithm>
#include <cmath>
#include <complex>
#include <map>
#include <memory>
#include <mutex>

namespace sphstk {

using cplx = std::complex<double>;

void gauss_legendre(int n, std::vector<double> &x, std::vector<double> &w) {
    x.assign(n, 0.0);
    w.assign(n, 0.0);
    for (int i = 0; i < (n + 1) / 2; i++) {
        // Newton iteration on P_n starting from the Tricomi approximation of root i (descending)
        double z = std::cos(kPi * (4.0 * i + 3.0) / (4.0 * n + 2.0));
        double pn = 0, dpn = 1;
        for (int it = 0; it < 60; it++) {
            double pm1 = 1.0, p0 = z;
            if (n == 0) p0 = 1.0;
            for (int k = 1; k < n; k++) {
                const double pk1 = ((2 * k + 1) * z * p0 - k * pm1) / (k + 1);
                pm1 = p0;
                p0 = pk1;
            }
            pn = p0;
            dpn = n * (pm1 - z * pn) / (1.0 - z * z);
            const double dz = pn / dpn;
            z -= dz;
            if (std::fabs(dz) <= 1e-17) break;
        }
        double pm1 = 1.0, p0 = z;
        for (int k = 1; k < n; k++) {
            const double pk1 = ((2 * k + 1) * z * p0 - k * pm1) / (k + 1);
            pm1 = p0;
            p0 = pk1;
        }
        dpn = n * (pm1 - z * p0) / (1.0 - z * z);
        x[n - 1 - i] = z;
        x[i] = -z;
        w[i] = w[n - 1 - i] = 2.0 / ((1.0 - z * z) * dpn * dpn);
    }
    if (n % 2) x[n / 2] = 0.0;
}

// D_n^m(x), 0<=m<=n<=P, by the diagonal and the three-term z recurrence.
static void solid_harmonics(int P, const double *x, std::vector<cplx> &D) {
    D.assign(tri_size(P), cplx(0, 0));
    const double r2 = x[0] * x[0] + x[1] * x[1] + x[2] * x[2];
    const double ir2 = 1.0 / r2;
    const cplx xy(x[0], x[1]);
    D[0] = 1.0 / std::sqrt(r2);
    for (int m = 1; m <= P; m++) D[tri(m, m)] = -(2.0 * m - 1.0) * ir2 * xy * D[tri(m - 1, m - 1)];
    for (int m = 0; m < P; m++) {
        cplx prev = 0.0, cur = D[tri(m, m)];
        for (int n = m; n < P; n++) {
            const cplx next = -((2.0 * n + 1.0) * x[2] * cur + double(n * n - m * m) * prev) * ir2;
            D[tri(n + 1, m)] = next;
            prev = cur;
            cur = next;
        }
    }
}

// Rows of the synthesis operator at one unit vector e (body frame): the value
// component c of the expansion at e is sum_j row[c * 6Q + j] coef[j].
static void synthesis_rows_at(int p, const double *e, std::vector<cplx> &D, double *row) {
    const int Q = tri_size(p), ncoef = 6 * Q;
    std::fill(row, row + 3 * ncoef, 0.0);
    solid_harmonics(p + 1, e, D);
    for (int n = 0; n <= p; n++)
        for (int m = 0; m <= n; m++) {
            const int k = tri(n, m);
            cplx g[3];
            g[2] = D[tri(n + 1, m)];
            if (m > 0) {
                g[0] = 0.5 * (D[tri(n + 1, m + 1)] - D[tri(n + 1, m - 1)]);
                g[1] = cplx(0, -0.5) * (D[tri(n + 1, m + 1)] + D[tri(n + 1, m - 1)]);
            } else {
                g[0] = D[tri(n + 1, 1)].real();
                g[1] = D[tri(n + 1, 1)].imag();
            }
            const cplx y = D[k];
            cplx gs[3], xt[3];
            for (int c = 0; c < 3; c++) gs[c] = g[c] + (n + 1.0) * y * e[c];
            xt[0] = e[1] * g[2] - e[2] * g[1];
            xt[1] = e[2] * g[0] - e[0] * g[2];
            xt[2] = e[0] * g[1] - e[1] * g[0];
            const double eps = m ? 2.0 : 1.0;
            for (int c = 0; c < 3; c++) {
                double *rc = row + size_t(c) * ncoef;
                const cplx br = y * e[c], bs = gs[c], bt = xt[c];
                rc[2 * k] = eps * br.real();
                rc[2 * k + 1] = -eps * br.imag();
                rc[2 * Q + 2 * k] = eps * bs.real();
                rc[2 * Q + 2 * k + 1] = -eps * bs.imag();
                rc[4 * Q + 2 * k] = eps * bt.real();
                rc[4 * Q + 2 * k + 1] = -eps * bt.imag();
            }
        }
}

std::vector<double> pole_rows(int p) {
    const int ncoef = 6 * tri_size(p);
    std::vector<double> rows(size_t(6) * ncoef);
    std::vector<cplx> D;
    const double north[3] = {0.0, 0.0, 1.0}, south[3] = {0.0, 0.0, -1.0};
    synthesis_rows_at(p, north, D, rows.data());
    synthesis_rows_at(p, south, D, rows.data() + size_t(3) * ncoef);
    return rows;
}

std::vector<double> synthesis_of_blocks(int p, const std::vector<double> &blocks) {
    const ShTables &t = sh_tables(p);
    const size_t n3 = 3 * (size_t)t.npts;
    std::vector<double> m(n3 * 6 * t.Q);
    for (int n = 0; n <= p; n++)
        for (int k = tri(n, 0); k < tri(n + 1, 0); k++)
            for (int c = 0; c < 2; c++) {
                const double *b = &blocks[5 * n];
                const double *sr = &t.synth[n3 * (2 * k + c)], *ss = &t.synth[n3 * (2 * t.Q + 2 * k + c)],
                             *st = &t.synth[n3 * (4 * t.Q + 2 * k + c)];
                double *mr = &m[n3 * (2 * k + c)], *ms = &m[n3 * (2 * t.Q + 2 * k + c)],
                       *mt = &m[n3 * (4 * t.Q + 2 * k + c)];
                for (size_t i = 0; i < n3; i++) {
                    mr[i] = b[0] * sr[i] + b[2] * ss[i];
                    ms[i] = b[1] * sr[i] + b[3] * ss[i];
                    mt[i] = b[4] * st[i];
                }
            }
    return m;
}

// Analysis and synthesis matrices of degree p on the points and weights of t.
static void fill_matrices(ShTables *t, int p);

static std::unique_ptr<ShTables> build_tables(int p) {
    auto t = std::make_unique<ShTables>();
    t->p = p;
    t->npts = grid_points(p);
    t->Q = tri_size(p);
    std::vector<double> xg, wg;
    gauss_legendre(p + 1, xg, wg);
    const int nphi = 2 * p + 2;
    t->eta.resize(3 * t->npts);
    t->w.resize(t->npts);
    for (int j = 0; j <= p; j++) {
        const double ct = xg[p - j], st = std::sqrt(1.0 - ct * ct);
        for (int k = 0; k < nphi; k++) {
            const double ph = 2.0 * kPi * k / nphi;
            const int q = j * nphi + k;
            t->eta[3 * q] = st * std::cos(ph);
            t->eta[3 * q + 1] = st * std::sin(ph);
            t->eta[3 * q + 2] = ct;
            t->w[q] = 2.0 * kPi / nphi * wg[p - j];
        }
    }
    fill_matrices(t.get(), p);
    return t;
}

// Quadrature rules on the sphere with octahedral symmetry (the structure is
// Lebedev's, Zh. Vychisl. Mat. Mat. Fiz. 16 (1976)): per orbit a point, its
// coordinates in ascending order, and the weight of each of its images under
// permutations and signs, the weights of a rule adding up to one.  Solved on the
// moments of (x^4 + y^4 + z^4)^a (xyz)^2b, which span the invariant polynomials on the
// sphere, by tests/golden/make_octahedral_rules.py.  A rule for
// order q integrates degree 2q + 1, as the Gauss-Legendre grid of 2 (q + 1)^2
// points does, with about two thirds of its points (order 6: nine tenths): a
// far-field level evaluates the product of two spheres' points.
struct Orbit {
    double x, y, z, w;
};
static const std::vector<Orbit> kRules[] = {
    // order 1: 6 points (degree 3)
    {{0.0, 0.0, 1.0, 0.16666666666666666}},
    // order 2: 14 points (degree 5)
    {{0.0, 0.0, 1.0, 0.06666666666666667},
     {0.5773502691896257, 0.5773502691896257, 0.5773502691896257, 0.075}},
    // order 3: 26 points (degree 7)
    {{0.0, 0.0, 1.0, 0.047619047619047616},
     {0.0, 0.7071067811865476, 0.7071067811865476, 0.0380952380952381},
     {0.5773502691896257, 0.5773502691896257, 0.5773502691896257, 0.03214285714285714}},
    // order 4: 38 points (degree 9)
    {{0.0, 0.0, 1.0, 0.009523809523809525},
     {0.5773502691896257, 0.5773502691896257, 0.5773502691896257, 0.03214285714285714},
     {0.0, 0.45970084338098305, 0.8880738339771153, 0.02857142857142857}},
    // order 5: 50 points (degree 11)
    {{0.0, 0.0, 1.0, 0.012698412698412698},
     {0.0, 0.7071067811865476, 0.7071067811865476, 0.022574955908289243},
     {0.5773502691896257, 0.5773502691896257, 0.5773502691896257, 0.02109375},
     {0.30151134457776363, 0.30151134457776363, 0.9045340337332909, 0.02017333553791887}},
    // order 6: order 7's 86 points (of the rules of degree 13 this family has one with
    // 74 points, whose vertices have a negative weight)
    {{0.0, 0.0, 1.0, 0.011544011544011544},
     {0.5773502691896257, 0.5773502691896257, 0.5773502691896257, 0.011943909085856283},
     {0.36960284645415026, 0.36960284645415026, 0.8525183117012676, 0.011110555710603402},
     {0.18906355288539547, 0.6943540066026663, 0.6943540066026663, 0.011876501294537142},
     {0.0, 0.3742430390903412, 0.9273306571511725, 0.011812303746904475}},
    // order 7: 86 points (degree 15)
    {{0.0, 0.0, 1.0, 0.011544011544011544},
     {0.5773502691896257, 0.5773502691896257, 0.5773502691896257, 0.011943909085856283},
     {0.36960284645415026, 0.36960284645415026, 0.8525183117012676, 0.011110555710603402},
     {0.18906355288539547, 0.6943540066026663, 0.6943540066026663, 0.011876501294537142},
     {0.0, 0.3742430390903412, 0.9273306571511725, 0.011812303746904475}},
    // order 8: 110 points (degree 17)
    {{0.0, 0.0, 1.0, 0.0038282704949371615},
     {0.5773502691896257, 0.5773502691896257, 0.5773502691896257, 0.009793737512487513},
     {0.18511563534473616, 0.18511563534473616, 0.9651240350865941, 0.008211737283191111},
     {0.39568947305594193, 0.39568947305594193, 0.8287699812525922, 0.009595471336070962},
     {0.21595729184584883, 0.6904210483822921, 0.6904210483822921, 0.009942814891178103},
     {0.0, 0.4783690288121502, 0.8781589106040661, 0.009694996361663029}},
    // order 9: 146 points (degree 19)
    {{0.0, 0.0, 1.0, 0.0005996313688621381},
     {0.0, 0.7071067811865476, 0.7071067811865476, 0.0073729997186207565},
     {0.5773502691896257, 0.5773502691896257, 0.5773502691896257, 0.007210515360144488},
     {0.15746766720390817, 0.15746766720390817, 0.9748886436771732, 0.007574394159054034},
     {0.41749612279654535, 0.41749612279654535, 0.8070898183595825, 0.006753829486314478},
     {0.29129888220952677, 0.6764410400114264, 0.6764410400114264, 0.007116355493117555},
     {0.14035538117131832, 0.44933283232695576, 0.8822700112603227, 0.0069910873533032625}},
    // order 10: 170 points (degree 21)
    {{0.0, 0.0, 1.0, 0.005544842902037364},
     {0.0, 0.7071067811865476, 0.7071067811865476, 0.006071332770670752},
     {0.5773502691896257, 0.5773502691896257, 0.5773502691896257, 0.006383674773515093},
     {0.3007935951377015, 0.6743601460362766, 0.6743601460362766, 0.006317929009813725},
     {0.431891069671941, 0.431891069671941, 0.7917955593934921, 0.006201670006589077},
     {0.25512526211141345, 0.25512526211141345, 0.9326425903126906, 0.00518338758774779},
     {0.0, 0.26139313603359887, 0.9652324219764483, 0.005477143385137348},
     {0.14466307443251153, 0.49904531617960374, 0.8544158046846588, 0.005968383987681156}},
};

static std::unique_ptr<ShTables> build_level_tables(int q) {
    auto t = std::make_unique<ShTables>();
    t->p = q;
    t->Q = tri_size(q);
    for (const Orbit &o : kRules[q - 1]) {
        double c[3] = {o.x, o.y, o.z};
        do {
            for (int s = 0; s < 8; s++) {
                bool twice = false;
                for (int k = 0; k < 3; k++) twice = twice || ((s >> k & 1) && c[k] == 0.0);
                if (twice) continue;
                for (int k = 0; k < 3; k++) t->eta.push_back(s >> k & 1 ? -c[k] : c[k]);
                t->w.push_back(4.0 * kPi * o.w);
            }
        } while (std::next_permutation(c, c + 3));
    }
    t->npts = (int)t->w.size();
    fill_matrices(t.get(), q);
    return t;
}

const ShTables &level_tables(int q) {
    if (q < 1 || q > (int)(sizeof kRules / sizeof kRules[0])) return sh_tables(q);
    static std::mutex mu;
    static std::map<int, std::unique_ptr<ShTables>> cache;
    std::lock_guard<std::mutex> lock(mu);
    auto &t = cache[q];
    if (!t) t = build_level_tables(q);
    return *t;
}

static void fill_matrices(ShTables *t, int p) {
    const int Q = t->Q, rows = 6 * Q, cols = 3 * t->npts;
    t->anal.assign(size_t(rows) * cols, 0.0);
    std::vector<double> invN(Q);
    for (int n = 0; n <= p; n++)
        for (int m = 0; m <= n; m++) {
            double f = 4.0 * kPi / (2.0 * n + 1.0);
            for (int k = 2; k <= n - m; k++) f *= k;
            for (int k = 2; k <= n + m; k++) f *= k;
            invN[tri(n, m)] = 1.0 / f;
        }
    t->synth.assign(size_t(cols) * rows, 0.0);
    std::vector<cplx> D;
    for (int q = 0; q < t->npts; q++) {
        const double *e = &t->eta[3 * q];
        solid_harmonics(p + 1, e, D);
        for (int n = 0; n <= p; n++)
            for (int m = 0; m <= n; m++) {
                const int k = tri(n, m);
                // Cartesian gradient of D_n^m from degree n+1
                cplx g[3];
                g[2] = D[tri(n + 1, m)];
                if (m > 0) {
                    g[0] = 0.5 * (D[tri(n + 1, m + 1)] - D[tri(n + 1, m - 1)]);
                    g[1] = cplx(0, -0.5) * (D[tri(n + 1, m + 1)] + D[tri(n + 1, m - 1)]);
                } else {
                    g[0] = D[tri(n + 1, 1)].real();
                    g[1] = D[tri(n + 1, 1)].imag();
                }
                const cplx y = D[k];
                cplx gs[3], xt[3];
                for (int c = 0; c < 3; c++) gs[c] = g[c] + (n + 1.0) * y * e[c];
                xt[0] = e[1] * g[2] - e[2] * g[1];
                xt[1] = e[2] * g[0] - e[0] * g[2];
                xt[2] = e[0] * g[1] - e[1] * g[0];
                // synthesis: value_c = sum_k eps_m Re(F_r y e_c + F_s gs_c + F_t xt_c), F stored (re, im)
                const double eps = m ? 2.0 : 1.0;
                for (int c = 0; c < 3; c++) {
                    const size_t r = size_t(3 * q + c);
                    const cplx br = y * e[c], bs = gs[c], bt = xt[c];
                    t->synth[size_t(2 * k) * cols + r] = eps * br.real();
                    t->synth[size_t(2 * k + 1) * cols + r] = -eps * br.imag();
                    t->synth[size_t(2 * Q + 2 * k) * cols + r] = eps * bs.real();
                    t->synth[size_t(2 * Q + 2 * k + 1) * cols + r] = -eps * bs.imag();
                    t->synth[size_t(4 * Q + 2 * k) * cols + r] = eps * bt.real();
                    t->synth[size_t(4 * Q + 2 * k + 1) * cols + r] = -eps * bt.imag();
                }
                const double wr = t->w[q] * invN[k];
                const double wt = n > 0 ? t->w[q] * invN[k] / (n * (n + 1.0)) : 0.0;
                for (int c = 0; c < 3; c++) {
                    const size_t col = size_t(3 * q + c) * rows;
                    const cplx cr = std::conj(y) * e[c] * wr;
                    const cplx cs = std::conj(gs[c]) * wt;
                    const cplx ctt = std::conj(xt[c]) * wt;
                    t->anal[col + 2 * k] = cr.real();
                    t->anal[col + 2 * Q + 2 * k] = cs.real();
                    t->anal[col + 4 * Q + 2 * k] = ctt.real();
                    if (m > 0) {
                        t->anal[col + 2 * k + 1] = cr.imag();
                        t->anal[col + 2 * Q + 2 * k + 1] = cs.imag();
                        t->anal[col + 4 * Q + 2 * k + 1] = ctt.imag();
                    }
                }
            }
    }
}

// rows of a coefficient vector (6Q layout) that belong to degrees <= pc
static std::vector<int> coef_rows_upto(int p, int pc) {
    const int Q = tri_size(p);
    std::vector<int> r;
    for (int blk = 0; blk < 3; blk++)
        for (int n = 0; n <= std::min(p, pc); n++)
            for (int m = 0; m <= n; m++) {
                r.push_back(blk * 2 * Q + 2 * tri(n, m));
                r.push_back(blk * 2 * Q + 2 * tri(n, m) + 1);
            }
    return r;
}

// Coefficients of degree q + 1 of a field given on the grid of a level of order
// q, one row per entry of `cols` (columns of the tables of degree q + 1), 3 npts
// columns, column-major.  The field that another sphere leaves on a level
// decays with the degree, so the part of it beyond degree q that is worth most is
// degree q + 1, and the grid shows most of that: its points are more than the
// degrees up to q need.  Least squares in the quadrature's norm, which leaves the
// degrees up to q alone (the rule integrates degree 2q + 1), held back by kFitNoise
// where the grid hardly shows a mode and the higher degrees would take it over:
//   c = (H + kFitNoise I)^-1 Phi^T W f,  H = Phi^T W Phi,  Phi of unit norm on the sphere.
// With it on both sides (the source side is the adjoint) a level's error is 0.06 to
// 0.79 of that of the Gauss-Legendre grid of its order, at no cost per apply: for two
// spheres of order 12 and random densities 0.14 for order 10 from 4.8 radius sums,
// 0.41 for order 7 from 3, 0.79 for order 5 from 2 and radii 1:3.  Without it the
// octahedral grids' was up to 1.03 of it.  (0.02 and 0.1 in place of 0.05 change the
// error by up to a tenth.)
constexpr double kFitNoise = 0.05;
static std::vector<double> next_degree(const ShTables &C, int q, std::vector<int> &cols) {
    ShTables T;
    T.p = q + 1;
    T.Q = tri_size(q + 1);
    T.npts = C.npts;
    T.eta = C.eta;
    T.w = C.w;
    fill_matrices(&T, q + 1);
    const ShTables &G = sh_tables(q + 1);
    const size_t n = 3 * (size_t)C.npts, ng = 3 * (size_t)G.npts;
    cols.clear();
    for (int blk = 0; blk < 3; blk++)
        for (int m = 0; m <= q + 1; m++)
            for (int c = 0; c < (m ? 2 : 1); c++) cols.push_back(2 * (blk * T.Q + tri(q + 1, m)) + c);
    const size_t k = cols.size();
    std::vector<double> phi(n * k), scale(k), H(k * k), Z(k * n);
    for (size_t a = 0; a < k; a++) {
        double norm = 0.0;
        for (size_t i = 0; i < ng; i++) norm += G.w[i / 3] * G.synth[cols[a] * ng + i] * G.synth[cols[a] * ng + i];
        scale[a] = 1.0 / std::sqrt(norm);
        for (size_t i = 0; i < n; i++) phi[a * n + i] = scale[a] * T.synth[cols[a] * n + i];
    }
    for (size_t a = 0; a < k; a++)
        for (size_t b = 0; b < k; b++) {
            double v = a == b ? kFitNoise : 0.0;
            for (size_t i = 0; i < n; i++) v += C.w[i / 3] * phi[a * n + i] * phi[b * n + i];
            H[a * k + b] = v;
        }
    for (size_t i = 0; i < n; i++)
        for (size_t a = 0; a < k; a++) Z[i * k + a] = C.w[i / 3] * phi[a * n + i];
    // Cholesky factor of H in its lower triangle, then the two substitutions
    for (size_t a = 0; a < k; a++)
        for (size_t b = 0; b <= a; b++) {
            double v = H[a * k + b];
            for (size_t c = 0; c < b; c++) v -= H[a * k + c] * H[b * k + c];
            H[a * k + b] = a == b ? std::sqrt(v) : v / H[b * k + b];
        }
    for (size_t i = 0; i < n; i++) {
        double *z = &Z[i * k];
        for (size_t a = 0; a < k; a++) {
            for (size_t c = 0; c < a; c++) z[a] -= H[a * k + c] * z[c];
            z[a] /= H[a * k + a];
        }
        for (size_t a = k; a-- > 0;) {
            for (size_t c = a + 1; c < k; c++) z[a] -= H[c * k + a] * z[c];
            z[a] /= H[a * k + a];
        }
        for (size_t a = 0; a < k; a++) z[a] *= scale[a];
    }
    return Z;
}

// (level: to and from a level grid, whose fields are taken up to degree pc + 1)
static std::unique_ptr<Resample> build_resample(int p, int pc, const ShTables &C, bool same, bool level = false) {
    auto rs = std::make_unique<Resample>();
    rs->p = p;
    rs->pc = pc;
    const ShTables &F = sh_tables(p);
    rs->n = F.npts;
    rs->nc = C.npts;
    const int QF = F.Q, QC = C.Q;
    const int rowsF = 6 * QF, rowsC = 6 * QC;
    if (same) { // same grid: identity in both directions
        const int nn = 3 * F.npts;
        rs->down.assign(size_t(nn) * nn, 0.0);
        for (int i = 0; i < nn; i++) rs->down[size_t(i) * nn + i] = 1.0;
        rs->up = rs->down;
        return rs;
    }
    const std::vector<int> rf = coef_rows_upto(p, rs->pc), rc = coef_rows_upto(rs->pc, rs->pc);
    // down = synth_C[:, rc] * anal_F[rf, :]
    const int nF = 3 * F.npts, nC = 3 * C.npts;
    rs->down.assign(size_t(nC) * nF, 0.0);
    for (int col = 0; col < nF; col++)
        for (size_t k = 0; k < rf.size(); k++) {
            const double a = F.anal[size_t(col) * rowsF + rf[k]];
            if (a == 0.0) continue;
            const double *sc = &C.synth[size_t(rc[k]) * nC];
            double *o = &rs->down[size_t(col) * nC];
            for (int r = 0; r < nC; r++) o[r] += sc[r] * a;
        }
    // up = synth_F[:, rf] * anal_C[rc, :]
    rs->up.assign(size_t(nF) * nC, 0.0);
    for (int col = 0; col < nC; col++)
        for (size_t k = 0; k < rc.size(); k++) {
            const double a = C.anal[size_t(col) * rowsC + rc[k]];
            if (a == 0.0) continue;
            const double *sf = &F.synth[size_t(rf[k]) * nF];
            double *o = &rs->up[size_t(col) * nF];
            for (int r = 0; r < nF; r++) o[r] += sf[r] * a;
        }
    if (level && p > pc) {
        std::vector<int> cols;
        const std::vector<double> Z = next_degree(C, pc, cols);
        const int Q1 = tri_size(pc + 1);
        std::vector<double> up(size_t(nF) * nC, 0.0);
        for (int col = 0; col < nC; col++)
            for (size_t k = 0; k < cols.size(); k++) {
                const int blk = cols[k] / (2 * Q1);
                const double a = Z[size_t(col) * cols.size() + k];
                const double *sf = &F.synth[size_t(cols[k] + 2 * blk * (QF - Q1)) * nF];
                double *o = &up[size_t(col) * nF];
                for (int r = 0; r < nF; r++) o[r] += sf[r] * a;
            }
        // the source side is the adjoint in the two quadratures
        for (int col = 0; col < nC; col++)
            for (int r = 0; r < nF; r++) {
                rs->up[size_t(col) * nF + r] += up[size_t(col) * nF + r];
                rs->down[size_t(r) * nC + col] += up[size_t(col) * nF + r] * F.w[r / 3] / C.w[col / 3];
            }
    }
    return rs;
}

const Resample &resample_tables(int p, int pc) {
    static Tables<std::pair<int, int>, Resample> kept;
    return kept.get({p, pc}, [&] { return build_resample(p, pc, sh_tables(pc), pc == p); });
}

const Resample &level_resample(int p, int pc) {
    static Tables<std::pair<int, int>, Resample> kept;
    return kept.get({p, pc}, [&] { return build_resample(p, pc, level_tables(pc), false, true); });
}

const ShTables &sh_tables(int p) {
    static std::mutex mu;
    static std::map<int, std::unique_ptr<ShTables>> cache;
    std::lock_guard<std::mutex> lock(mu);
    auto it = cache.find(p);
    if (it != cache.end()) return *it->second;
    auto t = build_tables(p);
    const ShTables &ref = *t;
    cache[p] = std::move(t);
    return ref;
}

} // namespace sphstk
