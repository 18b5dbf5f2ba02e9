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
// permutations and signs, the weights of a rule adding up to one.  Solved by
// Newton's method from random starts on the moments of (x^4 + y^4 + z^4)^a
// (xyz)^2b, which span the invariant polynomials on the sphere.  A rule for
// order q integrates degree 2q + 1, as the Gauss-Legendre grid of 2 (q + 1)^2
// points does, with about two thirds of its points: a far-field level evaluates
// the product of two spheres' points.
struct Orbit {
    double x, y, z, w;
};
static const std::vector<Orbit> kRules[] = {
    // order 1: 6 points (degree 3)
    {{0.0, 0.0, 1.0, 0.16666666666666666}},
    // order 2: 14 points (degree 5)
    {{0.0, 0.0, 1.0, 0.06666666666666611},
     {0.5773502691896258, 0.5773502691896258, 0.5773502691896258, 0.07500000000000041}},
    // order 3: 26 points (degree 7)
    {{0.0, 0.0, 1.0, 0.047619047619047006},
     {0.0, 0.7071067811865475, 0.7071067811865475, 0.03809523809523829},
     {0.5773502691896258, 0.5773502691896258, 0.5773502691896258, 0.0321428571428573}},
    // order 4: 38 points (degree 9)
    {{0.0, 0.0, 1.0, 0.00952380952380907},
     {0.5773502691896258, 0.5773502691896258, 0.5773502691896258, 0.0321428571428573},
     {0.0, 0.45970084338098427, 0.8880738339771146, 0.028571428571428636}},
    // order 5: 50 points (degree 11)
    {{0.0, 0.0, 1.0, 0.012698412698412223},
     {0.0, 0.7071067811865475, 0.7071067811865475, 0.022574955908289444},
     {0.5773502691896258, 0.5773502691896258, 0.5773502691896258, 0.021093750000000102},
     {0.30151134457776424, 0.30151134457776424, 0.9045340337332904, 0.02017333553791886}},
    // order 6: 74 points (degree 13)
    {{0.0, 0.0, 1.0, 0.000513067179731495},
     {0.0, 0.7071067811865475, 0.7071067811865475, 0.016604069565742573},
     {0.5773502691896258, 0.5773502691896258, 0.5773502691896258, -0.02958603896103527},
     {0.4803844614152578, 0.4803844614152578, 0.7337993857053474, 0.026576207082158427},
     {0.0, 0.3207726489807671, 0.947156221362591, 0.016522170993715835}},
    // order 7: 86 points (degree 15)
    {{0.0, 0.0, 1.0, 0.01154401154401075},
     {0.5773502691896258, 0.5773502691896258, 0.5773502691896258, 0.011943909085856397},
     {0.1890635528853951, 0.6943540066026664, 0.6943540066026664, 0.011876501294537375},
     {0.3696028464541496, 0.3696028464541496, 0.8525183117012681, 0.0111105557106034},
     {0.0, 0.37424303909033896, 0.9273306571511734, 0.011812303746904403}},
    // order 8: 110 points (degree 17)
    {{0.0, 0.0, 1.0, 0.003828270494933668},
     {0.5773502691896258, 0.5773502691896258, 0.5773502691896258, 0.009793737512487627},
     {0.1851156353447231, 0.1851156353447231, 0.9651240350865992, 0.00821173728319195},
     {0.39568947305593716, 0.39568947305593716, 0.8287699812525967, 0.009595471336071065},
     {0.21595729184585932, 0.6904210483822905, 0.6904210483822905, 0.009942814891177858},
     {0.0, 0.47836902881216736, 0.8781589106040568, 0.00969499636166317}},
    // order 9: 146 points (degree 19)
    {{0.0, 0.0, 1.0, 0.0005996313688613017},
     {0.0, 0.7071067811865475, 0.7071067811865475, 0.007372999718619262},
     {0.5773502691896258, 0.5773502691896258, 0.5773502691896258, 0.007210515360146086},
     {0.15746766720392918, 0.15746766720392918, 0.9748886436771664, 0.007574394159056108},
     {0.41749612279649856, 0.41749612279649856, 0.8070898183596309, 0.006753829486315507},
     {0.291298882209546, 0.6764410400114222, 0.6764410400114222, 0.007116355493118483},
     {0.14035538117128105, 0.4493328323269971, 0.8822700112603075, 0.0069910873533014575}},
    // order 10: 170 points (degree 21)
    {{0.0, 0.0, 1.0, 0.005544842902030009},
     {0.0, 0.7071067811865475, 0.7071067811865475, 0.00607133277067263},
     {0.5773502691896258, 0.5773502691896258, 0.5773502691896258, 0.0063836747735153895},
     {0.25512526211144787, 0.25512526211144787, 0.9326425903126717, 0.00518338758774642},
     {0.30079359513765364, 0.6743601460362872, 0.6743601460362872, 0.006317929009815409},
     {0.43189106967195323, 0.43189106967195323, 0.7917955593934788, 0.00620167000658926},
     {0.0, 0.2613931360334841, 0.9652324219764794, 0.005477143385138053},
     {0.1446630744324903, 0.49904531617954023, 0.8544158046846995, 0.005968383987680958}},
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

static std::unique_ptr<Resample> build_resample(int p, int pc, const ShTables &C, bool same) {
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
    return rs;
}

const Resample &resample_tables(int p, int pc) {
    static std::mutex mu;
    static std::map<std::pair<int, int>, std::unique_ptr<Resample>> cache;
    std::lock_guard<std::mutex> lock(mu);
    auto it = cache.find({p, pc});
    if (it != cache.end()) return *it->second;
    auto t = build_resample(p, pc, sh_tables(pc), pc == p);
    const Resample &ref = *t;
    cache[{p, pc}] = std::move(t);
    return ref;
}

const Resample &level_resample(int p, int pc) {
    static std::mutex mu;
    static std::map<std::pair<int, int>, std::unique_ptr<Resample>> cache;
    std::lock_guard<std::mutex> lock(mu);
    auto &t = cache[{p, pc}];
    if (!t) t = build_resample(p, pc, level_tables(pc), false);
    return *t;
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
