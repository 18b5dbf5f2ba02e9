// Device views and launch wrappers of the HIP kernels in kernels.hip.
#pragma once

#include "common.hpp"

namespace sphstk {

constexpr int kMaxOrder = 32;
constexpr int kMaxLevels = 6; // levels of a multi-level far field

// Read-only device view of one (possibly batched) operator's geometry.
// Spheres of one order, at most kTileSph of them (indices tile_sph[first ..
// first + count)), processed together by the tiled per-sphere matrix kernels.
constexpr int kTileSph = 16;
struct SphTile {
    int32_t p, first, count, pad;
};

struct DevGeom {
    int nsph = 0, nsusp = 0;
    int ntiles = 0;
    const SphTile *tiles = nullptr; // spheres grouped by order
    const int *tile_sph = nullptr;
    int64_t npts = 0;
    const double *pos = nullptr;   // 3N
    const double *rad = nullptr;   // N
    const double *quat = nullptr;  // 4N (w,x,y,z), unit
    const int *order = nullptr;    // N
    const int *sph_susp = nullptr; // N
    const int64_t *pt_off = nullptr;   // N+1
    const int64_t *coef_off = nullptr; // N+1 (6Q doubles per sphere)
    const int64_t *rec_off = nullptr;  // N+1 (2*kRecTracPad*tri(p+2) doubles per sphere with near neighbours)
    const double *coords = nullptr;    // 3P lab
    const double *norms = nullptr;     // 3P lab
    const double *w = nullptr;         // P
    const int64_t *near_off = nullptr; // N+1
    const int *near_src = nullptr;
    const int64_t *body_off = nullptr; // per tile: first element of its body-frame grid values (see body_cols)
    const int64_t *coef_body_off = nullptr; // per tile: first element of its coefficients in the same layout
};

// Chunks of the DOF vector used by the segmented BLAS-1 kernels.
struct Chunk {
    int64_t begin, end;
    int32_t seg, pad;
};

// Body-frame values of a tile: 3 values per point as matrix columns, padded to
// groups of 16, times 16 spheres (layout: transforms.hip).
__host__ __device__ inline int body_cols(int points) { return (3 * points + 15) & ~15; }

// A matrix per order in the layout of the transform GEMMs: nblk row blocks of
// 48 rows, ngrp groups of 16 columns (pack_gemm in engine.hip).
struct ShGemm {
    const void *tab[kMaxOrder + 1] = {}; // FP64, or FP32 (FP32 level sets)
    int nblk[kMaxOrder + 1] = {}, ngrp[kMaxOrder + 1] = {};
    int max_blk = 0;
};

// The levels of a multi-level far field as the transforms see them.  A sphere
// of order p has the points first[p][l] .. first[p][l + 1] - 1 of its stacked
// level points on level l, stored from off[l][S] on.
struct LevelViews {
    int nlev = 0;
    int first[kMaxOrder + 1][kMaxLevels + 1] = {};
    // levels on which spheres of order p keep their own grid (bits): these have no
    // stacked points; packing and gathering the fine grid serve them too
    unsigned own[kMaxOrder + 1] = {};
    const int64_t *off[kMaxLevels] = {};
    const double *w[kMaxLevels] = {};
    void *src[kMaxLevels] = {};              // source records (force words written per apply)
    const double *part[kMaxLevels] = {};     // partial-sum slots of the level's lists (level, then source cells)
    int nslot[kMaxLevels] = {};
    int64_t stride[kMaxLevels] = {};         // between slots
    const int64_t *body_off = nullptr;       // per tile: body-frame values of the stacked level points
};

// Partial sums of work lists: slot s of target t of target set k (of a joint list:
// the fine grid, then the levels) lies at base[k] + s stride[k] + 3 t.
struct SlotMap {
    int64_t base[1 + kMaxLevels] = {}, stride[1 + kMaxLevels] = {};
};

// source records (x, y, z, w*in, 0, 0) (in NULL: zero forces) and FP32 target records (x, n, 0, 0) of n points
void launch_pack_src_f64(int64_t n, const double *coords, const double *w, const double *in, double *src,
                         hipStream_t s);
void launch_pack_src_f32(int64_t n, const double *coords, const double *w, const double *in, float *src,
                         hipStream_t s);
void launch_pack_trg_f32(int64_t n, const double *coords, const double *norms, float *trg, hipStream_t s);

// far field (FP64: targets tcoords/tnorms, FP32: trg32 records):
// accumulate=1: out += coef * sum over the listed pairs;
// accumulate=0: slot k of out (slots) = coef * the sum over source slice k
void launch_far(int kind, int prec, int tpl, const void *src, const double *tcoords, const double *tnorms,
                const float *trg32, const SlotMap &slots, int ngroups, const int *group_order, const FarGroup *groups,
                const FarInterval *iv, const int *active, double *out, double coef, int accumulate, hipStream_t s,
                bool levels = false);

// Equivalent point forces of the far-field cells: the force words of eq
// (FP32 source records, K per cell) = rho_c P u_c (P 3K x 3Kc column-major, u_c
// the sum of nslot partial-sum slots of 3Kc check velocities per cell); cells
// of inactive suspensions are skipped.
void launch_equiv_forces(int ncell, int K, int Kc, const double *P, const double *u, int nslot, int64_t stride,
                         const double *rho, const int *susp, const int *active, float *eq, hipStream_t s);

// Transforms between grids and coefficients (transforms.hip).  pack_body: the
// body-frame values bd (FP64) and, if wanted, bf (FP32) of `in`, and the force words
// of the source records src64 / src32 (NULL: not wanted), on the fine grids and on
// the levels of L that are a sphere's own grid.
void launch_pack_body(const DevGeom &g, const double *in, double *bd, float *bf, double *src64, float *src32,
                      const LevelViews &L, int max_points, hipStream_t s);
// coef: per sphere; cbody: the same as GEMM columns (per tile)
void launch_analysis(const DevGeom &g, const ShGemm &M, const double *body, double *coef, double *cbody,
                     const int *active, hipStream_t s);
// out[mul dst_off[S] + 3 point + c] = coef R_S^rpow (M coefficients of S), lab frame: M a
// synthesis with per-degree blocks (a sphere's operator on its own surface)
void launch_synthesis(const DevGeom &g, const ShGemm &M, const double *cbody, const int64_t *dst_off, int mul,
                      double coef, int rpow, double *out, const int *active, hipStream_t s);
// Points of the levels of a set from their grids in the body frame: level l of order
// p has the n points (x, y, z, weight) from tab + 4 first on, grids[l (kMaxOrder + 1) + p]
// = (first, n).  Level l's points follow base[l] others in the set's coords, norms and
// src64 (FP64) or trg32 and src32 (FP32); w: the weights of all levels in a row.
struct LevelPoints {
    const double *tab = nullptr;
    const int2 *grids = nullptr;
    int64_t base[kMaxLevels] = {};
    double *w = nullptr, *coords = nullptr, *norms = nullptr, *src64 = nullptr;
    float *trg32 = nullptr, *src32 = nullptr;
};
void launch_level_points(const DevGeom &g, const LevelPoints &P, const LevelViews &L, hipStream_t s);
void launch_levels_down(const DevGeom &g, const ShGemm &M, bool fp64, const void *body, const LevelViews &L,
                        const int *active, hipStream_t s);
void launch_pack_levels(const DevGeom &g, bool fp64, const LevelViews &L, void *body, int max_points, hipStream_t s);
// out += the level fields on the fine grids
void launch_levels_up(const DevGeom &g, const ShGemm &M, bool fp64, const void *body, const LevelViews &L, double *out,
                      const int *active, hipStream_t s);
// mode 0: single-layer record (kRecSL arrays), 1: traction record (kRecTrac arrays)
// of the n spheres in list
void launch_expand(const DevGeom &g, int mode, const int *list, int n, const double *coef, double *rec,
                   const int *active, hipStream_t s, int max_order);
// One near evaluation work item: targets [tstart, tstart+tcount) (<= 128) of
// sphere trg against the expansion of sphere src; its contribution goes to
// scratch[slot ...] (3 doubles per target).
struct EvalItem {
    int32_t trg, src;
    int32_t tstart, tcount;
    int64_t slot;
};

// The same items grouped by source sphere: source S owns items
// [src_off[S], src_off[S + 1]).  The traction evaluation (mode 1) runs one
// workgroup per source with the source's record staged in LDS, one launch per
// sphere order (LDS sized to that order's record): srcs lists the spheres that
// have items by order, those of order p at [order_off[p], order_off[p + 1]).
struct SrcItems {
    const EvalItem *items = nullptr;
    const int64_t *src_off = nullptr;
    const int *srcs = nullptr;
    int order_off[kMaxOrder + 2] = {};
};

// Far-field sum on the fine grids as nslot partial-sum slots, stride apart.
struct FarSum {
    const double *part = nullptr;
    int nslot = 0;
    int64_t stride = 0;
};

// per-item near evaluations (mode 0: cSL single layer, 1: cTrac traction) into scratch
void launch_sheval_items(const DevGeom &g, int mode, const double *rec, const EvalItem *items, int nitems,
                         double *scratch, double cSL, double cTrac, const int *active, hipStream_t s,
                         const SrcItems *by_src = nullptr);
// per-target gather: out (+)= far sum (with that of the levels of L that are a
// sphere's own grid) + the target's items + cId in + cLOP L[in] (overwrite: out = ...,
// zero on inactive suspensions)
void launch_sheval_gather(const DevGeom &g, const int64_t *trg_slot_off, const int *trg_nsrc, const double *scratch,
                          const FarSum &far, const LevelViews &L, const double *in, double *out, double cId, double cLOP,
                          bool overwrite, const int *active, hipStream_t s);
void launch_identity(const DevGeom &g, const double *in, double *out, double cId, const int *active,
                     hipStream_t s);
void launch_lop(const DevGeom &g, const double *in, double *out, double cLOP, const int *active, hipStream_t s);
// segmented BLAS-1 over chunks (one segment per suspension)
void launch_seg_dot(const double *a, const double *b, const Chunk *chunks, int nchunks, double *partial,
                    const int *active, hipStream_t s);
// out[seg] = sum of partials of seg
void launch_seg_reduce(const double *partial, const int *seg_chunk_off, int nseg, double *out, const int *active,
                       hipStream_t s);
// y += sign * alpha[seg] * x
void launch_seg_axpy(double *y, const double *x, const double *alpha, double sign, const Chunk *chunks, int nchunks,
                     const int *active, hipStream_t s);
// y = alpha[seg] * x
void launch_seg_scale(double *y, const double *x, const double *alpha, const Chunk *chunks, int nchunks,
                      const int *active, hipStream_t s);
// modified Gram-Schmidt: h = (sums: added up from pprev, else) hprev, w -= h vprev (vprev NULL: not), then the
// chunk partials of w.v (v NULL: w.w); and w /= |w| from those of w.w, nv = |w|^2
void launch_seg_mgs(double *w, const double *vprev, const double *pprev, int sums, double *hprev, const double *v,
                    double *partial, const int *off, const Chunk *chunks, int nchunks, const int *active,
                    hipStream_t s);
void launch_seg_normalise(double *w, const double *partial, int sums, double *nv, const int *off, const Chunk *chunks,
                          int nchunks, const int *active, hipStream_t s);
// partial[j * nchunks + chunk] = w . V_j over the chunk, j < k <= 64 (one pass over w)
void launch_seg_multi_dot(const double *w, const double *V, int64_t ldv, int k, const Chunk *chunks, int nchunks,
                          double *partial, const int *active, hipStream_t s);
// out[j * nseg + seg] = sum of seg's chunk partials (op 2: negated), j < k
void launch_seg_multi_reduce(const double *partial, int nchunks, const int *off, int nseg, int k, double *out, int op,
                             const int *active, hipStream_t s);
// x += sum_i coef[i*nseg + seg] * V[i]   (i < k); norm (optional): chunk partials of x.x afterwards
void launch_seg_multi_axpy(double *x, const double *V, int64_t ldv, const double *coef, int k, int nseg,
                           const Chunk *chunks, int nchunks, const int *active, hipStream_t s,
                           double *norm = nullptr);
// x = sum_j coef[j nseg + seg] V_j over the active segments (x overwritten there)
void launch_seg_multi_comb(double *x, const double *V, int64_t ldv, const double *coef, int k, int nseg,
                           const Chunk *chunks, int nchunks, const int *active, hipStream_t s);
// GMRES least-squares bookkeeping on the device, one Krylov space per
// suspension (arrays: H B x (m+1) x m, cs/sn B x m, g B x (m+1), per-suspension
// ints and doubles of length B): cycle start (g = beta e_1, cur = cyc), the
// Givens update of column j from the orthogonalisation products hh (active set
// cur shrinks as suspensions converge; *nact = those still active), and the
// back substitution into coef[i B + s].
// residual coefficients of a finished cycle in its basis (m + 1 per suspension, coef[i B + s])
void launch_gmres_resid_coef(int B, int m, const double *g, const double *cs, const double *sn, const int *kdim,
                             const int *cyc, double *coef, hipStream_t s);
void launch_gmres_init(int B, int m, const double *beta, const int *cyc, double *g, int *cur, int *kdim, int *impok,
                       hipStream_t s);
void launch_gmres_givens(int B, int j, int m, const double *hh, double hsign, double *H, double *cs, double *sn,
                         double *g, const double *bn, double tol, int *cur, int *kdim, int *impok, double *relres,
                         int *nact, hipStream_t s);
void launch_gmres_backsub(int B, int m, const double *H, const double *g, const int *kdim, const int *cyc,
                          double *coef, hipStream_t s);
// out += sum of nslot partial-sum slots (far-field source slices)
void launch_slot_reduce(double *out, const double *part, int nslot, int64_t stride, const Chunk *chunks,
                        int nchunks, const int *active, hipStream_t s);
// y = a*x + b*y (plain, whole vector)
void launch_axpby(int64_t n, double a, const double *x, double b, double *y, hipStream_t s);
void launch_fill(int64_t n, double v, double *y, hipStream_t s);

// FP64 traction far field of ncol (1..8) densities on one geometry: `in` holds
// ncol DOF vectors col_stride apart, of which the first n0 points carry the
// geometry and work lists; src is scratch of 4 (ncol + 1) doubles per point;
// the slots (slot_stride apart) have the same column layout.  The work lists are
// those of kMultiTPL targets per lane.
constexpr int kMultiTPL = 2;
void launch_far_trac_multi(int ncol, int64_t n0, const double *coords, const double *norms, const double *w,
                           const double *in, int64_t col_stride, double *src, int ngroups, const int *go,
                           const FarGroup *gr, const FarInterval *iv, const int *active, int nsusp0, double *out,
                           double coef, int64_t slot_stride, hipStream_t s);
// sphere-centre far field (Faxen) of packed FP64 sources, 9 sums per centre and slot
// out (+)= coef K'[rho0] at grid points from distant spheres' rigid-body densities, in closed form (Stokeslet,
// degenerate quadrupole and rotlet at the centres); force holds (F, T) per sphere
void launch_far_rigid(const double *coords, const double *norms, const double *pos, const double *force,
                      const double *rad, int64_t ntrg, int ngroups, const int *go, const FarGroup *gr,
                      const FarInterval *iv, double *out, double coef, int acc, hipStream_t s);
void launch_far_centre(const double *src, const double *centres, int ngroups, const int *go, const FarGroup *gr,
                       const FarInterval *iv, double *part, int64_t ntrg, hipStream_t s);
void launch_centre_finish(int nsph, int nslot, const double *part, const double *rad, const double *vel_ns,
                          double inv_mu, double *vel, hipStream_t s);
void launch_rho0(const DevGeom &g, const double *force, double *rho, hipStream_t s);
void launch_rigid_avg(const DevGeom &g, const double *u, double inv_mu, double *vel, hipStream_t s);

} // namespace sphstk
