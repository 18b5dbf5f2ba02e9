// Per-sphere matrices on body-frame grid values, as GEMMs on the matrix cores
// (the spheres of one order are the columns), and the packing passes that
// bring their operands into the layout of the matrix instructions:
//   analysis     coef[S] = A_p q_S^-1 in_S                  (Shexp::calcSpectralCoeff, Sphere/Shexp.cpp:408-447)
//   level down   level sources of S = w q_S D_p q_S^-1 in_S (D_p: all levels' resampling matrices, stacked by rows)
//   level up     out_S += q_S U_p q_S^-1 levels_S           (U_p: the same, stacked by columns)
//   synthesis    out_S = q_S Y_p coef[S]                    (Y_p: with per-degree blocks, the operators of a sphere on
//                                                            its own surface, Sphere/Shexp.cpp:503-624)
//
// A workgroup computes 48 matrix rows (16 points x 3 components, or 48
// coefficients) for one tile of 16 spheres; its four waves split the columns
// and add up through LDS.  Both operands stream from memory in the order the
// lanes consume them (one 16- or 32-byte load per lane and 16 columns), with no
// staging and no barrier inside the loop.  What bounds it: the FP32 matrix rate
// where there are many spheres, latency below (this is why the columns are
// split over waves: 100 spheres of order 8 are 7 tiles).  Before, a launch per
// level and direction staged its input through LDS for 192 rows at a time (at
// most 7 x 3 workgroups at 100 spheres): whole mixed solves of 100 spheres p=8
// went from 36.7 to 13.1 ms, of 1024 p=12 from 119.9 to 82.5 ms, of 500 p=16
// from 143.9 to 113.3 ms, with the far field's slots, the identity and the
// rigid-body projector added up in one pass (k_sheval_gather).
#include "kernels.hpp"

namespace sphstk {

namespace {

typedef double dbl4 __attribute__((ext_vector_type(4)));
typedef float flt4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ dbl4 mfma16x16x4(double a, double b, dbl4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ flt4 mfma16x16x4(float a, float b, flt4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ void rotate(const double *q, double s, const double v[3], double o[3]) {
    const double w = q[0], ux = s * q[1], uy = s * q[2], uz = s * q[3];
    const double tx = 2.0 * (uy * v[2] - uz * v[1]);
    const double ty = 2.0 * (uz * v[0] - ux * v[2]);
    const double tz = 2.0 * (ux * v[1] - uy * v[0]);
    o[0] = v[0] + w * tx + (uy * tz - uz * ty);
    o[1] = v[1] + w * ty + (uz * tx - ux * tz);
    o[2] = v[2] + w * tz + (ux * ty - uy * tx);
}

// Element of column `col` (of a tile's body-frame values) and sphere t: 16
// columns per group, four consecutive columns per lane.
__device__ __forceinline__ int64_t body_at(int col, int t) {
    return ((int64_t)(col >> 4) * 64 + ((col >> 2) & 3) * 16 + t) * 4 + (col & 3);
}

// Grid values of every sphere, rotated to its body frame, as GEMM columns
// (zero for absent spheres and padding columns), and the force words w f of the
// far field's source records (whose positions were set at set-up).
template <bool F>
__global__ __launch_bounds__(256) void k_pack_body(DevGeom g, const double *__restrict__ in, double *__restrict__ bd,
                                                   float *__restrict__ bf, double *__restrict__ src64,
                                                   float *__restrict__ src32, LevelViews L) {
    const SphTile Ti = g.tiles[blockIdx.y];
    const int n = (Ti.p + 1) * (2 * Ti.p + 2), cols = body_cols(n);
    const int e = blockIdx.x * blockDim.x + threadIdx.x, t = e & 15, k = e >> 4;
    if (3 * k >= cols) return;
    double o[3] = {0.0, 0.0, 0.0};
    if (t < Ti.count && k < n) {
        const int S = g.tile_sph[Ti.first + t];
        const int64_t i = g.pt_off[S] + k;
        const double v[3] = {in[3 * i], in[3 * i + 1], in[3 * i + 2]};
        rotate(g.quat + 4 * S, -1.0, v, o);
        const double wi = g.w[i];
        if (src64)
            for (int c = 0; c < 3; c++) src64[8 * i + 3 + c] = wi * v[c];
        if (src32)
            for (int c = 0; c < 3; c++) src32[8 * i + 3 + c] = (float)(wi * v[c]);
        const unsigned own = L.own[Ti.p];
        for (int l = 0; own >> l; l++)
            if (own >> l & 1) {
                const int64_t q = 8 * (L.off[l][S] + k) + 3;
                if (src64)
                    for (int c = 0; c < 3; c++) static_cast<double *>(L.src[l])[q + c] = wi * v[c];
                if (src32)
                    for (int c = 0; c < 3; c++) static_cast<float *>(L.src[l])[q + c] = (float)(wi * v[c]);
            }
    }
    const int64_t base = g.body_off[blockIdx.y];
    for (int c = 0; c < 3; c++)
        if (3 * k + c < cols) {
            const int64_t a = base + body_at(3 * k + c, t);
            bd[a] = o[c];
            if (F) bf[a] = (float)o[c];
        }
}

// One workgroup per sphere and level; bound by its writes (232 bytes a point, FP64).
// Points and records made on the host, one sphere after the other, and sent over took
// most of a set's build: FP64 set of 48 suspensions of orders 6 to 16 (1.2e6 points)
// 0.19 -> 0.06 s, of 1024 spheres p=12 0.068 -> 0.040 s, both with the identity
// matrices of own-grid levels gone as well.
template <bool FP64>
__global__ __launch_bounds__(128) void k_level_points(DevGeom g, LevelPoints P, LevelViews L) {
    const int S = blockIdx.x, l = blockIdx.y;
    const int2 gr = P.grids[l * (kMaxOrder + 1) + g.order[S]];
    const double R = g.rad[S];
    const double q[4] = {g.quat[4 * S], g.quat[4 * S + 1], g.quat[4 * S + 2], g.quat[4 * S + 3]};
    for (int k = threadIdx.x; k < gr.y; k += blockDim.x) {
        const double *e = P.tab + 4 * ((int64_t)gr.x + k);
        const int64_t i = P.base[l] + L.off[l][S] + k;
        double nv[3];
        rotate(q, 1.0, e, nv);
        P.w[i - P.base[0]] = R * R * e[3];
        for (int c = 0; c < 3; c++) {
            const double x = g.pos[3 * S + c] + R * nv[c];
            if (FP64) {
                P.coords[3 * i + c] = x;
                P.norms[3 * i + c] = nv[c];
                P.src64[8 * i + c] = x;
                P.src64[8 * i + 3 + c] = 0.0;
            } else {
                P.trg32[8 * i + c] = P.src32[8 * i + c] = (float)x;
                P.trg32[8 * i + 3 + c] = (float)nv[c];
                P.src32[8 * i + 3 + c] = 0.f;
            }
        }
        for (int c = 6; c < 8; c++) {
            if (FP64)
                P.src64[8 * i + c] = 0.0;
            else
                P.trg32[8 * i + c] = P.src32[8 * i + c] = 0.f;
        }
    }
}

// The level fields of every sphere (each the sum of its far-field lists'
// partial-sum slots), rotated to the body frame, as GEMM columns.
template <typename T>
__global__ __launch_bounds__(256) void k_pack_levels(DevGeom g, LevelViews L, T *__restrict__ body) {
    const SphTile Ti = g.tiles[blockIdx.y];
    const int *first = L.first[Ti.p];
    const int n = first[L.nlev], cols = body_cols(n);
    const int e = blockIdx.x * blockDim.x + threadIdx.x, t = e & 15, k = e >> 4;
    if (3 * k >= cols) return;
    double o[3] = {0.0, 0.0, 0.0};
    if (t < Ti.count && k < n) {
        const int S = g.tile_sph[Ti.first + t];
        int l = 0;
        while (k >= first[l + 1]) l++;
        const int64_t i = 3 * (L.off[l][S] + k - first[l]);
        double v[3] = {0.0, 0.0, 0.0};
        const double *part = L.part[l] + i;
        for (int s = 0; s < L.nslot[l]; s++, part += L.stride[l])
            for (int c = 0; c < 3; c++) v[c] += part[c];
        rotate(g.quat + 4 * S, -1.0, v, o);
    }
    const int64_t base = L.body_off[blockIdx.y];
    for (int c = 0; c < 3; c++)
        if (3 * k + c < cols) body[base + body_at(3 * k + c, t)] = (T)o[c];
}

enum { ANALYSIS, LEVEL_DOWN, LEVEL_UP, SYNTHESIS };

struct SynthOut {
    const int64_t *off;
    int mul, rpow;
    double coef;
};

// blockIdx.x: row block of 48, blockIdx.y: tile.  Operands of the 16x16x4
// instructions: A[i][k] in lane i + 16k, B[k][j] in lane j + 16k; D[i][j] in lane
// j + 16 (i / 4), element i % 4 (FP32) or lane j + 16 (i % 4), element i / 4
// (FP64).  Row block `w` holds rows 3 (16 w + i) + rb of the resampling matrices
// (so that a lane ends up with the three components of a point) and rows
// 48 w + 16 rb + i of the analysis.
template <typename T, int KIND>
__global__ __launch_bounds__(256) void k_sh_gemm(DevGeom g, ShGemm M, const int64_t *__restrict__ body_off,
                                                 const T *__restrict__ body, LevelViews L, SynthOut Y,
                                                 double *__restrict__ out, double *__restrict__ cbody,
                                                 const int *__restrict__ active) {
    typedef T T4 __attribute__((ext_vector_type(4)));
    __shared__ T red[4][12][64];
    const SphTile Ti = g.tiles[blockIdx.y];
    const int p = Ti.p, w = blockIdx.x;
    if (w >= M.nblk[p]) return;
    const int G = M.ngrp[p];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const T4 *A = reinterpret_cast<const T4 *>(M.tab[p]) + (int64_t)w * 3 * G * 64 + lane;
    const T4 *B = reinterpret_cast<const T4 *>(body + body_off[blockIdx.y]) + lane;
    T4 acc[3];
#pragma unroll
    for (int rb = 0; rb < 3; rb++) acc[rb] = T4{T(0), T(0), T(0), T(0)};
    const int g1 = G * (wv + 1) / 4;
#pragma unroll 4
    for (int k = G * wv / 4; k < g1; k++) {
        const T4 b = B[k * 64];
        T4 a[3];
#pragma unroll
        for (int rb = 0; rb < 3; rb++) a[rb] = A[(rb * G + k) * 64];
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int rb = 0; rb < 3; rb++) acc[rb] = mfma16x16x4(a[rb][s], b[s], acc[rb]);
    }
#pragma unroll
    for (int rb = 0; rb < 3; rb++)
#pragma unroll
        for (int q = 0; q < 4; q++) red[wv][4 * rb + q][lane] = acc[rb][q];
    __syncthreads();
    // one thread per (row i of the blocks, sphere t)
    const int t = lane & 15, kq = lane >> 4, q = wv;
    if (t >= Ti.count) return;
    const int S = g.tile_sph[Ti.first + t];
    if (active && !active[g.sph_susp[S]]) return;
    const int i = sizeof(T) == 8 ? kq + 4 * q : 4 * kq + q;
    double v[3];
#pragma unroll
    for (int rb = 0; rb < 3; rb++)
        v[rb] = (double)((red[0][4 * rb + q][lane] + red[1][4 * rb + q][lane]) +
                         (red[2][4 * rb + q][lane] + red[3][4 * rb + q][lane]));
    if (KIND == ANALYSIS) {
        const int rows = 3 * (p + 1) * (p + 2);
        for (int rb = 0; rb < 3; rb++) {
            const int r = 48 * w + 16 * rb + i;
            if (r < rows) {
                out[g.coef_off[S] + r] = v[rb];
                cbody[g.coef_body_off[blockIdx.y] + body_at(r, t)] = v[rb];
            }
        }
        return;
    }
    const int j = 16 * w + i;
    double o[3];
    rotate(g.quat + 4 * S, 1.0, v, o);
    if (KIND == LEVEL_UP) {
        if (j >= (p + 1) * (2 * p + 2)) return;
        double *dst = out + 3 * (g.pt_off[S] + j);
        for (int c = 0; c < 3; c++) dst[c] += o[c];
        return;
    }
    if (KIND == SYNTHESIS) {
        if (j >= (p + 1) * (2 * p + 2)) return;
        const double f = Y.rpow ? Y.coef * g.rad[S] : Y.coef;
        double *dst = out + Y.mul * Y.off[S] + 3 * j;
        for (int c = 0; c < 3; c++) dst[c] = f * o[c];
        return;
    }
    const int *first = L.first[p];
    if (j >= first[L.nlev]) return;
    int l = 0;
    while (j >= first[l + 1]) l++;
    const int64_t k = L.off[l][S] + j - first[l];
    const double wk = L.w[l][k];
    T *src = reinterpret_cast<T *>(L.src[l]) + 8 * k + 3;
    for (int c = 0; c < 3; c++) src[c] = (T)(wk * o[c]);
}

dim3 pack_grid(const DevGeom &g, int max_points) {
    return dim3((unsigned)((16 * (body_cols(max_points) / 3 + 1) + 255) / 256), (unsigned)g.ntiles);
}

} // namespace

void launch_pack_body(const DevGeom &g, const double *in, double *bd, float *bf, double *src64, float *src32,
                      const LevelViews &L, int max_points, hipStream_t s) {
    if (!g.nsph || !g.ntiles) return;
    const dim3 grid = pack_grid(g, max_points);
    if (bf)
        k_pack_body<true><<<grid, dim3(256), 0, s>>>(g, in, bd, bf, src64, src32, L);
    else
        k_pack_body<false><<<grid, dim3(256), 0, s>>>(g, in, bd, bf, src64, src32, L);
}

void launch_level_points(const DevGeom &g, const LevelPoints &P, const LevelViews &L, hipStream_t s) {
    if (!g.nsph || !L.nlev) return;
    const dim3 grid((unsigned)g.nsph, (unsigned)L.nlev);
    if (P.coords)
        k_level_points<true><<<grid, dim3(128), 0, s>>>(g, P, L);
    else
        k_level_points<false><<<grid, dim3(128), 0, s>>>(g, P, L);
}

void launch_analysis(const DevGeom &g, const ShGemm &M, const double *body, double *coef, double *cbody,
                     const int *active, hipStream_t s) {
    if (!g.nsph || !g.ntiles) return;
    k_sh_gemm<double, ANALYSIS><<<dim3(M.max_blk, g.ntiles), dim3(256), 0, s>>>(g, M, g.body_off, body, LevelViews{},
                                                                               SynthOut{}, coef, cbody, active);
}

void launch_synthesis(const DevGeom &g, const ShGemm &M, const double *cbody, const int64_t *dst_off, int mul,
                      double coef, int rpow, double *out, const int *active, hipStream_t s) {
    if (!g.nsph || !g.ntiles) return;
    k_sh_gemm<double, SYNTHESIS><<<dim3(M.max_blk, g.ntiles), dim3(256), 0, s>>>(
        g, M, g.coef_body_off, cbody, LevelViews{}, SynthOut{dst_off, mul, rpow, coef}, out, nullptr, active);
}

void launch_levels_down(const DevGeom &g, const ShGemm &M, bool fp64, const void *body, const LevelViews &L,
                        const int *active, hipStream_t s) {
    if (!g.nsph || !g.ntiles || !M.max_blk) return;
    const dim3 grid(M.max_blk, g.ntiles);
    if (fp64)
        k_sh_gemm<double, LEVEL_DOWN><<<grid, dim3(256), 0, s>>>(g, M, g.body_off, (const double *)body, L, SynthOut{},
                                                                nullptr, nullptr, active);
    else
        k_sh_gemm<float, LEVEL_DOWN><<<grid, dim3(256), 0, s>>>(g, M, g.body_off, (const float *)body, L, SynthOut{},
                                                               nullptr, nullptr, active);
}

void launch_pack_levels(const DevGeom &g, bool fp64, const LevelViews &L, void *body, int max_points, hipStream_t s) {
    if (!g.nsph || !g.ntiles || !max_points) return;
    const dim3 grid = pack_grid(g, max_points);
    if (fp64)
        k_pack_levels<double><<<grid, dim3(256), 0, s>>>(g, L, (double *)body);
    else
        k_pack_levels<float><<<grid, dim3(256), 0, s>>>(g, L, (float *)body);
}

void launch_levels_up(const DevGeom &g, const ShGemm &M, bool fp64, const void *body, const LevelViews &L, double *out,
                      const int *active, hipStream_t s) {
    if (!g.nsph || !g.ntiles || !M.max_blk) return;
    const dim3 grid(M.max_blk, g.ntiles);
    if (fp64)
        k_sh_gemm<double, LEVEL_UP><<<grid, dim3(256), 0, s>>>(g, M, L.body_off, (const double *)body, L, SynthOut{}, out,
                                                              nullptr, active);
    else
        k_sh_gemm<float, LEVEL_UP><<<grid, dim3(256), 0, s>>>(g, M, L.body_off, (const float *)body, L, SynthOut{}, out,
                                                             nullptr, active);
}

} // namespace sphstk
