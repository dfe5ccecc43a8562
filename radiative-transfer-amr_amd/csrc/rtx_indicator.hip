// Error indicators of a nodal solution and the integrals hp steering reads.
//
// src/amr/Error_Indicator/error/error_angular_jump.py:14-99 (jumps of the
// angular traces between neighbouring cells of a column),
// error_spatial_jump.py:17-236 (jumps of the spatial face traces between
// neighbouring columns, projected onto a common node set) and the
// projection integrals of src/dg/projection/cell_intg_xy.py:13-36 and
// col_intg_th.py:13-37 that cell_hp_steer.py / col_hp_steer.py read.  The
// reference walks every cell in Python; here a wavefront owns a cell (angular
// jumps), or a workgroup a column and each of its wavefronts cells or face
// pairs of it; sums stay inside a wavefront until a last step over the
// workgroup's wavefronts, always in the same order.
#include <type_traits>

#include "rtx_internal.h"

namespace rtx {

constexpr int INM = RTX_NMAX;
constexpr int IWAVES = 8;
constexpr int ITHREADS = 64 * IWAVES;
constexpr int AWAVES = 4;           // cells per workgroup of the angular jumps

// w2[s] = wx_i wy_j of the column's nodes s = i ny + j, to LDS.
__device__ inline void node_weights(const DevMesh &m, int nx, int ny, double *w2) {
    const double *wx = m.lgl_w + nx * INM, *wy = m.lgl_w + ny * INM;
    for (int s = threadIdx.x; s < nx * ny; s += ITHREADS) w2[s] = wx[s / ny] * wy[s % ny];
    __syncthreads();
}

// Per cell: intg_xy[a] = (dx dy / 4) sum_ij wx_i wy_j u[i, j, a] at the
// cell's global angle index (cell_intg_xy.py:21-34), and, when norm2 is
// given, (dx dy / 4)(dth / 2) sum wx wy wth u^2.  Per column: intg_th[i, j] =
// sum over cells (dth / 2) sum_a wth_a u[i, j, a] (col_intg_th.py:22-35), at
// the column's spatial offset.
//
// Bound by reading u: a wavefront reads a cell's values in their order (lane
// = node group x angle), then once more from the cache with a lane per node.
// One launch; per-cell workgroups summing over nodes with one thread per
// angle, and a second launch of one thread per node and column, took 34 + 14
// us for 16,384 cells of 5 x 5 x 5 in 1,024 columns, this 12 us.
__global__ __launch_bounds__(ITHREADS) void k_moments(DevMesh m, const double *__restrict__ u,
                                                     double *__restrict__ intg_xy,
                                                     double *__restrict__ intg_th,
                                                     double *__restrict__ norm2) {
    __shared__ double w2[INM * INM], part[IWAVES][INM * INM];
    const int c = blockIdx.x, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nx = m.col_nx[c], ny = m.col_ny[c], nsp = nx * ny;
    const double dx = m.col_geom[4 * c + 2] - m.col_geom[4 * c + 0];
    const double dy = m.col_geom[4 * c + 3] - m.col_geom[4 * c + 1];
    node_weights(m, nx, ny, w2);
    const int k1 = m.col_cell_start[c + 1];
    double th[2] = {0.0, 0.0};                  // of nodes lane and lane + 64
    for (int k = m.col_cell_start[c] + wave; k < k1; k += IWAVES) {
        const int nt = m.cell_nth[k], G = 64 / nt;          // node groups
        const double dth = m.cell_geom[2 * k + 1] - m.cell_geom[2 * k + 0];
        const double *wt = m.lg_w + nt * INM, *uk = u + m.cell_dof_off[k];
        const int g = lane / nt, a = lane - g * nt;
        double sx = 0.0, s2 = 0.0;
        if (g < G)
            for (int s = g; s < nsp; s += G) {
                const double v = uk[s * nt + a], w = w2[s] * v;
                sx += w;
                s2 += w * v;
            }
        s2 *= g < G ? wt[a] : 0.0;
        // over the node groups (lanes of the same angle)
        for (int h = 32; h > 0; h >>= 1) {
            const double o = __shfl(sx, (lane + h * nt) & 63);
            if (g < h && g + h < G) sx += o;
        }
        if (lane < nt) intg_xy[m.col_ang_start[c] + m.cell_ang_off[k] + lane] = dx * dy / 4.0 * sx;
        if (norm2) {
            s2 = wave_sum(s2);
            if (lane == 0) norm2[k] = dx * dy / 4.0 * (dth / 2.0) * s2;
        }
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int s = lane + 64 * b;
            if (s >= nsp) continue;
            double t = 0.0;
            for (int e = 0; e < nt; ++e) t += wt[e] * uk[s * nt + e];
            th[b] += dth / 2.0 * t;
        }
    }
#pragma unroll
    for (int b = 0; b < 2; ++b)
        if (lane + 64 * b < nsp) part[wave][lane + 64 * b] = th[b];
    __syncthreads();
    for (int s = threadIdx.x; s < nsp; s += ITHREADS) {
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < IWAVES; ++w) t += part[w][s];
        intg_th[m.col_sp_off[c] + s] = t;
    }
}

// Per cell: traces at the bottom (theta pulled back to -1) and top (+1) of
// the cell and of its lower / upper neighbours in the column, and
// err[k] = (1/4) sum_ij wx_i wy_j (1/2)((bot_k - top_lo)^2 + (top_k - bot_up)^2)
// (error_angular_jump.py:36-81).  lend[(n 2 + s) INM + a] = l_a(2 s - 1) of
// the n-point Gauss-Legendre basis.
//
// Bound by reading u three times (a cell and its two neighbours, mostly from
// the cache).  A wavefront per cell of the mesh, a lane per node, so that
// columns of many cells fill the chip as well as many columns do:
// 16,384 cells of 5 x 5 x 5 in 1,024 columns 12 us, 1,024 cells of 10 x 10 x 10
// in 16 columns 7.8 us (a workgroup per column of cells took 12 and 57 us, a
// workgroup per cell 28 and 8.3 us).
__global__ __launch_bounds__(64 * AWAVES) void k_angular_jump(DevMesh m, const double *__restrict__ u,
                                                             const int32_t *__restrict__ nbr,
                                                             const double *__restrict__ lend,
                                                             double *__restrict__ err) {
    const int lane = threadIdx.x & 63;
    // workgroups go to the 8 XCDs round-robin; XCD j takes the j-th eighth of
    // the cells, so a cell's neighbours are read through the same L2
    const int blk = blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8;
    const int k = blk * AWAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (k >= m.ncell) return;
    const int c = m.cell_col[k];
    const int nx = m.col_nx[c], ny = m.col_ny[c], nsp = nx * ny;
    const int lo = nbr[2 * k], up = nbr[2 * k + 1];
    const int nt = m.cell_nth[k], ntl = m.cell_nth[lo], ntu = m.cell_nth[up];
    const double *uk = u + m.cell_dof_off[k], *ul = u + m.cell_dof_off[lo],
                 *uu = u + m.cell_dof_off[up];
    const double *bot_k = lend + (nt * 2 + 0) * INM, *top_k = lend + (nt * 2 + 1) * INM;
    const double *top_l = lend + (ntl * 2 + 1) * INM, *bot_u = lend + (ntu * 2 + 0) * INM;
    const double *wx = m.lgl_w + nx * INM, *wy = m.lgl_w + ny * INM;
    double acc = 0.0;
    // Q nodes per lane, side by side; past the last node that node again
    const auto nodes = [&](auto per_lane) {
        constexpr int Q = decltype(per_lane)::value;
        int at[Q];
        double b0[Q] = {}, t0[Q] = {}, tl[Q] = {}, bu[Q] = {};
#pragma unroll
        for (int q = 0; q < Q; ++q) at[q] = min(lane + 64 * q, nsp - 1);
        for (int a = 0; a < nt; ++a)
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const double v = uk[at[q] * nt + a];
                b0[q] += v * bot_k[a];
                t0[q] += v * top_k[a];
            }
        for (int a = 0; a < ntl; ++a)
#pragma unroll
            for (int q = 0; q < Q; ++q) tl[q] += ul[at[q] * ntl + a] * top_l[a];
        for (int a = 0; a < ntu; ++a)
#pragma unroll
            for (int q = 0; q < Q; ++q) bu[q] += uu[at[q] * ntu + a] * bot_u[a];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const double jl = (b0[q] - tl[q]) * (b0[q] - tl[q]), ju = (t0[q] - bu[q]) * (t0[q] - bu[q]);
            if (lane + 64 * q < nsp) acc += wx[at[q] / ny] * wy[at[q] % ny] * 0.5 * (jl + ju);
        }
    };
    static_assert(INM * INM <= 128, "two nodes per lane cover a column");
    if (nsp <= 64) nodes(std::integral_constant<int, 1>());
    else nodes(std::integral_constant<int, 2>());
    acc = wave_sum(acc);
    if (lane == 0) err[k] = 0.25 * acc;
}

// One side of a face pair, U[b][r] = sum_t psi[t][b] sum_a h[t][a] xsi[a][r],
// as two chained products: rows t, then rows b; columns r.  KS: K steps of
// four that cover n and nt.  Indices past the sizes read the last entry; h is
// zero there, and rows and columns past nB, nH are left out by the caller.
template <int KS>
__device__ inline mm_d4 jump_side(const double *h, int st, int n, int nt, const double *psi,
                                  int nB, const double *xsi, int nH, int l16, int lg) {
    double hv[KS], xv[KS], pv[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const int k = lg + 4 * s, a = min(k, nt - 1);
        hv[s] = keep_if(h[min(l16, n - 1) * st + a], l16 < n && k < nt);
        xv[s] = xsi[a * nH + min(l16, nH - 1)];
        pv[s] = psi[min(k, n - 1) * nB + min(l16, nB - 1)];
    }
    mm_d4 d = {0, 0, 0, 0}, e = d;
#pragma unroll
    for (int s = 0; s < KS; ++s) d = mma_f64(hv[s], xv[s], d);
#pragma unroll
    for (int s = 0; s < KS; ++s) e = mma_f64(pv[s], d[s], e);
    return e;
}

// Per column: the squared jumps of the face traces against every
// neighbouring cell across every face (error_spatial_jump.py:61-225).  Pair
// p (pairs of column c: col_pair_start[c] .. col_pair_start[c + 1] - 1) is
//   pair[RTX_JUMP_PAIR_INTS p + 0..8] = own cell, neighbour cell, face F,
//   nB, nH, and pool offsets of psi_0 (n0 x nB), psi_1 (n1 x nB),
//   xsi_0 (nth0 x nH), xsi_1 (nth1 x nH), row-major;
//   scale[p] = d_A dth_G / 4.
// The own trace is taken on face F, the neighbour's on the opposite face;
// both are projected onto nB LGL nodes x nH Gauss-Legendre nodes of the
// shared interval and col_err[c] = sum scale sum wB wH (U0 - U1)^2 /
// (perimeter 2 pi) (:227).
//
// Bound by gathered loads and latency: a pair is a chain of table reads and
// four short matrix chains.  A wavefront takes every IWAVES-th pair of its
// column, and its lanes read 64 of its pairs' tables at once; with a
// workgroup per pair and the products in LDS a column's pairs waited for each
// other.  1,024 columns of 5 x 5 nodes, 63,488 pairs: 243 -> 42 us.  (Keeping
// the projections in registers while pairs share them spills and holds 5
// wavefronts per SIMD instead of 8: 58 us.)
__global__ __launch_bounds__(ITHREADS) __attribute__((amdgpu_waves_per_eu(8)))
void k_spatial_jump(DevMesh m, const double *__restrict__ u,
                    const int32_t *__restrict__ col_pair_start, const int32_t *__restrict__ pair,
                    const double *__restrict__ scale, const double *__restrict__ pool,
                    double *__restrict__ col_err) {
    __shared__ double part[IWAVES];
    const int c = blockIdx.x, lane = threadIdx.x & 63, l16 = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int p1 = col_pair_start[c + 1];
    double acc = 0.0;
    for (int p0 = col_pair_start[c] + wave; p0 < p1; p0 += ITHREADS) {
        // lane l: the tables of pair p0 + l IWAVES
        int off0 = 0, off1 = 0, st = 0, dims = 0, q5 = 0, q6 = 0, q7 = 0, q8 = 0;
        double sc = 0.0;
        const int pl = p0 + lane * IWAVES;
        if (pl < p1) {
            const int32_t *q = pair + size_t(RTX_JUMP_PAIR_INTS) * pl;
            const int k0 = q[0], k1 = q[1], F = q[2], nB = q[3], nH = q[4];
            q5 = q[5];
            q6 = q[6];
            q7 = q[7];
            q8 = q[8];
            sc = scale[pl];
            const int c0 = m.cell_col[k0], c1 = m.cell_col[k1];
            const int nx0 = m.col_nx[c0], ny0 = m.col_ny[c0], nt0 = m.cell_nth[k0];
            const int nx1 = m.col_nx[c1], ny1 = m.col_ny[c1], nt1 = m.cell_nth[k1];
            const bool even = (F % 2) == 0;
            // own face: F = 0 -> i = nx - 1, 1 -> j = ny - 1, 2 -> i = 0, 3 ->
            // j = 0; the neighbour's is the opposite face
            off0 = m.cell_dof_off[k0] + (F == 0 ? (nx0 - 1) * ny0 * nt0 : F == 1 ? (ny0 - 1) * nt0 : 0);
            off1 = m.cell_dof_off[k1] + (F == 2 ? (nx1 - 1) * ny1 * nt1 : F == 3 ? (ny1 - 1) * nt1 : 0);
            st = (even ? nt0 : ny0 * nt0) | (even ? nt1 : ny1 * nt1) << 16;
            dims = (even ? ny0 : nx0) | (even ? ny1 : nx1) << 4 | nt0 << 8 | nt1 << 12 | nB << 16 |
                   nH << 20;
        }
        const int here = min(64, (p1 - p0 + IWAVES - 1) / IWAVES);
        for (int i = 0; i < here; ++i) {
            const auto at = [&](int v) { return __builtin_amdgcn_readlane(v, i); };
            const int d = at(dims), s2 = at(st);
            const int n0 = d & 15, n1 = (d >> 4) & 15, nt0 = (d >> 8) & 15, nt1 = (d >> 12) & 15;
            const int nB = (d >> 16) & 15, nH = (d >> 20) & 15;
            const double *h0 = u + at(off0), *h1 = u + at(off1);
            const double w = __hiloint2double(at(__double2hiint(sc)), at(__double2loint(sc)));
            const double *ps0 = pool + at(q5), *ps1 = pool + at(q6);
            const double *xs0 = pool + at(q7), *xs1 = pool + at(q8);
            const auto side = [&](auto ks) {
                constexpr int KS = decltype(ks)::value;
                const mm_d4 a = jump_side<KS>(h0, s2 & 0xffff, n0, nt0, ps0, nB, xs0, nH, l16, lg);
                const mm_d4 b = jump_side<KS>(h1, s2 >> 16, n1, nt1, ps1, nB, xs1, nH, l16, lg);
                const double wh = w * m.lg_w[nH * INM + min(l16, nH - 1)];
#pragma unroll
                for (int v = 0; v < KS; ++v) {
                    const int bq = lg + 4 * v;
                    const double wb = m.lgl_w[nB * INM + min(bq, nB - 1)];
                    const double df = bq < nB && l16 < nH ? a[v] - b[v] : 0.0;
                    acc += wb * wh * df * df;
                }
            };
            const int n = max(max(max(n0, n1), max(nt0, nt1)), nB);
            if (n <= 4) side(std::integral_constant<int, 1>());
            else if (n <= 8) side(std::integral_constant<int, 2>());
            else side(std::integral_constant<int, 3>());
        }
    }
    acc = wave_sum(acc);
    if (lane == 0) part[wave] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < IWAVES; ++w) t += part[w];
        const double dx = m.col_geom[4 * c + 2] - m.col_geom[4 * c + 0];
        const double dy = m.col_geom[4 * c + 3] - m.col_geom[4 * c + 1];
        const double perim = 2.0 * dx + 2.0 * dy;
        col_err[c] = t / (perim * 2.0 * 3.141592653589793);
    }
}

}  // namespace rtx

using namespace rtx;

namespace {
int check_cells(rtx_plan *p, const char *who) {
    RTX_CHECK(p->max_cell_ndof <= INM * INM * INM, "%s: cell too large", who);
    return RTX_OK;
}
}  // namespace

extern "C" int rtx_indicator_moments(rtx_plan *p, const double *d_u, double *d_intg_xy,
                                     double *d_intg_th, double *d_norm2, void *stream) {
    RTX_CHECK(p && d_u && d_intg_xy && d_intg_th, "rtx_indicator_moments: null argument");
    if (int rc = check_cells(p, "rtx_indicator_moments")) return rc;
    if (p->m.ncell == 0) return RTX_OK;
    const hipStream_t st = static_cast<hipStream_t>(stream);
    k_moments<<<p->m.ncol, ITHREADS, 0, st>>>(p->m, d_u, d_intg_xy, d_intg_th, d_norm2);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

extern "C" int rtx_error_angular_jump(rtx_plan *p, const double *d_u, const int32_t *d_nbr,
                                      const double *d_lend, double *d_cell_err, void *stream) {
    RTX_CHECK(p && d_u && d_nbr && d_lend && d_cell_err, "rtx_error_angular_jump: null argument");
    if (int rc = check_cells(p, "rtx_error_angular_jump")) return rc;
    if (p->m.ncell == 0) return RTX_OK;
    const int nblk = (p->m.ncell + AWAVES - 1) / AWAVES;
    k_angular_jump<<<(nblk + 7) / 8 * 8, 64 * AWAVES, 0, static_cast<hipStream_t>(stream)>>>(
        p->m, d_u, d_nbr, d_lend, d_cell_err);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

extern "C" int rtx_error_spatial_jump(rtx_plan *p, const double *d_u, const int32_t *d_col_pair_start,
                                      const int32_t *d_pair, const double *d_scale,
                                      const double *d_pool, double *d_col_err, void *stream) {
    RTX_CHECK(p && d_u && d_col_pair_start && d_pair && d_scale && d_pool && d_col_err,
              "rtx_error_spatial_jump: null argument");
    if (int rc = check_cells(p, "rtx_error_spatial_jump")) return rc;
    if (p->m.ncol == 0) return RTX_OK;
    k_spatial_jump<<<p->m.ncol, ITHREADS, 0, static_cast<hipStream_t>(stream)>>>(
        p->m, d_u, d_col_pair_start, d_pair, d_scale, d_pool, d_col_err);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}
