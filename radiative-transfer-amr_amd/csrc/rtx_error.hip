// L2 error of a nodal solution against values at more nodes, per cell.
//
// src/amr/Error_Indicator/error/error_analytic.py:102-137 interpolates each
// cell's nodal solution (nx, ny, nth) to nx + 3, ny + 3, nth + 3 nodes (LGL
// in space, Gauss-Legendre in angle) with a quintuple loop and sums
// (dx dy dth / 8) w_p w_q w_r (u - u_hr)^2 against the analytic solution;
// error_high_resolution.py:103-203 does the same against the nodal solution
// of a p-refined mesh (mx, my, mth nodes per cell, read per cell).  Here one
// wavefront per cell does the interpolation as three 1-D contractions in
// registers: angle and y on the matrix cores, x fused with the weighted
// squared difference.
#include "rtx_internal.h"

namespace rtx {

constexpr int ENM = RTX_NMAX;       // largest node count
constexpr int EMM = RTX_NMAX + 3;   // largest high-resolution node count
constexpr int EWAVES = 4;           // cells per workgroup

// What a cell's contractions share.
struct ErrCell {
    int nx, ny, nt, mx, my, mt;
    const double *u, *hr;                       // the cell's values
    const double *Px, *Py, *Pt, *wx, *wy, *wt;  // n x m matrices, m weights
};

// Sums over this lane's target nodes of w (u_hr - I u)^2 (and w u_hr^2), of the
// target x-planes p0, p0 + step, ..
// IM >= max(nx, ny, nt): loads without branches (indices past a size read its
// last entry, and u is zero there, so the rows and terms past the sizes are).
template <bool NODAL, int IM>
__device__ inline void error_cell(const ErrCell &c, int l16, int lg, int p0, int step, double &acc,
                                  double &acc2) {
    constexpr int KS = (IM + 3) / 4;            // K steps of four
    double pt[KS], py[KS], uv[IM][KS];
    const int r = min(l16, c.mt - 1), qr = min(l16, c.my - 1), jr = min(l16, c.ny - 1);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const int k = lg + 4 * s, at = min(k, c.nt - 1);
        pt[s] = c.Pt[at * c.mt + r];
        py[s] = c.Py[min(k, c.ny - 1) * c.my + qr];
#pragma unroll
        for (int i = 0; i < IM; ++i)
            uv[i][s] = keep_if(c.u[(min(i, c.nx - 1) * c.ny + jr) * c.nt + at],
                               l16 < c.ny && k < c.nt && i < c.nx);
    }
    // e[i] (q, r) = sum_j Py[j][q] sum_a u[i][j][a] Pt[a][r]
    mm_d4 e[IM];
#pragma unroll
    for (int i = 0; i < IM; ++i) {
        mm_d4 d = {0, 0, 0, 0};
        e[i] = d;
        if (i < c.nx) {                         // uniform
#pragma unroll
            for (int s = 0; s < KS; ++s) d = mma_f64(uv[i][s], pt[s], d);
#pragma unroll
            for (int s = 0; s < KS; ++s) e[i] = mma_f64(py[s], d[s], e[i]);
        }
    }
    double wq[4];
    int off[4];
    const double wr = c.wt[r];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int q = lg + 4 * v, qc = min(q, c.my - 1);
        wq[v] = keep_if(c.wy[qc] * wr, q < c.my && l16 < c.mt);
        off[v] = qc * c.mt + r;
    }
    double hv[4], hn[4];                        // one target x-plane ahead
    const auto hr_load = [&](int p, double (&o)[4]) {
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (4 * v < c.my) o[v] = c.hr[min(p, c.mx - 1) * c.my * c.mt + off[v]];
    };
    hr_load(p0, hv);
    for (int p = p0; p < c.mx; p += step) {
        hr_load(p + step, hn);
        double px[IM];
#pragma unroll
        for (int i = 0; i < IM; ++i) px[i] = c.Px[min(i, c.nx - 1) * c.mx + p];   // uniform
        const double wp = c.wx[p];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            if (4 * v >= c.my) continue;        // uniform
            const bool in = lg + 4 * v < c.my && l16 < c.mt;
            double s = 0.0;
#pragma unroll
            for (int i = 0; i < IM; ++i) s += px[i] * e[i][v];
            const double d = in ? hv[v] - s : 0.0, w = wp * wq[v];
            acc += w * d * d;
            if (NODAL) {
                const double h = in ? hv[v] : 0.0;
                acc2 += w * h * h;
            }
            hv[v] = hn[v];
        }
    }
}

// NODAL: target node counts from hr_dims[3 k + 0..2] and the (n, m) table
// at tab + (n (EMM + 1) + m) RTX_ERR_TAB_STRIDE; also hr_norm2[k] =
// (dx dy dth / 8) sum w_p w_q w_r u_hr^2.  Otherwise m = n + 3 and the table
// of n at tab + n RTX_ERR_TAB_STRIDE.
//
// Bound by reading u_hr (512 values of a cell of 5 x 5 x 5).  One wavefront
// per cell and no LDS: the workgroup of 256 threads with the three products
// in LDS spent the time on barriers and on index divisions.  16,384 such
// cells (84 MB): 122 -> 57 us.  (Px one plane ahead as well spills scalar
// registers: 3 us more.)
//
// WPC wavefronts per cell, 1 or EWAVES: each contracts the cell and takes every
// WPC-th of its target x-planes.
template <bool NODAL, int WPC>
__global__ __launch_bounds__(64 * EWAVES) __attribute__((amdgpu_waves_per_eu(4)))
void k_error_l2(DevMesh m, const double *__restrict__ uh, const double *__restrict__ u_hr,
                const int64_t *__restrict__ hr_off, const int32_t *__restrict__ hr_dims,
                const double *__restrict__ tab, double *__restrict__ cell_err,
                double *__restrict__ hr_norm2) {
    const int lane = threadIdx.x & 63, l16 = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int k = WPC == 1 ? blockIdx.x * EWAVES + wave : blockIdx.x;
    const int p0 = WPC == 1 ? 0 : wave;
    if (k >= m.ncell) return;
    const int c = m.cell_col[k];
    ErrCell e;
    e.nx = m.col_nx[c];
    e.ny = m.col_ny[c];
    e.nt = m.cell_nth[k];
    e.mx = NODAL ? hr_dims[3 * k + 0] : e.nx + 3;
    e.my = NODAL ? hr_dims[3 * k + 1] : e.ny + 3;
    e.mt = NODAL ? hr_dims[3 * k + 2] : e.nt + 3;
    auto tab_of = [&](int n, int mm) {
        return tab + (NODAL ? size_t(n) * (EMM + 1) + mm : size_t(n)) * RTX_ERR_TAB_STRIDE;
    };
    e.Px = tab_of(e.nx, e.mx);                            // LGL nx -> mx
    e.Py = tab_of(e.ny, e.my);                            // LGL ny -> my
    e.Pt = tab_of(e.nt, e.mt) + ENM * EMM;                // LG nt -> mt
    e.wx = e.Px + 2 * ENM * EMM;                          // LGL mx weights
    e.wy = e.Py + 2 * ENM * EMM;
    e.wt = tab_of(e.nt, e.mt) + 2 * ENM * EMM + EMM;      // LG mt weights
    e.u = uh + m.cell_dof_off[k];
    e.hr = u_hr + hr_off[k];
    double acc = 0.0, acc2 = 0.0;
    // the smallest of three unrolled sizes (one, two or three K steps)
    const int n = max(max(e.nx, e.ny), e.nt);
    if (n <= 4) error_cell<NODAL, 4>(e, l16, lg, p0, WPC, acc, acc2);
    else if (n <= 7) error_cell<NODAL, 7>(e, l16, lg, p0, WPC, acc, acc2);
    else error_cell<NODAL, ENM>(e, l16, lg, p0, WPC, acc, acc2);
    const double dx = m.col_geom[4 * c + 2] - m.col_geom[4 * c + 0];
    const double dy = m.col_geom[4 * c + 3] - m.col_geom[4 * c + 1];
    const double dth = m.cell_geom[2 * k + 1] - m.cell_geom[2 * k + 0];
    acc = wave_sum(acc);
    if (NODAL) acc2 = wave_sum(acc2);
    if constexpr (WPC > 1) {
        __shared__ double part[2][WPC];
        if (lane == 0) {
            part[0][wave] = acc;
            part[1][wave] = acc2;
        }
        __syncthreads();
        acc = acc2 = 0.0;
#pragma unroll
        for (int w = 0; w < WPC; ++w) {
            acc += part[0][w];
            acc2 += part[1][w];
        }
        if (wave != 0) return;
    }
    if (lane == 0) {
        cell_err[k] = dx * dy * dth / 8.0 * acc;
        if (NODAL) hr_norm2[k] = dx * dy * dth / 8.0 * acc2;
    }
}

// A cell's wavefronts wait for its values, so few cells are a chain of one
// wavefront's target planes: up to two cells per CU they are shared by EWAVES
// wavefronts.  256 cells of 5 x 5 x 5 8.4 -> 6.5 us, of 8 x 8 x 8 12.1 -> 8.8,
// 512 of 10 x 10 x 10 14.8 -> 13.0, of 5 x 5 x 5 8.4 either way; from 1,024 cells
// on (8.7, 13.1 and 16.1 us) one wavefront per cell fills the chip.
template <bool NODAL>
static int launch_error(const rtx_plan *p, const double *uh, const double *u_hr,
                        const int64_t *hr_off, const int32_t *hr_dims, const double *tab,
                        double *cell_err, double *hr_norm2, void *stream) {
    const hipStream_t st = static_cast<hipStream_t>(stream);
    const int ncell = p->m.ncell;
    if (ncell <= 2 * p->n_cu)
        k_error_l2<NODAL, EWAVES><<<ncell, 64 * EWAVES, 0, st>>>(p->m, uh, u_hr, hr_off, hr_dims,
                                                                 tab, cell_err, hr_norm2);
    else
        k_error_l2<NODAL, 1><<<(ncell + EWAVES - 1) / EWAVES, 64 * EWAVES, 0, st>>>(
            p->m, uh, u_hr, hr_off, hr_dims, tab, cell_err, hr_norm2);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

}  // namespace rtx

using namespace rtx;

extern "C" int rtx_error_l2(rtx_plan *p, const double *d_uh, const double *d_u_hr,
                            const int64_t *d_hr_off, const double *d_tab, double *d_cell_err,
                            void *stream) {
    RTX_CHECK(p && d_uh && d_u_hr && d_hr_off && d_tab && d_cell_err,
              "rtx_error_l2: null argument");
    RTX_CHECK(p->max_cell_ndof <= ENM * ENM * ENM, "rtx_error_l2: cell too large");
    if (p->m.ncell == 0) return RTX_OK;
    return launch_error<false>(p, d_uh, d_u_hr, d_hr_off, nullptr, d_tab, d_cell_err, nullptr,
                               stream);
}

extern "C" int rtx_error_l2_nodal(rtx_plan *p, const double *d_uh, const double *d_u_hr,
                                  const int64_t *d_hr_off, const int32_t *d_hr_dims,
                                  const double *d_tab, double *d_cell_err, double *d_hr_norm2,
                                  void *stream) {
    RTX_CHECK(p && d_uh && d_u_hr && d_hr_off && d_hr_dims && d_tab && d_cell_err && d_hr_norm2,
              "rtx_error_l2_nodal: null argument");
    RTX_CHECK(p->max_cell_ndof <= ENM * ENM * ENM, "rtx_error_l2_nodal: cell too large");
    if (p->m.ncell == 0) return RTX_OK;
    return launch_error<true>(p, d_uh, d_u_hr, d_hr_off, d_hr_dims, d_tab, d_cell_err, d_hr_norm2,
                              stream);
}
