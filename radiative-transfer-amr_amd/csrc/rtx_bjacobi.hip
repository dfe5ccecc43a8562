// Per-cell block-Jacobi preconditioner.
//
// The reference solves with PETSc bjacobi (src/rt/solve.py:93-95; one block
// per MPI rank with an ILU(0) sub-solver) and computes, but discards, a dense
// inverse of each column block (src/rt/preconditioner_matrix.py:259-262).
// Here the blocks are the angular cells: the cell's diagonal block of the
// interior system A_II (mass, interior convection, outflow faces, in-cell
// scattering and any self-coupling link), identity on inflow-boundary DOFs.
//
// Build: one workgroup per block assembles it from its structure (per-node
// angular scattering blocks, the diagonal, the x/y derivative lines), inverts
// it by Gauss-Jordan with partial pivoting (blocked, in registers with matrix
// instructions, for blocks of up to 128 DOFs; in LDS or a global scratch block
// otherwise), and stores the inverse column-major so the apply is a coalesced
// batched GEMV.
#include <algorithm>
#include <type_traits>

#include "rtx_internal.h"

namespace rtx {

constexpr int NMq = RTX_NMAX;
constexpr int BJ_THREADS = 256;
#ifndef BJ_APPLY8_THREADS
#define BJ_APPLY8_THREADS 256    // threads per block of the FP8 apply
#endif
#ifndef BJ_APPLY16_THREADS
#define BJ_APPLY16_THREADS 512   // threads per block of the packed BF16 apply (measured
                                 // best of 128, 256, 512, 1024 on 125-DOF blocks)
#endif
constexpr int BJ_COLS = 128;     // column threads in the elimination
constexpr int BJ_SPLIT = 128;    // larger cells are split into groups of angles

__device__ inline bool bj_on_bdry(int bd, int i, int j, int nx, int ny) {
    return ((bd & 1) && i == nx - 1) || ((bd & 2) && j == ny - 1) || ((bd & 4) && i == 0) ||
           ((bd & 8) && j == 0);
}

// Assemble the cell's diagonal block into row-major A (n x n).
__device__ void bj_assemble(const DevMesh &m, int k, int restrict_, double *A, const double *cth,
                            const double *sth) {
    const int tid = threadIdx.x;
    const int c = m.cell_col[k];
    const int nx = m.col_nx[c], ny = m.col_ny[c], nth = m.cell_nth[k];
    const int n = nx * ny * nth, nyt = ny * nth, nsp = nx * ny;
    const double dx = m.col_geom[4 * c + 2] - m.col_geom[4 * c + 0];
    const double dy = m.col_geom[4 * c + 3] - m.col_geom[4 * c + 1];
    const double th0 = m.cell_geom[2 * k], dth = m.cell_geom[2 * k + 1] - th0;
    const double *wx = m.lgl_w + nx * NMq, *wy = m.lgl_w + ny * NMq, *wt = m.lg_w + nth * NMq;
    const double *Dx = m.lgl_D + size_t(nx) * NMq * NMq, *Dy = m.lgl_D + size_t(ny) * NMq * NMq;
    const int ao = m.cell_ang_off[k], na = m.col_nang[c];
    const double *G = m.G + m.col_G_off[c];
    const double *kap = m.kappa + m.col_sp_off[c], *sig = m.sigma + m.col_sp_off[c];
    for (int e = tid; e < n * n; e += BJ_THREADS) A[e] = 0.0;
    __syncthreads();
    // in-cell scattering: row (s, r), column (s, a)
    for (int e = tid; e < nsp * nth * nth; e += BJ_THREADS) {
        const int s = e / (nth * nth), r = (e / nth) % nth, a = e % nth;
        const int p = s / ny, q = s % ny;
        A[size_t(s * nth + r) * n + s * nth + a] =
            -dx * dy * wx[p] * wy[q] * sig[s] * G[size_t(ao + a) * na + ao + r];
    }
    __syncthreads();
    // mass and outflow faces on the diagonal
    const int quad = m.cell_quad[k];
    for (int t = tid; t < n; t += BJ_THREADS) {
        const int p = t / nyt, q = (t / nth) % ny, r = t % nth;
        double v = (dx * dy * dth * 0.125) * wx[p] * wy[q] * wt[r] * kap[p * ny + q];
        if (quad >= 0)
            for (int h = 0; h < 2; ++h) {
                const int F = (quad + h) & 3;
                const bool on = (F == 0 && p == nx - 1) || (F == 2 && p == 0) ||
                                (F == 1 && q == ny - 1) || (F == 3 && q == 0);
                if (on) {
                    const double tf = F == 0 ? cth[r] : (F == 1 ? sth[r] : (F == 2 ? -cth[r] : -sth[r]));
                    v += ((F & 1) ? dx : dy) * dth * 0.25 * ((F & 1) ? wx[p] : wy[q]) * wt[r] * tf;
                }
            }
        A[size_t(t) * n + t] += v;
    }
    __syncthreads();
    // -IC, x-derivative: row (p, q, r), column (i, q, r)
    for (int e = tid; e < n * nx; e += BJ_THREADS) {
        const int t = e / nx, i = e % nx;
        const int p = t / nyt, q = (t / nth) % ny, r = t % nth;
        A[size_t(t) * n + i * nyt + q * nth + r] -=
            (dy * dth * 0.25) * wy[q] * wt[r] * cth[r] * wx[i] * Dx[p * NMq + i];
    }
    __syncthreads();
    // -IC, y-derivative: row (p, q, r), column (p, j, r)
    for (int e = tid; e < n * ny; e += BJ_THREADS) {
        const int t = e / ny, j = e % ny;
        const int p = t / nyt, q = (t / nth) % ny, r = t % nth;
        A[size_t(t) * n + p * nyt + j * nth + r] -=
            (dx * dth * 0.25) * wx[p] * wt[r] * sth[r] * wy[j] * Dy[q * NMq + j];
    }
    __syncthreads();
    // a cell coupled to itself through a periodic face
    for (int l = m.link_start[k]; l < m.link_start[k + 1]; ++l) {
        if (m.link_src[l] != k) continue;
        const int F = m.link_face[l];
        const int n0 = (F & 1) ? nx : ny;
        const double cf = ((F & 1) ? dx : dy) * dth * 0.25;
        const double *Es = m.Es_pool + m.link_Es_off[l];
        const double *Et = m.Eth_pool + m.link_Eth_off[l];
        for (int e = tid; e < n0 * nth * n0 * nth; e += BJ_THREADS) {
            const int m0 = e / (nth * n0 * nth), r = (e / (n0 * nth)) % nth;
            const int m1 = (e / nth) % n0, a = e % nth;
            int row, col;
            if (F == 0) { row = (nx - 1) * nyt + m0 * nth + r; col = m1 * nth + a; }
            else if (F == 2) { row = m0 * nth + r; col = (nx - 1) * nyt + m1 * nth + a; }
            else if (F == 1) { row = m0 * nyt + (ny - 1) * nth + r; col = m1 * nyt + a; }
            else { row = m0 * nyt + r; col = m1 * nyt + (ny - 1) * nth + a; }
            A[size_t(row) * n + col] += cf * Es[m1 * n0 + m0] * Et[a * nth + r];
        }
        __syncthreads();
    }
    // identity rows/columns on inflow-boundary DOFs
    const int bd = restrict_ ? m.cell_bdry[k] : 0;
    if (bd) {
        for (int e = tid; e < n * n; e += BJ_THREADS) {
            const int row = e / n, col = e % n;
            const bool rb = bj_on_bdry(bd, row / nyt, (row / nth) % ny, nx, ny);
            const bool cb = bj_on_bdry(bd, col / nyt, (col / nth) % ny, nx, ny);
            if (rb || cb) A[e] = (row == col) ? 1.0 : 0.0;
        }
        __syncthreads();
    }
}

// In-place Gauss-Jordan inversion with partial pivoting of row-major A.
// Returns false on a zero pivot.  colk: n doubles of LDS.
__device__ bool bj_invert(double *A, int n, double *colk, int *perm, int *piv_row) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int k = 0; k < n; ++k) {
        if (wave == 0) {
            double best = -1.0;
            int bi = k;
            for (int i = k + lane; i < n; i += 64) {
                const double v = fabs(A[size_t(i) * n + k]);
                if (v > best) { best = v; bi = i; }
            }
            for (int o = 32; o > 0; o >>= 1) {
                const double ov = __shfl_xor(best, o);
                const int oi = __shfl_xor(bi, o);
                if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
            }
            if (lane == 0) {
                *piv_row = (best > 0.0) ? bi : -1;
                perm[k] = bi;
            }
        }
        __syncthreads();
        const int pr = *piv_row;
        if (pr < 0) return false;
        if (pr != k)
            for (int c = tid; c < n; c += BJ_THREADS) {
                const double t = A[size_t(k) * n + c];
                A[size_t(k) * n + c] = A[size_t(pr) * n + c];
                A[size_t(pr) * n + c] = t;
            }
        __syncthreads();
        for (int i = tid; i < n; i += BJ_THREADS) colk[i] = A[size_t(i) * n + k];
        __syncthreads();
        const double inv = 1.0 / colk[k];
        for (int c = tid; c < n; c += BJ_THREADS)
            A[size_t(k) * n + c] = (c == k) ? inv : A[size_t(k) * n + c] * inv;
        __syncthreads();
        // Rows are processed in register-staged batches of 8 so that the LDS
        // loads of a batch are in flight together (the row updates of one
        // column are independent).
        const int g = tid / BJ_COLS, ng = BJ_THREADS / BJ_COLS;
        for (int c = tid % BJ_COLS; c < n; c += BJ_COLS) {
            const double akc = A[size_t(k) * n + c];
            const bool pivcol = (c == k);
            int i = g;
            for (; i + 7 * ng < n; i += 8 * ng) {
                double v[8], f[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    v[u] = A[size_t(i + u * ng) * n + c];
                    f[u] = colk[i + u * ng];
                }
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    v[u] = (i + u * ng == k) ? v[u] : (pivcol ? -f[u] * inv : v[u] - f[u] * akc);
#pragma unroll
                for (int u = 0; u < 8; ++u) A[size_t(i + u * ng) * n + c] = v[u];
            }
            for (; i < n; i += ng)
                if (i != k) A[size_t(i) * n + c] = pivcol ? -colk[i] * inv : A[size_t(i) * n + c] - colk[i] * akc;
        }
        __syncthreads();
    }
    // undo the row interchanges as column interchanges, in reverse order
    for (int k = n - 1; k >= 0; --k) {
        const int pr = perm[k];
        if (pr != k)
            for (int i = tid; i < n; i += BJ_THREADS) {
                const double t = A[size_t(i) * n + k];
                A[size_t(i) * n + k] = A[size_t(i) * n + pr];
                A[size_t(i) * n + pr] = t;
            }
        __syncthreads();
    }
    return true;
}

// One workgroup per cell.  USE_LDS: the block lives in dynamic LDS; else in
// the global scratch block of the cell.  The inverse goes to out,
// column-major.
template <bool USE_LDS>
__global__ __launch_bounds__(BJ_THREADS) void k_bj_build(DevMesh m, int restrict_,
                                                        const int64_t *inv_off,
                                                        double *__restrict__ out,
                                                        double *__restrict__ scratch,
                                                        int *__restrict__ status) {
    extern __shared__ double lds[];
    __shared__ double cth[NMq], sth[NMq];
    __shared__ double colk[RTX_NMAX * RTX_NMAX * RTX_NMAX];
    __shared__ int perm[RTX_NMAX * RTX_NMAX * RTX_NMAX];
    __shared__ int piv_row;
    const int k = blockIdx.x, tid = threadIdx.x;
    const int c = m.cell_col[k];
    const int nth = m.cell_nth[k];
    const int n = m.col_nx[c] * m.col_ny[c] * nth;
    if (tid < nth) {
        const double th0 = m.cell_geom[2 * k], dth = m.cell_geom[2 * k + 1] - th0;
        double s, cc;
        sincos(th0 + dth * 0.5 * (m.lg_x[nth * NMq + tid] + 1.0), &s, &cc);
        cth[tid] = cc;
        sth[tid] = s;
    }
    __syncthreads();
    double *A = USE_LDS ? lds : scratch + inv_off[k];
    bj_assemble(m, k, restrict_, A, cth, sth);
    const bool ok = bj_invert(A, n, colk, perm, &piv_row);
    if (!ok) {
        if (tid == 0) atomicMax(status, k + 1);
        return;
    }
    double *o = out + inv_off[k];
    for (int col = 0; col < n; ++col)
        for (int row = tid; row < n; row += BJ_THREADS) o[size_t(col) * n + row] = A[size_t(row) * n + col];
}

// FP8 e4m3 (bias 7, largest finite 448, no infinities): nearest code, ties to
// even, by the hardware conversion; |v| above 448 saturates; -0 gets code 0.
__device__ inline uint8_t bj_to_e4m3(float v) {
    v = fminf(fmaxf(v, -448.f), 448.f) + 0.f;
    return uint8_t(__builtin_amdgcn_cvt_pk_fp8_f32(v, v, 0, false));
}

// FP4 e2m1 (OCP: bias 1, one mantissa bit, largest 6, no infinities or
// NaN; magnitudes 0, 0.5, 1, 1.5, 2, 3, 4, 6 for codes 0..7): nearest code,
// ties to the even code, by the hardware conversion; |v| above 6 saturates;
// -0 gets code 0.
__device__ inline uint32_t bj_to_e2m1(float v) {
    v = fminf(fmaxf(v, -6.f), 6.f) + 0.f;
    return __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(0u, v, v, 1.f, 0) & 15u;
}

// ---- register-resident build for blocks of up to 128 DOFs.
struct BJCell {
    int nx, ny, nth, quad, bd;
    double dx, dy, dth;
    const double *wx, *wy, *wt, *Dx, *Dy, *kap, *sig;
};

struct BJSelf {                  // links of a cell to itself (periodic faces), in LDS
    int n;
    int F[4];
    int es[4], et[4];
};

// The block's entry at row (p, q, r), column (i, j, a): spatial nodes and
// angles of the cell; Gb = the cell's scattering block G[a][r] from angle a0
// on, g x g.
__device__ inline double bj_entry(const DevMesh &m, const BJCell &x, const BJSelf &sl,
                                  const double *cth, const double *sth, const double *Gb, int a0,
                                  int g, int p, int q, int r, int i, int j, int a) {
    if (x.bd) {
        const bool rb = bj_on_bdry(x.bd, p, q, x.nx, x.ny);
        const bool cb = bj_on_bdry(x.bd, i, j, x.nx, x.ny);
        if (rb || cb) return (p == i && q == j && r == a) ? 1.0 : 0.0;
    }
    double v = 0.0;
    if (p == i && q == j) {
        v = -x.dx * x.dy * x.wx[p] * x.wy[q] * x.sig[p * x.ny + q] * Gb[(a - a0) * g + r - a0];
        if (r == a) {
            double d = (x.dx * x.dy * x.dth * 0.125) * x.wx[p] * x.wy[q] * x.wt[r] * x.kap[p * x.ny + q];
            if (x.quad >= 0)
                for (int h = 0; h < 2; ++h) {
                    const int F = (x.quad + h) & 3;
                    const bool on = (F == 0 && p == x.nx - 1) || (F == 2 && p == 0) ||
                                    (F == 1 && q == x.ny - 1) || (F == 3 && q == 0);
                    if (on) {
                        const double tf = F == 0 ? cth[r] : (F == 1 ? sth[r] : (F == 2 ? -cth[r] : -sth[r]));
                        d += ((F & 1) ? x.dx : x.dy) * x.dth * 0.25 * ((F & 1) ? x.wx[p] : x.wy[q]) *
                             x.wt[r] * tf;
                    }
                }
            v += d;
        }
    }
    if (q == j && r == a)
        v -= (x.dy * x.dth * 0.25) * x.wy[q] * x.wt[r] * cth[r] * x.wx[i] * x.Dx[p * NMq + i];
    if (p == i && r == a)
        v -= (x.dx * x.dth * 0.25) * x.wx[p] * x.wt[r] * sth[r] * x.wy[j] * x.Dy[q * NMq + j];
    for (int l = 0; l < sl.n; ++l) {
        const int F = sl.F[l];
        int m0, m1;
        bool hit;
        if (F == 0) { hit = p == x.nx - 1 && i == 0; m0 = q; m1 = j; }
        else if (F == 2) { hit = p == 0 && i == x.nx - 1; m0 = q; m1 = j; }
        else if (F == 1) { hit = q == x.ny - 1 && j == 0; m0 = p; m1 = i; }
        else { hit = q == 0 && j == x.ny - 1; m0 = p; m1 = i; }
        if (hit) {
            const int n0 = (F & 1) ? x.nx : x.ny;
            v += ((F & 1) ? x.dx : x.dy) * x.dth * 0.25 * m.Es_pool[sl.es[l] + m1 * n0 + m0] *
                 m.Eth_pool[sl.et[l] + a * x.nth + r];
        }
    }
    return v;
}

// One workgroup per block, the block's index from the size-class list bl
// (blocks of 16 (NT - 1) + 1 .. 16 NT DOFs).  T: the elimination's arithmetic
// and the inverse's storage (FP64, or FP32 for the reduced-precision copies
// alone; the entries are assembled in FP64 either way).
//
// Blocked Gauss-Jordan on M = (block)^T, in registers.  Wave w holds columns
// 16 w .. 16 w + 15 of M in the accumulator layout of the 16 x 16 matrix
// instruction.  The columns are eliminated in panels of 16, panel k by wave k
// alone: it turns its tile to one row (two for NT > 4) per lane through LDS,
// sweeps its 16 columns with partial pivoting (wavefront maximum by DPP, the
// pivot row broadcast by readlane, no block barrier), and leaves the swept
// panel W in LDS.  After the sweeps every other column c is
//     M[:, c] <- M[:, c] with the panel's pivot rows zeroed + W M_P[:, c],
// M_P the 16 pivot rows before the panel: four matrix instructions per 16 x
// 16 tile.  Rows are never moved: with p_k the pivot row of column k and q =
// p^-1, inv(M)[q_i][p_j] is what M[i][j] ends as, so inv(block)[p_j][q_i],
// and a tile's 16 lanes store runs of one column of the inverse.
//
// Bound by the panels (half of the FP64 time: pivot search, broadcast and
// reciprocal in series) and the matrix instructions.  A rank-1 form with two
// block barriers per column and five instructions per element and column
// took 14.6 ms for 16,384 blocks of 125 in FP64 (this: 3.2, the FP64 rate's
// floor 0.9) and 31.3 ms for the 91,352 blocks of an hp mesh of 8.3 M DOF in
// FP32 (this: 6.9).  One barrier per panel is left; the next panel's wave
// starts as soon as its own tile is updated (W is double-buffered), at raised
// priority because the panels are the serial chain.  Registers: two blocks of
// eight waves per CU in FP64 (128 VGPRs); in FP32 four (64 VGPRs with 2 to 15
// spilled, 43 where NT is 6 and the inverse is stored: 16,384 blocks of 125 in
// 1.83 ms, against 2.0 at 80 VGPRs and 2.5 without a limit, before the
// assembly's index tables took it to 1.68).  Measured at NT = 8 alone.
template <int NT, typename T>
struct BJReg {
    static constexpr int NR = 16 * NT;
    static constexpr int WS = 18;                 // row stride of W: lane rows and operand
                                                  // reads both spread over the banks
    static constexpr int SS = NR + 2;             // row stride of the assembly strip
    static constexpr int H = NT > 4 ? 2 : 1;      // rows per lane of a panel
    static_assert(32 * SS <= 2 * NR * WS, "a 32-row strip fits the panel buffers");
};

__device__ inline uint32_t bj_key(double v) {
    return static_cast<uint32_t>(__double2hiint(v)) & 0x7fffff80u;
}
__device__ inline uint32_t bj_key(float v) { return __float_as_uint(v) & 0x7fffff80u; }
// keys of NaN start here
template <typename T>
__device__ constexpr uint32_t bj_key_nan() { return sizeof(T) == 8 ? 0x7ff00080u : 0x7f800080u; }

__device__ inline double bj_lane(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}
__device__ inline float bj_lane(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Largest value over the wavefront, in every lane's scalar view.
__device__ inline uint32_t bj_wave_max(uint32_t v) {
    auto step = [&](uint32_t o) { v = o > v ? o : v; };
    step(uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x111, 0xf, 0xf, false)));   // row_shr:1
    step(uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x112, 0xf, 0xf, false)));   // row_shr:2
    step(uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x114, 0xf, 0xf, false)));   // row_shr:4
    step(uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x118, 0xf, 0xf, false)));   // row_shr:8
    step(uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x142, 0xf, 0xf, false)));   // row_bcast:15
    step(uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x143, 0xf, 0xf, false)));   // row_bcast:31
    return uint32_t(__builtin_amdgcn_readlane(int(v), 63));
}

template <typename T> struct BJMma;
template <> struct BJMma<double> {
    typedef double v4 __attribute__((ext_vector_type(4)));
    __device__ static v4 step(double a, double b, v4 c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    // row of accumulator v in lane group lg, and its inverse: row r is entry
    // (r >> 4) 4 + v of lane group lg
    __device__ static int row(int lg, int v) { return lg + 4 * v; }
    __device__ static int slot(int r) { return (r & 3) * 32 + (r >> 2); }
};
template <> struct BJMma<float> {
    typedef float v4 __attribute__((ext_vector_type(4)));
    __device__ static v4 step(float a, float b, v4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ static int row(int lg, int v) { return 4 * lg + v; }
    __device__ static int slot(int r) { return ((r >> 2) & 3) * 32 + (r >> 4) * 4 + (r & 3); }
};

// A wave's own LDS writes made visible to its other lanes.
__device__ inline void bj_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// 1 / p to an ulp (hardware reciprocal and Newton steps): a pivot's relative
// perturbation of that size is one rounding of the elimination.  0 for an
// infinite p (where a Newton step gives NaN).
__device__ inline double bj_recip(double p) {
    const double r = __builtin_amdgcn_rcp(p);
    double q = fma(fma(-p, r, 1.0), r, r);
    q = fma(fma(-p, q, 1.0), q, q);
    return r == 0.0 ? 0.0 : q;
}
__device__ inline float bj_recip(float p) {
    const float r = __builtin_amdgcn_rcpf(p);
    const float q = fmaf(fmaf(-p, r, 1.f), r, r);
    return r == 0.f ? 0.f : q;
}

// Sweep the 16 columns of a panel held one row (H rows, 64 apart) per lane.
// q: byte table of the step that each row was pivot of (BJMma::slot order);
// perm: pivot row of each step.  False on a zero or NaN pivot (the
// same for every lane; what the panel holds then is void).
template <int H, typename T>
__device__ __forceinline__ bool bj_panel(T (&P0)[16], T (&P1)[16], int k0, int lane, bool used0,
                                         bool used1, uint8_t *q, int32_t *perm) {
    bool bad = false;
    // In-place Gauss-Jordan with the pivot rows' division left to the end: a
    // step adds -c_r / p times the pivot row to every other row (the pivot
    // row's factor is 0) and puts -c_r / p (1 in the pivot row) in its
    // column; the panel's pivot rows are divided by their pivots at the end.
    // Nothing but the FMAs touches a whole row, and the pivot row's values
    // are scalar operands of them.
    T s0 = T(1), s1 = T(1);
    int step0 = -1, step1 = -1;          // steps that this lane's rows were pivots of
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        // key: the high bits of |value| (13 mantissa bits in FP64, 16 in
        // FP32) over 127 - row: a pivot within 2^-13 of the largest, the
        // lowest row among ties
        uint32_t key = used0 ? 0u : bj_key(P0[k]) | uint32_t(127 - lane);
        if constexpr (H == 2) {
            const uint32_t v = used1 ? 0u : bj_key(P1[k]) | uint32_t(63 - lane);
            key = v > key ? v : key;
        }
        key = bj_wave_max(key);
        bad |= key < 0x80u || key >= bj_key_nan<T>();
        const int pr = 127 - int(key & 127u), pl = pr & 63;
        const bool low = H == 1 || pr < 64;
        T row[16];
        if (low) {
#pragma unroll
            for (int c = 0; c < 16; ++c) row[c] = bj_lane(P0[c], pl);
        } else {
#pragma unroll
            for (int c = 0; c < 16; ++c) row[c] = bj_lane(P1[c], pl);
        }
        const T inv = bj_recip(row[k]);
        const bool is0 = low && lane == pl, is1 = !low && lane == pl;
        const T f0 = P0[k] * inv, f1 = P1[k] * inv;
        const T g0 = is0 ? T(0) : -f0, g1 = is1 ? T(0) : -f1;
#pragma unroll
        for (int c = 0; c < 16; ++c)
            if (c != k) {
                P0[c] = fma(g0, row[c], P0[c]);
                if constexpr (H == 2) P1[c] = fma(g1, row[c], P1[c]);
            }
        P0[k] = is0 ? T(1) : g0;
        s0 = is0 ? inv : s0;
        used0 = used0 || is0;
        if constexpr (H == 2) {
            P1[k] = is1 ? T(1) : g1;
            s1 = is1 ? inv : s1;
            used1 = used1 || is1;
        }
        step0 = is0 ? k0 + k : step0;
        if constexpr (H == 2) step1 = is1 ? k0 + k : step1;
    }
    if (step0 >= 0) {
        q[BJMma<T>::slot(lane)] = uint8_t(step0);
        perm[step0] = lane;
    }
    if (H == 2 && step1 >= 0) {
        q[BJMma<T>::slot(lane + 64)] = uint8_t(step1);
        perm[step1] = lane + 64;
    }
#pragma unroll
    for (int c = 0; c < 16; ++c) {
        P0[c] *= s0;
        if constexpr (H == 2) P1[c] *= s1;
    }
    return !bad;
}

//
// BITS 8 or 4 (T = float): the inverse is not stored; each of its columns is
// scaled and rounded to FP8 / FP4 codes in registers, in the layout and with
// the bytes of k_bj_pack_fp8 / _fp4, through an image in the dead panel
// buffers. The FP32 pool that the separate pass reads (3.2 GB on the hp mesh
// above) is neither allocated nor written: 7.5 ms instead of 7.2 + 2.7.
template <int NT, typename T, int BITS = 0>
__global__ __launch_bounds__(64 * NT)
__attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? (NT > 4 ? 4 : 5) : 8)))
void k_bj_build_reg(DevMesh m, int restrict_, const int64_t *inv_off,
                    const int32_t *__restrict__ blk, const int32_t *__restrict__ bl,
                    typename std::conditional<BITS == 0, T, uint8_t>::type *__restrict__ out,
                    const int64_t *soff, float *__restrict__ scales, int *__restrict__ status) {
    typedef BJReg<NT, T> R;
    typedef BJMma<T> Mma;
    typedef typename Mma::v4 v4;
    constexpr int NR = R::NR, WS = R::WS, SS = R::SS, H = R::H;
    __shared__ __attribute__((aligned(16))) T buf[2 * NR * WS];   // strip, then W of two panels
    __shared__ T piv[NT][17 * 16];                // each wave's pivot rows of its own columns
    __shared__ double cth[NMq], sth[NMq], wx[NMq], wy[NMq], wt[NMq];
    __shared__ double Dx[NMq * NMq], Dy[NMq * NMq], kap[NMq * NMq], sig[NMq * NMq], Gb[NMq * NMq];
    __shared__ int32_t at[NR];                    // node i | j << 8 | angle << 16 of a block index
    __shared__ __attribute__((aligned(16))) uint8_t q[4 * 32];
    __shared__ int32_t perm[NR];
    __shared__ int failed;
    __shared__ BJSelf sl;
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b = bl[blockIdx.x];
    const int k = blk[3 * b], a0 = blk[3 * b + 1], g = blk[3 * b + 2];
    BJCell x;
    const int c = m.cell_col[k];
    x.nx = m.col_nx[c];
    x.ny = m.col_ny[c];
    x.nth = m.cell_nth[k];
    x.dx = m.col_geom[4 * c + 2] - m.col_geom[4 * c + 0];
    x.dy = m.col_geom[4 * c + 3] - m.col_geom[4 * c + 1];
    const double th0 = m.cell_geom[2 * k];
    x.dth = m.cell_geom[2 * k + 1] - th0;
    x.wx = wx;
    x.wy = wy;
    x.wt = wt;
    x.Dx = Dx;
    x.Dy = Dy;
    x.kap = kap;
    x.sig = sig;
    x.quad = m.cell_quad[k];
    x.bd = restrict_ ? m.cell_bdry[k] : 0;
    const int nsp = x.nx * x.ny, sp0 = m.col_sp_off[c], na = m.col_nang[c];
    const double *G = m.G + m.col_G_off[c] + size_t(m.cell_ang_off[k] + a0) * (na + 1);
    // the block: angles a0 .. a0 + g - 1 of the cell at every spatial node;
    // block index t <-> cell DOF (t / g) nth + a0 + t % g
    const int n = nsp * g;
    for (int t = tid; t < NMq * NMq; t += 64 * NT) {
        if (t < g * g) Gb[t] = G[size_t(t / g) * na + t % g];
        Dx[t] = m.lgl_D[size_t(x.nx) * NMq * NMq + t];
        Dy[t] = m.lgl_D[size_t(x.ny) * NMq * NMq + t];
        if (t < nsp) {
            kap[t] = m.kappa[sp0 + t];
            sig[t] = m.sigma[sp0 + t];
        }
        if (t < NMq) {
            wx[t] = m.lgl_w[x.nx * NMq + t];
            wy[t] = m.lgl_w[x.ny * NMq + t];
            wt[t] = m.lg_w[x.nth * NMq + t];
        }
    }
    if (tid == 0) {
        int ns = 0;
        for (int l = m.link_start[k]; l < m.link_start[k + 1] && ns < 4; ++l)
            if (m.link_src[l] == k) {
                sl.F[ns] = m.link_face[l];
                sl.es[ns] = m.link_Es_off[l];
                sl.et[ns] = m.link_Eth_off[l];
                ++ns;
            }
        sl.n = ns;
        failed = 0;
    }
    if (tid < x.nth) {
        double s, cc;
        sincos(th0 + x.dth * 0.5 * (m.lg_x[x.nth * NMq + tid] + 1.0), &s, &cc);
        cth[tid] = cc;
        sth[tid] = s;
    }
    for (int t = tid; t < 4 * 32; t += 64 * NT) q[t] = 0xff;
    for (int t = tid; t < n; t += 64 * NT) {
        const int node = t / g, i = node / x.ny;
        at[t] = i | (node - i * x.ny) << 8 | (t - node * g) << 16;
    }
    for (int t = tid; t < 32 * SS; t += 64 * NT) buf[t] = T(0);
    // Assembly by strips of 32 rows of M (columns of the block): of a row's n
    // entries at most g + nx + ny - 2 are not zero (the node's angles, the
    // two derivative lines), so those alone are evaluated, one per thread,
    // and cleared again after the strip is read.
    v4 acc[NT];
    __syncthreads();
    const int each = sl.n ? n : g + x.nx + x.ny - 2;   // self links couple whole faces
    const float r_each = 1.f / float(each);            // e < 32 128: exact quotients
    const auto entries = [&](int s, auto put) {
        const int rows = min(32, n - 32 * s);
        for (int e = tid; e < rows * each; e += 64 * NT) {
            const int rr = int((float(e) + 0.5f) * r_each), f = e - rr * each;
            const int c0 = at[32 * s + rr], i = c0 & 255, j = (c0 >> 8) & 255, r = c0 >> 16;
            int p = i, pq = j, a = r;
            if (sl.n) {
                const int c1 = at[f];
                p = c1 & 255;
                pq = (c1 >> 8) & 255;
                a = c1 >> 16;
            } else if (f < g)
                a = f;
            else if (f < g + x.nx - 1)
                p = f - g + (f - g >= i);
            else
                pq = f - g - x.nx + 1 + (f - g - x.nx + 1 >= j);
            put(rr * SS + (p * x.ny + pq) * g + a, p, pq, a, i, j, r);
        }
    };
#pragma unroll
    for (int s = 0; s < (NT + 1) / 2; ++s) {
        entries(s, [&](int o, int p, int pq, int a, int i, int j, int r) {
            buf[o] = T(bj_entry(m, x, sl, cth, sth, Gb, a0, g, p, pq, a0 + a, i, j, a0 + r));
        });
        // unit diagonal past the block: those columns pivot on their own rows
        if (tid < 32 && 32 * s + tid >= n && 32 * s + tid < NR) buf[tid * SS + 32 * s + tid] = T(1);
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (2 * s + h < NT) {
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    acc[2 * s + h][v] = buf[(16 * h + Mma::row(lg, v)) * SS + 16 * wave + l16];
            }
        __syncthreads();
        if (2 * s + 2 < NT) {
            entries(s, [&](int o, int, int, int, int, int, int) { buf[o] = T(0); });
            __syncthreads();
        }
    }
    // Panel p of another wave: update this wave's tile.
    auto update = [&](int p) {
        const T *W = buf + (p & 1) * NR * WS;
        __syncthreads();
        // This wave's entries of the panel's pivot rows -> piv, zero in M.
        // q may get entries of the next panel meanwhile: those steps are
        // 16 (p + 1) or more, no match either way.
#pragma unroll
        for (int rt = 0; rt < NT; ++rt) {
            const uint32_t qs = *reinterpret_cast<const uint32_t *>(q + lg * 32 + rt * 4);
            // a byte of t is zero where a row of this lane is a pivot of
            // panel p; most row tiles have none
            const uint32_t t = ((qs >> 4) & 0x0f0f0f0fu) ^ (uint32_t(p) * 0x01010101u);
            if (__any(((t - 0x01010101u) & ~t & 0x80808080u) != 0)) {
                v4 keep;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    // rows that are no pivots go to the spare row 16
                    const uint32_t s = min(((qs >> (8 * v)) & 255u) - 16u * p, 16u);
                    piv[wave][s * 16 + l16] = acc[rt][v];
                    keep[v] = s < 16u ? T(0) : T(1);
                }
                acc[rt] *= keep;
            }
        }
        bj_wave_sync();
#pragma unroll 1
        for (int s = 0; s < 4; ++s) {
            const T bv = piv[wave][(4 * s + lg) * 16 + l16];
#pragma unroll
            for (int rt = 0; rt < NT; ++rt)
                acc[rt] = Mma::step(W[(16 * rt + l16) * WS + 4 * s + lg], bv, acc[rt]);
        }
        bj_wave_sync();                              // piv is written again by the next panel
    };
    // Straight-line phases rather than one loop with a branch on the panel's
    // owner: the branch made the compiler keep two copies of the tile.
#pragma unroll 1
    for (int p = 0; p < wave; ++p) update(p);
    {
        T *W = buf + (wave & 1) * NR * WS;
        __builtin_amdgcn_s_setprio(3);
#pragma unroll
        for (int rt = 0; rt < NT; ++rt)
#pragma unroll
            for (int v = 0; v < 4; ++v) W[(16 * rt + Mma::row(lg, v)) * WS + l16] = acc[rt][v];
        bj_wave_sync();
        // rows that earlier panels took are no candidates
        const int r0 = NT > 3 ? lane : min(lane, NR - 1), r1 = H == 2 ? min(lane + 64, NR - 1) : 0;
        T P0[16], P1[16];
#pragma unroll
        for (int cc = 0; cc < 16; ++cc) {
            P0[cc] = W[r0 * WS + cc];
            P1[cc] = H == 2 ? W[r1 * WS + cc] : T(0);
        }
        const bool ok = bj_panel<H, T>(P0, P1, 16 * wave, lane,
                                       lane >= NR || q[Mma::slot(r0)] != 0xff,
                                       lane + 64 >= NR || q[Mma::slot(r1)] != 0xff, q, perm);
        if (!ok && lane == 0) {
            failed = 1;
            atomicMax(status, k + 1);
        }
#pragma unroll
        for (int cc = 0; cc < 16; ++cc) {
            if (NT > 3 || lane < NR) W[r0 * WS + cc] = P0[cc];
            if (H == 2 && lane + 64 < NR) W[r1 * WS + cc] = P1[cc];
        }
        __builtin_amdgcn_s_setprio(0);
        __syncthreads();
#pragma unroll
        for (int rt = 0; rt < NT; ++rt)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[rt][v] = W[(16 * rt + Mma::row(lg, v)) * WS + l16];
    }
#pragma unroll 1
    for (int p = wave + 1; p < NT; ++p) update(p);
    __syncthreads();
    if (failed) return;
    const int j = 16 * wave + l16;
    if constexpr (BITS == 0) {
        if (j >= n) return;
        T *o = out + inv_off[b] + perm[j];
#pragma unroll
        for (int rt = 0; rt < NT; ++rt) {
            const uint32_t qs = *reinterpret_cast<const uint32_t *>(q + lg * 32 + rt * 4);
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (16 * rt + Mma::row(lg, v) < n) o[size_t((qs >> (8 * v)) & 255u) * n] = acc[rt][v];
        }
    } else {
        // largest magnitude of each row i of M (column q_i of the inverse):
        // over a wave's 16 columns, then over the waves; columns past the
        // block are zero there
        static_assert(NT * 17 * 16 >= NT * NR, "row maxima of every wave fit piv");
        static_assert(NR * NR <= int(sizeof(buf)), "the code image fits the panel buffers");
        static_assert(NR * 4 <= int(sizeof(Dx)), "the scales fit Dx");
        float *const mx = reinterpret_cast<float *>(piv);
        float *const inv_s = reinterpret_cast<float *>(Dx);
        uint8_t *const img = reinterpret_cast<uint8_t *>(buf);
#pragma unroll
        for (int rt = 0; rt < NT; ++rt)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                float a = fabsf(acc[rt][v]);
#pragma unroll
                for (int o = 8; o > 0; o >>= 1) a = fmaxf(a, __shfl_xor(a, o, 16));
                if (l16 == 0) mx[wave * NR + 16 * rt + Mma::row(lg, v)] = a;
            }
        __syncthreads();
        for (int i = tid; i < NR; i += 64 * NT) {
            float a = 0.f;
#pragma unroll
            for (int w = 0; w < NT; ++w) a = fmaxf(a, mx[w * NR + i]);
            const float sc = a > 0.f ? a / (BITS == 8 ? 448.f : 6.f) : 1.f;
            inv_s[i] = 1.f / sc;
            if (i < n) scales[soff[b] + q[Mma::slot(i)]] = sc;
        }
        __syncthreads();
        // one code per byte at [column q_i][row p_j] of the inverse; rows
        // past the block are zero in M, so they get code 0
        const int pj = perm[j];
#pragma unroll
        for (int rt = 0; rt < NT; ++rt) {
            const uint32_t qs = *reinterpret_cast<const uint32_t *>(q + lg * 32 + rt * 4);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = 16 * rt + Mma::row(lg, v);
                const float f = acc[rt][v] * inv_s[i];
                const uint32_t cd = BITS == 8 ? uint32_t(bj_to_e4m3(f)) : bj_to_e2m1(f);
                img[((qs >> (8 * v)) & 255u) * NR + pj] = uint8_t(cd);
            }
        }
        __syncthreads();
        const uint4 *I = reinterpret_cast<const uint4 *>(img);
        if constexpr (BITS == 8) {
            uint4 *D = reinterpret_cast<uint4 *>(out + inv_off[b]);
            for (int e = tid; e < n * NT; e += 64 * NT) D[e] = I[e];
        } else {
            // bytes 2 t and 2 t + 1 -> the nibbles of byte t
            auto two = [](uint32_t lo, uint32_t hi) {
                auto half = [](uint32_t w) {
                    w |= w >> 4;
                    return (w & 0xffu) | ((w >> 8) & 0xff00u);
                };
                return half(lo) | (half(hi) << 16);
            };
            uint2 *D = reinterpret_cast<uint2 *>(out + inv_off[b] / 2);
            for (int e = tid; e < n * NT; e += 64 * NT) {
                const uint4 w = I[e];
                D[e] = make_uint2(two(w.x, w.y), two(w.z, w.w));
            }
        }
    }
}

__global__ void k_to_f32_bj(const double *__restrict__ s, float *__restrict__ d, int64_t n) {
    int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    for (; i < n; i += int64_t(gridDim.x) * blockDim.x) d[i] = float(s[i]);
}

// z_K = inv_K r_K, inv column-major.  One workgroup per cell; the columns
// are split across the four wavefronts' partial sums when n is small.
// BF16 storage of an inverse entry, widened on load.
template <typename T, typename M>
__global__ __launch_bounds__(BJ_THREADS) void k_bj_apply(DevMesh m, const int64_t *inv_off,
                                                        const int4 *__restrict__ apd,
                                                        const M *__restrict__ inv,
                                                        const T *__restrict__ r,
                                                        T *__restrict__ z) {
    __shared__ double rs[RTX_NMAX * RTX_NMAX * RTX_NMAX];
    __shared__ double part[BJ_THREADS];
    const int b = blockIdx.x, tid = threadIdx.x;
    const int4 d = apd[b];                // n, first DOF, cell angles, angles g
    const int n = d.x, nth = d.z, g = d.w;
    // block index t <-> cell DOF (t / g) nth + a0 + t % g (identity for a whole cell)
    const int off = d.y;
    for (int i = tid; i < n; i += BJ_THREADS) rs[i] = double(r[off + (i / g) * nth + i % g]);
    __syncthreads();
    const M *B = inv + inv_off[b];
    if (n <= BJ_THREADS / 2) {
        // two column halves per output row
        const int half = tid / (BJ_THREADS / 2), i = tid % (BJ_THREADS / 2);
        double acc = 0.0;
        if (i < n) {
            const int j0 = half * ((n + 1) / 2), j1 = half ? n : (n + 1) / 2;
#pragma unroll 4
            for (int j = j0; j < j1; ++j) acc += double(B[size_t(j) * n + i]) * rs[j];
        }
        part[tid] = acc;
        __syncthreads();
        if (tid < n) z[off + (tid / g) * nth + tid % g] = T(part[tid] + part[tid + BJ_THREADS / 2]);
    } else {
        for (int i = tid; i < n; i += BJ_THREADS) {
            double acc = 0.0;
#pragma unroll 4
            for (int j = 0; j < n; ++j) acc += double(B[size_t(j) * n + i]) * rs[j];
            z[off + (i / g) * nth + i % g] = T(acc);
        }
    }
}

__device__ inline uint16_t bj_to_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return uint16_t(u >> 16);
}

__device__ inline int bj_block_n(const DevMesh &m, const int32_t *blk, int b) {
    const int k = blk[3 * b], g = blk[3 * b + 2];
    const int c = m.cell_col[k];
    return m.col_nx[c] * m.col_ny[c] * g;
}

// Packed BF16 copy: column j of block b at off16[b] + j * ldp, ldp = n
// rounded up to 8 (padding rows zero), so every column starts on 16 bytes.
__global__ __launch_bounds__(BJ_THREADS) void k_bj_pack_bf16(DevMesh m, const int64_t *off,
                                                             const int64_t *off16,
                                                             const int32_t *__restrict__ blk,
                                                             const float *__restrict__ src,
                                                             uint16_t *__restrict__ dst) {
    const int b = blockIdx.x;
    const int n = bj_block_n(m, blk, b), ldp = (n + 7) / 8 * 8;
    const float *S = src + off[b];
    uint16_t *D = dst + off16[b];
    for (int e = threadIdx.x; e < n * ldp; e += BJ_THREADS) {
        const int j = e / ldp, i = e % ldp;
        D[e] = i < n ? bj_to_bf16(S[size_t(j) * n + i]) : uint16_t(0);
    }
}

// z = B r for one block from the packed BF16 inverse: thread (cg, rg) owns
// rows 8 rg .. 8 rg + 7 and columns cg, cg + CG, ...; one 16-byte load per
// column; the CG partial sums of each row are added in LDS.
template <int NT>
__global__ __launch_bounds__(NT) void k_bj_apply_bf16(DevMesh m, const int64_t *off16,
                                                              const int4 *__restrict__ apd,
                                                              const uint16_t *__restrict__ inv,
                                                              const float *__restrict__ r,
                                                              float *__restrict__ z) {
    __shared__ float rs[RTX_NMAX * RTX_NMAX * RTX_NMAX];
    __shared__ float part[NT * 8];
    const int b = blockIdx.x, tid = threadIdx.x;
    const int4 d = apd[b];                // n, first DOF, cell angles, angles g
    const int n = d.x, nth = d.z, g = d.w;
    const int ldp = (n + 7) / 8 * 8, RG = ldp / 8, CG = NT / RG;
    const int off = d.y;
    const int rg = tid % RG, cg = tid / RG;
    const uint4 *B = reinterpret_cast<const uint4 *>(inv + off16[b]) + rg;
    const int ldq = ldp / 8;
    // the first 8 columns of this thread are fetched before the wait on r,
    // so the inverse loads and the r gather are in flight together
    constexpr int PF = 2048 / NT;
    uint4 q[PF];
#pragma unroll
    for (int u = 0; u < PF; ++u) {
        const int j = cg + u * CG;
        q[u] = (cg < CG && j < n) ? B[size_t(j) * ldq] : make_uint4(0u, 0u, 0u, 0u);
    }
    for (int i = tid; i < n; i += NT) rs[i] = r[off + (i / g) * nth + i % g];
    __syncthreads();
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    auto fma8 = [&](const uint4 &v, float rj) {
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            acc[2 * u] += __uint_as_float(w[u] << 16) * rj;
            acc[2 * u + 1] += __uint_as_float(w[u] & 0xffff0000u) * rj;
        }
    };
    if (cg < CG) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            const int j = cg + u * CG;
            if (j < n) fma8(q[u], rs[j]);
        }
#pragma unroll 4
        for (int j = cg + PF * CG; j < n; j += CG) fma8(B[size_t(j) * ldq], rs[j]);
#pragma unroll
        for (int u = 0; u < 8; ++u) part[cg * ldp + rg * 8 + u] = acc[u];
    }
    __syncthreads();
    for (int i = tid; i < n; i += NT) {
        float s = 0.f;
        for (int q = 0; q < CG; ++q) s += part[q * ldp + i];
        z[off + (i / g) * nth + i % g] = s;
    }
}

// Column scales of one block for the coded copies: scale_j = max_i |B_ij| /
// div (1 for an all-zero column) into sc[j] and its reciprocal into inv_s[j].
// One wavefront per column: coalesced loads of the column and a shuffle
// reduction (the maximum does not depend on the order).
__device__ inline void bj_col_scales(const float *__restrict__ S, int n, float div,
                                     float *__restrict__ sc, float *inv_s) {
    static_assert(BJ_THREADS % 64 == 0, "whole wavefronts");
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int j = wave; j < n; j += BJ_THREADS / 64) {
        float mx = 0.f;
        for (int i = lane; i < n; i += 64) mx = fmaxf(mx, fabsf(S[size_t(j) * n + i]));
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
        if (lane == 0) {
            const float v = mx > 0.f ? mx / div : 1.f;
            sc[j] = v;
            inv_s[j] = 1.f / v;
        }
    }
}

// FP8 copy of block b: column j of codes at off8[b] + j * ldp (ldp = n
// rounded up to 16, padding zero), scale_j = max_i |B_ij| / 448 at
// scales[soff[b] + j]; code = e4m3(B_ij / scale_j).
__global__ __launch_bounds__(BJ_THREADS) void k_bj_pack_fp8(DevMesh m, const int64_t *off,
                                                            const int64_t *off8,
                                                            const int64_t *soff,
                                                            const int32_t *__restrict__ blk,
                                                            const float *__restrict__ src,
                                                            uint8_t *__restrict__ dst,
                                                            float *__restrict__ scales) {
    __shared__ float inv_s[RTX_NMAX * RTX_NMAX * RTX_NMAX];
    const int b = blockIdx.x;
    const int n = bj_block_n(m, blk, b), ldp = (n + 15) / 16 * 16;
    const float *S = src + off[b];
    uint8_t *D = dst + off8[b];
    bj_col_scales(S, n, 448.f, scales + soff[b], inv_s);
    __syncthreads();
    for (int e = threadIdx.x; e < n * ldp; e += BJ_THREADS) {
        const int j = e / ldp, i = e % ldp;
        D[e] = i < n ? bj_to_e4m3(S[size_t(j) * n + i] * inv_s[j]) : uint8_t(0);
    }
}

// FP4 copy of block b: the FP8 copy's layout at half the bytes (column j's
// codes at off8[b] / 2 + j * ldp / 2, row i in byte i / 2, the even row in
// the low nibble), scale_j = max_i |B_ij| / 6 at scales[soff[b] + j];
// code = e2m1(B_ij / scale_j).
__global__ __launch_bounds__(BJ_THREADS) void k_bj_pack_fp4(DevMesh m, const int64_t *off,
                                                            const int64_t *off8,
                                                            const int64_t *soff,
                                                            const int32_t *__restrict__ blk,
                                                            const float *__restrict__ src,
                                                            uint8_t *__restrict__ dst,
                                                            float *__restrict__ scales) {
    __shared__ float inv_s[RTX_NMAX * RTX_NMAX * RTX_NMAX];
    const int b = blockIdx.x;
    const int n = bj_block_n(m, blk, b), ldp = (n + 15) / 16 * 16, hp = ldp / 2;
    const float *S = src + off[b];
    uint8_t *D = dst + off8[b] / 2;
    bj_col_scales(S, n, 6.f, scales + soff[b], inv_s);
    __syncthreads();
    for (int e = threadIdx.x; e < n * hp; e += BJ_THREADS) {
        const int j = e / hp, i = 2 * (e % hp);
        const uint32_t lo = i < n ? bj_to_e2m1(S[size_t(j) * n + i] * inv_s[j]) : 0u;
        const uint32_t hi = i + 1 < n ? bj_to_e2m1(S[size_t(j) * n + i + 1] * inv_s[j]) : 0u;
        D[e] = uint8_t(lo | (hi << 4));
    }
}

// Sixteen consecutive codes of one column (rows 16 rg .. 16 rg + 15),
// decoded to FP32 by the gfx950 hardware conversions and multiplied into
// the row sums: acc[v] += code_v * rj.  FP8 e4m3: one 16-byte load, two
// codes per conversion; FP4 e2m1: one 8-byte load, two codes per
// conversion (scale 1).
template <int BITS>
struct BjCodes;
template <>
struct BjCodes<8> {
    typedef uint4 V;
    static constexpr int SHIFT = 0;    // byte offset of a block = off8[b] >> SHIFT
    __device__ static V zero() { return make_uint4(0u, 0u, 0u, 0u); }
    __device__ static void fma16(const V &v, float rj, float (&acc)[16]) {
        typedef float f2 __attribute__((ext_vector_type(2)));
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const f2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(int(w[u]), false);
            const f2 hi = __builtin_amdgcn_cvt_pk_f32_fp8(int(w[u]), true);
            acc[4 * u + 0] += lo.x * rj;
            acc[4 * u + 1] += lo.y * rj;
            acc[4 * u + 2] += hi.x * rj;
            acc[4 * u + 3] += hi.y * rj;
        }
    }
};
template <>
struct BjCodes<4> {
    typedef uint2 V;
    static constexpr int SHIFT = 1;
    __device__ static V zero() { return make_uint2(0u, 0u); }
    __device__ static void fma16(const V &v, float rj, float (&acc)[16]) {
        typedef float f2 __attribute__((ext_vector_type(2)));
        const uint32_t w[2] = {v.x, v.y};
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            // byte s of word u holds rows 8 u + 2 s (low nibble) and + 1
            const f2 p0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[u], 1.f, 0);
            const f2 p1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[u], 1.f, 1);
            const f2 p2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[u], 1.f, 2);
            const f2 p3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[u], 1.f, 3);
            acc[8 * u + 0] += p0.x * rj;
            acc[8 * u + 1] += p0.y * rj;
            acc[8 * u + 2] += p1.x * rj;
            acc[8 * u + 3] += p1.y * rj;
            acc[8 * u + 4] += p2.x * rj;
            acc[8 * u + 5] += p2.y * rj;
            acc[8 * u + 6] += p3.x * rj;
            acc[8 * u + 7] += p3.y * rj;
        }
    }
};

// z = B r from the FP8 (BITS 8) or FP4 (BITS 4) pool: thread (cg, rg) owns
// rows 16 rg .. 16 rg + 15 and columns cg, cg + CG, ...; one load of sixteen
// codes per column, decoded by the hardware conversion; the column scales
// are folded into r.
template <int NT, typename RT = float, int BITS = 8>
__global__ __launch_bounds__(NT) void k_bj_apply_fp8(DevMesh m, const int64_t *off8,
                                                     const int64_t *soff,
                                                     const int4 *__restrict__ apd,
                                                     const uint8_t *__restrict__ inv,
                                                     const float *__restrict__ scales,
                                                     const RT *__restrict__ r,
                                                     float *__restrict__ z) {
    __shared__ float rs[RTX_NMAX * RTX_NMAX * RTX_NMAX];
    __shared__ float part[NT * 16];
    const int b = blockIdx.x, tid = threadIdx.x;
    const int4 d = apd[b];                // n, first DOF, cell angles, angles g
    const int n = d.x, nth = d.z, g = d.w;
    const int ldp = (n + 15) / 16 * 16, RG = ldp / 16, CG = NT / RG;
    const int off = d.y;
    const int rg = tid % RG, cg = tid / RG;
    typedef BjCodes<BITS> Codes;
    typedef typename Codes::V CV;
    const CV *B = reinterpret_cast<const CV *>(inv + (off8[b] >> Codes::SHIFT)) + rg;
    const int ldq = ldp / 16;
    constexpr int PF = 4;
    CV q[PF];
#pragma unroll
    for (int u = 0; u < PF; ++u) {
        const int j = cg + u * CG;
        q[u] = (cg < CG && j < n) ? B[size_t(j) * ldq] : Codes::zero();
    }
    const float *sc = scales + soff[b];
    for (int i = tid; i < n; i += NT) rs[i] = float(r[off + (i / g) * nth + i % g]) * sc[i];
    __syncthreads();
    float acc[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) acc[u] = 0.f;
    auto fma16 = [&](const CV &v, float rj) { Codes::fma16(v, rj, acc); };
    if (cg < CG) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            const int j = cg + u * CG;
            if (j < n) fma16(q[u], rs[j]);
        }
        for (int j = cg + PF * CG; j < n; j += CG) fma16(B[size_t(j) * ldq], rs[j]);
#pragma unroll
        for (int u = 0; u < 16; ++u) part[cg * ldp + rg * 16 + u] = acc[u];
    }
    __syncthreads();
    for (int i = tid; i < n; i += NT) {
        float s = 0.f;
        for (int qq = 0; qq < CG; ++qq) s += part[qq * ldp + i];
        z[off + (i / g) * nth + i % g] = s;
    }
}

// z = B r from the FP8 (or FP4) pool, one wavefront per block of at most 128 rows
// (the register-built blocks), four blocks per workgroup: lane (rg, cg),
// rg = lane mod RG (RG = ldp / 16 row groups of 16), owns rows
// 16 rg .. 16 rg + 15 and columns cg, cg + CG, ... (CG = 64 / RG, at most 16
// columns per lane), all its 16-byte code loads and r entries in flight
// together; the CG partial sums of a row are added in a per-wave LDS tile.
// A quarter of the threads per block of k_bj_apply_fp8 and no block-wide
// barrier, so more blocks' loads are in flight per CU.  LOOP: the grid holds
// at most seven workgroups per CU and each wavefront applies blocks b,
// b + W, ... (W wavefronts in the grid), the next block's descriptor loaded
// while the current block is applied; taken for pools that fit the 256 MB
// last-level cache (FP4 on 16,384 blocks of 125: 26.9 against 28.5 us).
// Streaming from HBM, one block per wavefront was faster (FP4 on 65,536
// blocks of 125: 110 against 120 us).
constexpr int BJ_W_MAXN = 128;
constexpr int BJ_W_KMAX = 16;      // columns per lane: ceil(n / CG) <= 16 for n <= 128
constexpr int BJ_W_WAVES = 4;
template <typename RT = float, int BITS = 8, bool LOOP = false>
__global__ __launch_bounds__(64 * BJ_W_WAVES) void k_bj_apply_fp8_w(
    DevMesh m, const int64_t *off8, const int64_t *soff, const int4 *__restrict__ apd, int nblk,
    const uint8_t *__restrict__ inv, const float *__restrict__ scales,
    const RT *__restrict__ r, float *__restrict__ z) {
    __shared__ float part[BJ_W_WAVES][BJ_W_MAXN * 8];   // CG x ldp <= 1024 per wave
    __shared__ float rsh[BJ_W_WAVES][BJ_W_MAXN];        // r_j s_j of the block
    const int wave = LOOP ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    const int nw = LOOP ? gridDim.x * BJ_W_WAVES : nblk;
    int b = blockIdx.x * BJ_W_WAVES + wave;
    if (b >= nblk) return;                               // whole waves; no block barrier below
    int4 dcur = apd[b];
    int64_t o8cur = off8[b], socur = soff[b];
    for (; b < nblk; b += nw) {
        // the next block's descriptor in flight while this one is applied
        int4 dnx = dcur;
        int64_t o8nx = o8cur, sonx = socur;
        if constexpr (LOOP) {
            const int bn = b + nw < nblk ? b + nw : b;
            dnx = apd[bn];
            o8nx = off8[bn];
            sonx = soff[bn];
        }
        const int4 d = dcur;                  // n, first DOF, cell angles, angles g
        const int n = d.x, nth = d.z, g = d.w;
        const int ldp = (n + 15) / 16 * 16, RG = ldp / 16, CG = 64 / RG;
        const int rg = lane % RG, cg = lane / RG;
        const int off = d.y;
        typedef BjCodes<BITS> Codes;
        typedef typename Codes::V CV;
        const CV *B = reinterpret_cast<const CV *>(inv + (o8cur >> Codes::SHIFT)) + rg;
        const int ldq = ldp / 16;
        const float *sc = scales + socur;
        // r_j s_j once per block entry (two per lane)
        float *rs = rsh[wave];
        for (int i = lane; i < n; i += 64) rs[i] = float(r[off + (i / g) * nth + i % g]) * sc[i];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        float acc[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[v] = 0.f;
        // FP8: two batches of eight columns, each batch's loads in flight
        // together (all sixteen at once: 132 VGPRs, three waves per SIMD,
        // slower); FP4: the half-size loads of all sixteen columns at once
        constexpr int BATCH = BITS == 4 ? BJ_W_KMAX : BJ_W_KMAX / 2;
#pragma unroll 1
        for (int u0 = 0; u0 < BJ_W_KMAX; u0 += BATCH) {
            CV q[BATCH];
            float rj[BATCH];
#pragma unroll
            for (int u = 0; u < BATCH; ++u) {
                const int j = cg + (u0 + u) * CG;
                const bool ok = cg < CG && j < n;
                q[u] = ok ? B[size_t(j) * ldq] : Codes::zero();
                rj[u] = ok ? rs[j] : 0.f;
            }
#pragma unroll
            for (int u = 0; u < BATCH; ++u) Codes::fma16(q[u], rj[u], acc);
        }
        float *pw = part[wave];
        if (cg < CG) {
#pragma unroll
            for (int v = 0; v < 16; ++v) pw[cg * ldp + rg * 16 + v] = acc[v];
        }
        // the wave's own LDS writes, read back by other lanes of the same wave
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        for (int i = lane; i < n; i += 64) {
            float s = 0.f;
            for (int qq = 0; qq < CG; ++qq) s += pw[qq * ldp + i];
            z[off + (i / g) * nth + i % g] = s;
        }
        if constexpr (!LOOP) break;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        dcur = dnx;
        o8cur = o8nx;
        socur = sonx;
    }
}

}  // namespace rtx

using namespace rtx;

extern "C" int rtx_bjacobi_size(rtx_plan *p, int64_t *n_entries) {
    RTX_CHECK(p && n_entries, "rtx_bjacobi_size: null argument");
    const int split = (p->bj_method != 0) ? 1 : 0;
    if (p->bj_off && p->bj_split == split) {      // the plan's mesh never changes
        *n_entries = p->bj_entries;
        return RTX_OK;
    }
    std::vector<int32_t> nx(p->m.ncol), ny(p->m.ncol), cc(p->m.ncell), nt(p->m.ncell);
    RTX_HIP(hipMemcpy(nx.data(), p->m.col_nx, nx.size() * 4, hipMemcpyDeviceToHost));
    RTX_HIP(hipMemcpy(ny.data(), p->m.col_ny, ny.size() * 4, hipMemcpyDeviceToHost));
    RTX_HIP(hipMemcpy(cc.data(), p->m.cell_col, cc.size() * 4, hipMemcpyDeviceToHost));
    RTX_HIP(hipMemcpy(nt.data(), p->m.cell_nth, nt.size() * 4, hipMemcpyDeviceToHost));
    std::vector<int32_t> dof0(p->m.ncell);
    RTX_HIP(hipMemcpy(dof0.data(), p->m.cell_dof_off, dof0.size() * 4, hipMemcpyDeviceToHost));
    std::vector<int32_t> blk, apd, cls[BJ_NCLS];
    std::vector<int64_t> off(1, 0), off16(1, 0), off8(1, 0), soff(1, 0);
    int32_t maxb = 0;
    for (int k = 0; k < p->m.ncell; ++k) {
        const int nsp = nx[cc[k]] * ny[cc[k]], nth = nt[k];
        const int g = (split && nsp * nth > BJ_SPLIT) ? std::max(1, BJ_SPLIT / nsp) : nth;
        for (int a0 = 0; a0 < nth; a0 += g) {
            const int gg = std::min(g, nth - a0);
            const int64_t n = int64_t(nsp) * gg;
            blk.push_back(k);
            blk.push_back(a0);
            blk.push_back(gg);
            apd.push_back(int32_t(n));
            apd.push_back(dof0[k] + a0);
            apd.push_back(nth);
            apd.push_back(gg);
            cls[std::min<int64_t>((n - 1) / 16, BJ_NCLS - 1)].push_back(int32_t(blk.size() / 3 - 1));
            off.push_back(off.back() + n * n);
            off16.push_back(off16.back() + n * ((n + 7) / 8 * 8));
            off8.push_back(off8.back() + n * ((n + 15) / 16 * 16));
            soff.push_back(soff.back() + n);
            maxb = std::max<int32_t>(maxb, int32_t(n));
        }
    }
    p->bj_split = -1;
    if (p->bj_off) RTX_HIP(hipFree(p->bj_off));
    if (p->bj_off16) RTX_HIP(hipFree(p->bj_off16));
    if (p->bj_off8) RTX_HIP(hipFree(p->bj_off8));
    if (p->bj_soff) RTX_HIP(hipFree(p->bj_soff));
    if (p->bj_blk) RTX_HIP(hipFree(p->bj_blk));
    if (p->bj_apd) RTX_HIP(hipFree(p->bj_apd));
    if (p->bj_cls) RTX_HIP(hipFree(p->bj_cls));
    p->bj_off = p->bj_off16 = p->bj_off8 = p->bj_soff = nullptr;
    p->bj_blk = p->bj_apd = p->bj_cls = nullptr;
    RTX_HIP(hipMalloc(&p->bj_off, off.size() * sizeof(int64_t)));
    RTX_HIP(hipMemcpy(p->bj_off, off.data(), off.size() * sizeof(int64_t),
                      hipMemcpyHostToDevice));
    RTX_HIP(hipMalloc(&p->bj_off16, off16.size() * sizeof(int64_t)));
    RTX_HIP(hipMemcpy(p->bj_off16, off16.data(), off16.size() * sizeof(int64_t),
                      hipMemcpyHostToDevice));
    RTX_HIP(hipMalloc(&p->bj_off8, off8.size() * sizeof(int64_t)));
    RTX_HIP(hipMemcpy(p->bj_off8, off8.data(), off8.size() * sizeof(int64_t),
                      hipMemcpyHostToDevice));
    RTX_HIP(hipMalloc(&p->bj_soff, soff.size() * sizeof(int64_t)));
    RTX_HIP(hipMemcpy(p->bj_soff, soff.data(), soff.size() * sizeof(int64_t),
                      hipMemcpyHostToDevice));
    RTX_HIP(hipMalloc(&p->bj_blk, blk.size() * sizeof(int32_t)));
    RTX_HIP(hipMemcpy(p->bj_blk, blk.data(), blk.size() * sizeof(int32_t),
                      hipMemcpyHostToDevice));
    RTX_HIP(hipMalloc(&p->bj_apd, apd.size() * sizeof(int32_t)));
    RTX_HIP(hipMemcpy(p->bj_apd, apd.data(), apd.size() * sizeof(int32_t),
                      hipMemcpyHostToDevice));
    std::vector<int32_t> all;
    for (int q = 0; q < BJ_NCLS; ++q) {
        p->bj_cls_start[q] = int32_t(all.size());
        all.insert(all.end(), cls[q].begin(), cls[q].end());
    }
    p->bj_cls_start[BJ_NCLS] = int32_t(all.size());
    RTX_HIP(hipMalloc(&p->bj_cls, std::max<size_t>(all.size(), 1) * sizeof(int32_t)));
    if (!all.empty())
        RTX_HIP(hipMemcpy(p->bj_cls, all.data(), all.size() * sizeof(int32_t),
                          hipMemcpyHostToDevice));
    p->bj_split = split;
    p->bj_ready = false;
    p->bj_nblk = int32_t(blk.size() / 3);
    p->bj_max_block = maxb;
    p->bj_entries = off.back();
    p->bj_entries16 = off16.back();
    p->bj_codes8 = (off8.back() + 15) / 16 * 16;
    p->bj_bytes8 = p->bj_codes8 + soff.back() * int64_t(sizeof(float));
    p->bj_codes4 = (off8.back() / 2 + 15) / 16 * 16;
    p->bj_bytes4 = p->bj_codes4 + soff.back() * int64_t(sizeof(float));
    *n_entries = off.back();
    return RTX_OK;
}

extern "C" int rtx_bjacobi_size_fp8(rtx_plan *p, int64_t *n_bytes) {
    RTX_CHECK(p && n_bytes, "rtx_bjacobi_size_fp8: null argument");
    if (!p->bj_off8) {
        int64_t n;
        const int rc = rtx_bjacobi_size(p, &n);
        if (rc) return rc;
    }
    *n_bytes = p->bj_bytes8;
    return RTX_OK;
}

extern "C" int rtx_bjacobi_pack_fp8(rtx_plan *p, const float *d_inv32, uint8_t *d_inv8,
                                    void *stream) {
    RTX_CHECK(p && d_inv32 && d_inv8, "rtx_bjacobi_pack_fp8: null argument");
    RTX_CHECK(p->bj_off8 && p->bj_nblk > 0, "rtx_bjacobi_pack_fp8: call rtx_bjacobi_size first");
    k_bj_pack_fp8<<<p->bj_nblk, BJ_THREADS, 0, static_cast<hipStream_t>(stream)>>>(
        p->m, p->bj_off, p->bj_off8, p->bj_soff, p->bj_blk, d_inv32, d_inv8,
        reinterpret_cast<float *>(d_inv8 + p->bj_codes8));
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

extern "C" int rtx_bjacobi_size_fp4(rtx_plan *p, int64_t *n_bytes) {
    RTX_CHECK(p && n_bytes, "rtx_bjacobi_size_fp4: null argument");
    if (!p->bj_off8) {
        int64_t n;
        const int rc = rtx_bjacobi_size(p, &n);
        if (rc) return rc;
    }
    *n_bytes = p->bj_bytes4;
    return RTX_OK;
}

extern "C" int rtx_bjacobi_pack_fp4(rtx_plan *p, const float *d_inv32, uint8_t *d_inv4,
                                    void *stream) {
    RTX_CHECK(p && d_inv32 && d_inv4, "rtx_bjacobi_pack_fp4: null argument");
    RTX_CHECK(p->bj_off8 && p->bj_nblk > 0, "rtx_bjacobi_pack_fp4: call rtx_bjacobi_size first");
    k_bj_pack_fp4<<<p->bj_nblk, BJ_THREADS, 0, static_cast<hipStream_t>(stream)>>>(
        p->m, p->bj_off, p->bj_off8, p->bj_soff, p->bj_blk, d_inv32, d_inv4,
        reinterpret_cast<float *>(d_inv4 + p->bj_codes4));
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

/* Entries (uint16) of the packed BF16 inverse pool. */
extern "C" int rtx_bjacobi_size_bf16(rtx_plan *p, int64_t *n_entries) {
    RTX_CHECK(p && n_entries, "rtx_bjacobi_size_bf16: null argument");
    if (!p->bj_off16) {
        int64_t n;
        const int rc = rtx_bjacobi_size(p, &n);
        if (rc) return rc;
    }
    *n_entries = p->bj_entries16;
    return RTX_OK;
}

/* Round the FP32 inverses to BF16 (nearest even) into the packed layout. */
extern "C" int rtx_bjacobi_pack_bf16(rtx_plan *p, const float *d_inv32, uint16_t *d_inv16,
                                     void *stream) {
    RTX_CHECK(p && d_inv32 && d_inv16, "rtx_bjacobi_pack_bf16: null argument");
    RTX_CHECK(p->bj_off16 && p->bj_nblk > 0, "rtx_bjacobi_pack_bf16: call rtx_bjacobi_size first");
    k_bj_pack_bf16<<<p->bj_nblk, BJ_THREADS, 0, static_cast<hipStream_t>(stream)>>>(
        p->m, p->bj_off, p->bj_off16, p->bj_blk, d_inv32, d_inv16);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

// The register build, each size class (steps of 16 DOFs, one wave per 16) on
// the kernel that holds it, the largest blocks first: the small classes fill
// the tail.
template <typename T, int BITS, typename O>
static void launch_bj_build(const rtx_plan *p, int restrict_interior, const int64_t *off, O *out,
                            float *scales, int *d_status, hipStream_t st) {
    const int32_t *cs = p->bj_cls, *c0 = p->bj_cls_start;
    auto build = [&](auto nt) {
        constexpr int NT = decltype(nt)::value;
        const int cnt = c0[NT] - c0[NT - 1];
        if (cnt)
            k_bj_build_reg<NT, T, BITS><<<cnt, 64 * NT, 0, st>>>(
                p->m, restrict_interior, off, p->bj_blk, cs + c0[NT - 1], out, p->bj_soff, scales,
                d_status);
    };
    build(std::integral_constant<int, 8>());
    build(std::integral_constant<int, 7>());
    build(std::integral_constant<int, 6>());
    build(std::integral_constant<int, 5>());
    build(std::integral_constant<int, 4>());
    build(std::integral_constant<int, 3>());
    build(std::integral_constant<int, 2>());
    build(std::integral_constant<int, 1>());
}

// Wait for a build and read its status: the 1-based cell of a singular block.
static int bj_build_status(rtx_plan *p, int *d_status, hipStream_t st, const char *who) {
    int h_status = 0;
    RTX_HIP(hipMemcpyAsync(&h_status, d_status, sizeof(int), hipMemcpyDeviceToHost, st));
    RTX_HIP(hipStreamSynchronize(st));
    RTX_HIP(hipFreeAsync(d_status, st));
    if (h_status) {
        set_error("%s: singular diagonal block in cell %d", who, h_status - 1);
        return RTX_ERR_NUMERIC;
    }
    p->bj_ready = true;
    return RTX_OK;
}

extern "C" int rtx_bjacobi_factor(rtx_plan *p, int restrict_interior, double *d_inv,
                                  float *d_inv_f32, double *d_scratch, void *stream) {
    RTX_CHECK(p && (d_inv || d_inv_f32), "rtx_bjacobi_factor: null argument");
    if (!p->has_coeffs) {
        set_error("rtx_bjacobi_factor: coefficients not set");
        return RTX_ERR_STATE;
    }
    if (!p->bj_off || p->bj_split != ((p->bj_method != 0) ? 1 : 0)) {
        int64_t n;
        int rc = rtx_bjacobi_size(p, &n);
        if (rc) return rc;
    }
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int64_t nmax = p->bj_max_block;
    const size_t lds = size_t(nmax) * nmax * sizeof(double);
    int dev = 0, max_lds = 0;
    RTX_HIP(hipGetDevice(&dev));
    RTX_HIP(hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    const size_t static_lds = 2 * NMq * 8 + RTX_NMAX * RTX_NMAX * RTX_NMAX * 12 + 16;
    int *d_status = nullptr;
    RTX_HIP(hipMallocAsync((void **)&d_status, sizeof(int), st));
    RTX_HIP(hipMemsetAsync(d_status, 0, sizeof(int), st));
    const bool reg = p->bj_method != 0 && nmax <= 128;
    // no FP64 inverse wanted: the register build eliminates in FP32 straight
    // into d_inv_f32 (the FP32, BF16, FP8 and FP4 copies all start there)
    const bool f32_only = d_inv == nullptr;
    if (f32_only && !reg) {
        (void)hipFreeAsync(d_status, st);
        set_error("rtx_bjacobi_factor: an FP32-only factorisation needs the register build "
                  "(blocks of up to 128 DOFs, method -1 or 1); blocks of %lld DOFs",
                  (long long)nmax);
        return RTX_ERR_ARG;
    }
    if (reg && f32_only)
        launch_bj_build<float, 0>(p, restrict_interior, p->bj_off, d_inv_f32, nullptr, d_status, st);
    else if (reg) {
        launch_bj_build<double, 0>(p, restrict_interior, p->bj_off, d_inv, nullptr, d_status, st);
    } else if (p->bj_method == 1) {
        (void)hipFreeAsync(d_status, st);
        set_error("rtx_bjacobi_factor: the register build handles blocks of up to 128 DOFs, "
                  "not %lld", (long long)nmax);
        return RTX_ERR_ARG;
    } else if (lds + static_lds <= size_t(max_lds)) {
        RTX_HIP(hipFuncSetAttribute((const void *)k_bj_build<true>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
        k_bj_build<true><<<p->m.ncell, BJ_THREADS, lds, st>>>(p->m, restrict_interior, p->bj_off,
                                                            d_inv, nullptr, d_status);
    } else {
        if (d_scratch == nullptr) {
            (void)hipFreeAsync(d_status, st);
            set_error("rtx_bjacobi_factor: blocks of %lld DOFs do not fit LDS; a scratch buffer "
                      "of the same size as the inverses is required",
                      (long long)nmax);
            return RTX_ERR_ARG;
        }
        k_bj_build<false><<<p->m.ncell, BJ_THREADS, 0, st>>>(p->m, restrict_interior, p->bj_off,
                                                           d_inv, d_scratch, d_status);
    }
    RTX_HIP(hipGetLastError());
    if (d_inv_f32 && !f32_only)
        k_to_f32_bj<<<2048, 256, 0, st>>>(d_inv, d_inv_f32, p->bj_entries);
    return bj_build_status(p, d_status, st, "rtx_bjacobi_factor");
}

extern "C" int rtx_bjacobi_factor_coded(rtx_plan *p, int restrict_interior, int precision,
                                        uint8_t *d_codes, void *stream) {
    RTX_CHECK(p && d_codes, "rtx_bjacobi_factor_coded: null argument");
    RTX_CHECK(precision == RTX_PREC_FP8 || precision == RTX_PREC_FP4,
              "rtx_bjacobi_factor_coded: precision must be RTX_PREC_FP8 or RTX_PREC_FP4, not %d",
              precision);
    if (!p->has_coeffs) {
        set_error("rtx_bjacobi_factor_coded: coefficients not set");
        return RTX_ERR_STATE;
    }
    int64_t n;
    if (const int rc = rtx_bjacobi_size(p, &n)) return rc;
    RTX_CHECK(p->bj_method != 0 && p->bj_max_block <= BJ_SPLIT,
              "rtx_bjacobi_factor_coded: the FP32-only factorisation needs the register build "
              "(blocks of up to 128 DOFs, method -1 or 1); blocks of %d DOFs",
              int(p->bj_max_block));
    hipStream_t st = static_cast<hipStream_t>(stream);
    int *d_status = nullptr;
    RTX_HIP(hipMallocAsync((void **)&d_status, sizeof(int), st));
    RTX_HIP(hipMemsetAsync(d_status, 0, sizeof(int), st));
    if (precision == RTX_PREC_FP8)
        launch_bj_build<float, 8>(p, restrict_interior, p->bj_off8, d_codes,
                                  reinterpret_cast<float *>(d_codes + p->bj_codes8), d_status, st);
    else
        launch_bj_build<float, 4>(p, restrict_interior, p->bj_off8, d_codes,
                                  reinterpret_cast<float *>(d_codes + p->bj_codes4), d_status, st);
    RTX_HIP(hipGetLastError());
    return bj_build_status(p, d_status, st, "rtx_bjacobi_factor_coded");
}

extern "C" int rtx_bjacobi_set_method(rtx_plan *p, int method) {
    RTX_CHECK(p && method >= -1 && method <= 1, "rtx_bjacobi_set_method: method must be -1, 0 or 1");
    p->bj_method = method;
    return RTX_OK;
}

// The FP8 / FP4 applies: the wavefront-per-block kernel for blocks of at
// most BJ_W_MAXN rows, else the slab kernel; r of type RT, z FP32.
template <int BITS, typename RT>
static void launch_bj_coded(const rtx_plan *p, const void *d_inv, const RT *r, float *z,
                            hipStream_t st) {
    const uint8_t *codes = static_cast<const uint8_t *>(d_inv);
    const float *scales =
        reinterpret_cast<const float *>(codes + (BITS == 4 ? p->bj_codes4 : p->bj_codes8));
    const int4 *apd = reinterpret_cast<const int4 *>(p->bj_apd);
    const int nwg = (p->bj_nblk + BJ_W_WAVES - 1) / BJ_W_WAVES;
    if (p->bj_max_block <= BJ_W_MAXN && (BITS == 4 ? p->bj_bytes4 : p->bj_bytes8) <= (int64_t(256) << 20))
        k_bj_apply_fp8_w<RT, BITS, true><<<std::min(nwg, std::max(7 * p->n_cu, 1)),
                                           64 * BJ_W_WAVES, 0, st>>>(
            p->m, p->bj_off8, p->bj_soff, apd, p->bj_nblk, codes, scales, r, z);
    else if (p->bj_max_block <= BJ_W_MAXN)
        k_bj_apply_fp8_w<RT, BITS, false><<<nwg, 64 * BJ_W_WAVES, 0, st>>>(
            p->m, p->bj_off8, p->bj_soff, apd, p->bj_nblk, codes, scales, r, z);
    else
        k_bj_apply_fp8<BJ_APPLY8_THREADS, RT, BITS><<<p->bj_nblk, BJ_APPLY8_THREADS, 0, st>>>(
            p->m, p->bj_off8, p->bj_soff, apd, codes, scales, r, z);
}

extern "C" int rtx_bjacobi_apply(rtx_plan *p, int precision, const void *d_inv, const void *d_r,
                                 void *d_z, void *stream) {
    RTX_CHECK(p && d_inv && d_r && d_z, "rtx_bjacobi_apply: null argument");
    RTX_CHECK(d_r != d_z, "rtx_bjacobi_apply: r and z must not alias");
    if (!p->bj_ready) {
        set_error("rtx_bjacobi_apply: call rtx_bjacobi_factor first");
        return RTX_ERR_STATE;
    }
    const int4 *apd = reinterpret_cast<const int4 *>(p->bj_apd);
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (precision == RTX_PREC_F64)
        k_bj_apply<double, double><<<p->bj_nblk, BJ_THREADS, 0, st>>>(
            p->m, p->bj_off, apd, (const double *)d_inv, (const double *)d_r, (double *)d_z);
    else if (precision == RTX_PREC_F32)
        k_bj_apply<float, float><<<p->bj_nblk, BJ_THREADS, 0, st>>>(
            p->m, p->bj_off, apd, (const float *)d_inv, (const float *)d_r, (float *)d_z);
    else if (precision == RTX_PREC_MIXED)
        k_bj_apply_bf16<BJ_APPLY16_THREADS><<<p->bj_nblk, BJ_APPLY16_THREADS, 0, st>>>(
            p->m, p->bj_off16, apd, (const uint16_t *)d_inv, (const float *)d_r,
            (float *)d_z);
    else if (precision == RTX_PREC_FP8)
        launch_bj_coded<8, float>(p, d_inv, (const float *)d_r, (float *)d_z, st);
    else if (precision == RTX_PREC_FP4)
        launch_bj_coded<4, float>(p, d_inv, (const float *)d_r, (float *)d_z, st);
    else {
        set_error("rtx_bjacobi_apply: unsupported precision %d", precision);
        return RTX_ERR_ARG;
    }
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

/* z = M r with the FP8 (RTX_PREC_FP8) or FP4 (RTX_PREC_FP4) inverses, r in
   FP16 (IEEE binary16) and z in FP32: the preconditioner of GMRES on an
   FP16 basis.  Same inverses and arithmetic as rtx_bjacobi_apply; only the
   input type differs. */
extern "C" int rtx_bjacobi_apply_h(rtx_plan *p, int precision, const void *d_inv, const void *d_r,
                                   void *d_z, void *stream) {
    RTX_CHECK(p && d_inv && d_r && d_z, "rtx_bjacobi_apply_h: null argument");
    RTX_CHECK(d_r != d_z, "rtx_bjacobi_apply_h: r and z must not alias");
    RTX_CHECK(precision == RTX_PREC_FP8 || precision == RTX_PREC_FP4,
              "rtx_bjacobi_apply_h: precision must be RTX_PREC_FP8 or RTX_PREC_FP4, not %d",
              precision);
    if (!p->bj_ready) {
        set_error("rtx_bjacobi_apply_h: call rtx_bjacobi_factor first");
        return RTX_ERR_STATE;
    }
    RTX_CHECK(p->bj_off8, "rtx_bjacobi_apply_h: call rtx_bjacobi_size first");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (precision == RTX_PREC_FP8)
        launch_bj_coded<8, _Float16>(p, d_inv, (const _Float16 *)d_r, (float *)d_z, st);
    else
        launch_bj_coded<4, _Float16>(p, d_inv, (const _Float16 *)d_r, (float *)d_z, st);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

extern "C" int rtx_bjacobi_apply_fp8_h(rtx_plan *p, const void *d_inv, const void *d_r, void *d_z,
                                       void *stream) {
    return rtx_bjacobi_apply_h(p, RTX_PREC_FP8, d_inv, d_r, d_z, stream);
}
