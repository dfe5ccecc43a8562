// Krylov building blocks for the device-resident GMRES.
//
// The reference hands the assembled interior system to PETSc KSP
// (src/rt/solve.py:81-100: GMRES(50), which orthogonalises with classical
// Gram-Schmidt).  Here one Arnoldi step (classical Gram-Schmidt with a
// device-side "twice is enough" re-orthogonalisation test, then
// normalisation) is a fixed sequence of fused FP64 kernels over the tall
// basis V; reductions are two-phase and deterministic (per-block partial
// sums, then one reduction per output).
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "rtx_internal.h"

namespace rtx {

constexpr int KT = 256;          // threads per block
constexpr int KW = KT / 64;      // wavefronts per block
constexpr int KCH = 8;           // basis vectors per mdot block (gridDim.y chunks)
constexpr int KNB = 1024;        // most row blocks of the tall-skinny kernels
constexpr int KMAXV = 256;       // largest basis handled by one Arnoldi step
constexpr double REORTH = 0.5;   // re-orthogonalise when |w'|^2 < 0.5 |w|^2
// state block after the partials (doubles): [0] |w|^2, [1] |w'|^2, [4] flag (int)
constexpr int WORK_TAIL = 16;

// Values per thread and load: 16 bytes of the basis (8 bytes of an FP16 one
// whose rows start on 8 bytes only), or one where rows are not aligned.
template <typename T>
constexpr int kvec() { return 16 / int(sizeof(T)); }

// Row blocks: one pass of the block's threads each, up to KNB (fewer blocks
// leave fewer partial sums to add; more would be nearly empty).
static int row_blocks(int64_t n, int vw) {
    const int64_t per = int64_t(KT) * vw;
    return int(std::max<int64_t>(1, std::min<int64_t>(KNB, (n + per - 1) / per)));
}

// N sums over a wavefront at once (N = 8): each step halves the values a
// lane carries, 10 exchanges instead of 6 N.  Lane l returns the sum of value
// bit-reversed(l / 8): 4 (l >> 5 & 1) + 2 (l >> 4 & 1) + (l >> 3 & 1).
__device__ inline double wave_sum8(double (&v)[8], int lane) {
#pragma unroll
    for (int h = 4, off = 32; h > 0; h >>= 1, off >>= 1) {
        const bool up = lane & off;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (j < h) {
                const double keep = up ? v[j + h] : v[j], send = up ? v[j] : v[j + h];
                v[j] = keep + __shfl_xor(send, off);
            }
    }
    double r = v[0];
#pragma unroll
    for (int off = 4; off > 0; off >>= 1) r += __shfl_xor(r, off);
    return r;
}

// Sum over the block in a fixed order, for every thread (sh: KW doubles).
__device__ inline double block_sum1(double v, double *sh) {
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = sh[0];
#pragma unroll
    for (int w = 1; w < KW; ++w) t += sh[w];
    return t;
}

// VW consecutive values, loaded and stored 16 bytes at a time (8 for four FP16
// values); the caller checks the alignment.
template <typename T, int VW> struct KVec {
    T v[VW];
};
template <typename T, int VW>
constexpr int kelem() { return VW * int(sizeof(T)) > 16 ? 16 / int(sizeof(T)) : VW; }

template <typename T, int VW>
__device__ inline KVec<T, VW> ldv(const T *p) {
    KVec<T, VW> o;
    if constexpr (VW == 1) {
        o.v[0] = p[0];
    } else {
        constexpr int E = kelem<T, VW>();
        typedef T V __attribute__((ext_vector_type(E)));
#pragma unroll
        for (int u = 0; u < VW / E; ++u) {
            const V q = *reinterpret_cast<const V *>(p + u * E);
#pragma unroll
            for (int e = 0; e < E; ++e) o.v[u * E + e] = q[e];
        }
    }
    return o;
}
template <typename T, int VW>
__device__ inline void stv(T *p, const T (&v)[VW]) {
    if constexpr (VW == 1) {
        p[0] = v[0];
    } else {
        constexpr int E = kelem<T, VW>();
        typedef T V __attribute__((ext_vector_type(E)));
#pragma unroll
        for (int u = 0; u < VW / E; ++u) {
            V q;
#pragma unroll
            for (int e = 0; e < E; ++e) q[e] = v[u * E + e];
            *reinterpret_cast<V *>(p + u * E) = q;
        }
    }
}
// a double rounded to a basis storage type (FP16 through FP32)
template <typename T>
__device__ inline T to_store(double x) {
    if constexpr (std::is_same<T, _Float16>::value) return _Float16(float(x));
    else return T(x);
}

// Row range of block b, starting on a multiple of VW.
template <int VW>
__device__ inline void row_range(int64_t n, int b, int nb, int64_t &i0, int64_t &i1) {
    int64_t per = (n + nb - 1) / nb;
    per = (per + VW - 1) / VW * VW;
    i0 = int64_t(b) * per;
    i1 = (i0 + per < n) ? i0 + per : n;
    if (i0 > n) i0 = n;
}

// One block's dot products with NJ basis vectors: the loads of a pass are
// independent (NJ is compiled in: a test per vector would make each load wait
// for the one before).
template <typename T, int VW, typename TW, int NJ>
__device__ inline void mdot_rows(const T *V, int64_t ld, const TW *w, int64_t i0, int64_t i1,
                                 double (&acc)[KCH], double &ww) {
    const int64_t nq = (i1 - i0) / VW;
    for (int64_t q = threadIdx.x; q < nq; q += KT) {
        const int64_t i = i0 + VW * q;
        const KVec<TW, VW> wv = ldv<TW, VW>(w + i);
        KVec<T, VW> vv[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) vv[j] = ldv<T, VW>(V + j * ld + i);
#pragma unroll
        for (int e = 0; e < VW; ++e) {
            const double we = double(wv.v[e]);
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[j] += double(vv[j].v[e]) * we;
            ww += we * we;
        }
    }
    const int64_t i = i0 + VW * nq + threadIdx.x;       // fewer than VW rows past the passes
    if (VW > 1 && i < i1) {
        const double wi = double(w[i]);
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[j] += double(V[j * ld + i]) * wi;
        ww += wi * wi;
    }
}

// partial[j * nb + b] = sum over block b's rows of V_j[i] w[i], j < nv;
// if with_ww, partial[nv * nb + b] = sum w[i]^2 (computed by chunk 0).
//
// Bound by reading V where n is large; one pass of loads and the sums over
// the block where it is not.  2,048,000 rows, FP16, 1 to 15 vectors: 12.0 ->
// 10.9 us on average; 65,536 rows, FP64, 1 to 50 vectors: 15.8 -> 5.8 us
// (1,024 blocks of 64 rows and a tree of eight barriers before).
template <typename T, int VW, typename TW = T>
__global__ __launch_bounds__(KT) void k_mdot(const T *__restrict__ V, int64_t ld, int nv,
                                             const TW *__restrict__ w, int64_t n, int nb,
                                             double *__restrict__ partial, int with_ww,
                                             const int *__restrict__ skip) {
    if (skip && *skip) return;
    __shared__ double sh[KW][KCH + 1];
    // workgroups go to the XCDs round-robin: the chunks of row block b one after
    // another on XCD b % 8 (where k_update's block b runs too), so that w is
    // read from memory once
    const int nch = (nv + KCH - 1) / KCH, slot = blockIdx.x / 8;
    const int b = slot / nch * 8 + blockIdx.x % 8;
    const int chunk = slot % nch, j0 = chunk * KCH, nj = min(nv - j0, KCH);
    if (b >= nb) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int64_t i0, i1;
    row_range<VW>(n, b, nb, i0, i1);
    double acc[KCH] = {0.0}, ww = 0.0;
    const T *Vj = V + int64_t(j0) * ld;
    switch (nj) {
#define KCASE(NJ)                                                   \
    case NJ:                                                        \
        mdot_rows<T, VW, TW, NJ>(Vj, ld, w, i0, i1, acc, ww);       \
        break;
        KCASE(1) KCASE(2) KCASE(3) KCASE(4) KCASE(5) KCASE(6) KCASE(7) KCASE(8)
#undef KCASE
    }
    const double s = wave_sum8(acc, lane);
    if ((lane & 7) == 0)
        sh[wave][((lane >> 5) & 1) * 4 + ((lane >> 4) & 1) * 2 + ((lane >> 3) & 1)] = s;
    const bool sq = with_ww && chunk == 0;
    if (sq) {
        ww = wave_sum(ww);
        if (lane == 0) sh[wave][KCH] = ww;
    }
    __syncthreads();
    if (tid < nj || (sq && tid == KCH)) {
        double t = sh[0][tid];
#pragma unroll
        for (int v = 1; v < KW; ++v) t += sh[v][tid];
        partial[int64_t(tid == KCH ? nv : j0 + tid) * nb + b] = t;
    }
}

// out[j] (+)= sum_b partial[j * nb + b], nb <= KNB; one wavefront per j.
__global__ __launch_bounds__(KT) void k_reduce(const double *__restrict__ partial, int nb, int nj,
                                               double *__restrict__ out, int accumulate,
                                               const int *__restrict__ skip) {
    if (skip && *skip) return;
    const int j = blockIdx.x * KW + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (j >= nj) return;
    const double *p = partial + int64_t(j) * nb;
    double v = 0.0;
#pragma unroll
    for (int u = 0; u < KNB / 64; ++u)
        v += keep_if(p[min(lane + 64 * u, nb - 1)], lane + 64 * u < nb);
    v = wave_sum(v);
    if (lane == 0) out[j] = accumulate ? out[j] + v : v;
}

// acc -= V h at VW rows from i: eight (then four) basis vectors' loads at a
// time; past the last one the last vector again with a zero factor.
template <typename T, int VW>
__device__ inline void subtract_rows(const T *V, int64_t ld, int nv, const double *hs, int64_t i,
                                     double (&acc)[VW]) {
    int j = 0;
    const auto some = [&](auto cnt) {
        constexpr int N = decltype(cnt)::value;
        KVec<T, VW> vv[N];
#pragma unroll
        for (int u = 0; u < N; ++u) vv[u] = ldv<T, VW>(V + int64_t(min(j + u, nv - 1)) * ld + i);
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const double h = j + u < nv ? hs[j + u] : 0.0;
#pragma unroll
            for (int e = 0; e < VW; ++e) acc[e] -= double(vv[u].v[e]) * h;
        }
        j += N;
    };
    while (j + 8 <= nv) some(std::integral_constant<int, 8>());
    while (j < nv) some(std::integral_constant<int, 4>());
}

// w -= V h (nv vectors); partial[b] = sum over block b of the new w^2
// (accumulated in FP64 for either storage type).
template <typename T, int VW>
__global__ __launch_bounds__(KT) void k_update(const T *__restrict__ V, int64_t ld, int nv,
                                               const double *__restrict__ h,
                                               T *__restrict__ w, int64_t n,
                                               double *__restrict__ partial,
                                               const int *__restrict__ skip) {
    if (skip && *skip) return;
    __shared__ double hs[KMAXV];
    __shared__ double sh[KW];
    for (int j = threadIdx.x; j < nv; j += KT) hs[j] = h[j];
    __syncthreads();
    const int b = blockIdx.x, nb = gridDim.x;
    int64_t i0, i1;
    row_range<VW>(n, b, nb, i0, i1);
    double ss = 0.0;
    const int64_t nq = (i1 - i0) / VW;
    for (int64_t q = threadIdx.x; q < nq; q += KT) {
        const int64_t i = i0 + VW * q;
        const KVec<T, VW> wv = ldv<T, VW>(w + i);
        double acc[VW];
#pragma unroll
        for (int e = 0; e < VW; ++e) acc[e] = double(wv.v[e]);
        subtract_rows<T, VW>(V, ld, nv, hs, i, acc);
        T out[VW];
#pragma unroll
        for (int e = 0; e < VW; ++e) {
            out[e] = T(acc[e]);
            ss += double(out[e]) * double(out[e]);
        }
        stv<T, VW>(w + i, out);
    }
    const int64_t i = i0 + VW * nq + threadIdx.x;
    if (VW > 1 && i < i1) {
        double acc[1] = {double(w[i])};
        subtract_rows<T, 1>(V, ld, nv, hs, i, acc);
        const T wn = T(acc[0]);
        w[i] = wn;
        ss += double(wn) * double(wn);
    }
    ss = block_sum1(ss, sh);
    if (threadIdx.x == 0) partial[b] = ss;
}

// Fold Hessenberg column j (hc[0..j] in LDS, then beta) into the QR
// factorisation of the cycle's least-squares problem (k_gmres_givens's
// recurrence), by one block with the rotations staged in LDS; hc is
// overwritten.
__device__ inline void givens_column(double *hc, double beta, int j, int m, double *state) {
    __shared__ double cs_[KMAXV], sn_[KMAXV];
    double *cs = state, *sn = state + m, *g = state + 2 * m;
    double *Rj = state + 3 * m + 1 + int64_t(j) * m;
    double *Hj = state + 3 * m + 1 + int64_t(m) * m + int64_t(j) * (m + 1);
    double *est = state + 3 * m + 1 + int64_t(m) * m + int64_t(m + 1) * m;
    const int tid = threadIdx.x;
    for (int t = tid; t < j; t += KT) {
        cs_[t] = cs[t];
        sn_[t] = sn[t];
    }
    for (int t = tid; t <= j + 1; t += KT) Hj[t] = t <= j ? hc[t] : beta;
    const double gj = g[j];
    __syncthreads();                 // hc is rotated in place below
    if (tid == 0) {
        double carry = hc[0];
        for (int t = 0; t < j; ++t) {
            const double b = hc[t + 1];
            hc[t] = cs_[t] * carry + sn_[t] * b;
            carry = -sn_[t] * carry + cs_[t] * b;
        }
        const double den = hypot(carry, beta);
        const double c = den != 0.0 ? carry / den : 1.0;
        const double sv = den != 0.0 ? beta / den : 0.0;
        cs[j] = c;
        sn[j] = sv;
        hc[j] = den;
        g[j + 1] = -sv * gj;
        g[j] = c * gj;
        est[j] = fabs(sv * gj);
    }
    __syncthreads();
    for (int t = tid; t <= j; t += KT) Rj[t] = hc[t];
}

// One Arnoldi update for an FP32 basis with the norm taken from the dot
// products: hd[0..nv-1] = V^T w, hd[nv] = |w|^2 (FP64 sums of FP32 data),
// |w'|^2 = |w|^2 - sum h_j^2 (every wavefront computes it, in the same
// order), v_out = (w - V h) / |w'| written directly (w itself is left as it
// was); a relative norm below 1e-6 counts as a breakdown (v_out = 0, h = 0).
// The last block has no rows: it writes hcol[0..nv] and, when state is given,
// folds the column into the Givens factorisation while the others work.
template <typename T, int VW, typename TW = T>
__global__ __launch_bounds__(KT) void k_update_pyth(const T *__restrict__ V, int64_t ld, int nv,
                                                    const double *__restrict__ hd,
                                                    const TW *__restrict__ w,
                                                    T *__restrict__ v_out, int64_t n,
                                                    double *__restrict__ hcol, int j, int m,
                                                    double *state) {
    __shared__ double hs[KMAXV + 1];
    for (int q = threadIdx.x; q <= nv; q += KT) hs[q] = hd[q];
    __syncthreads();
    double hh = 0.0;
    for (int q = threadIdx.x & 63; q < nv; q += 64) hh += hs[q] * hs[q];
    hh = wave_sum(hh);
    const double r2 = hs[nv] - hh;
    const double beta = (r2 > 1e-12 * hs[nv]) ? sqrt(r2) : 0.0;
    const double sc = beta > 0.0 ? 1.0 / beta : 0.0;
    const int b = blockIdx.x, nb = gridDim.x - 1;
    if (b == nb) {
        for (int q = threadIdx.x; q <= nv; q += KT) hcol[q] = q < nv ? hs[q] : beta;
        if (state) givens_column(hs, beta, j, m, state);
        return;
    }
    int64_t i0, i1;
    row_range<VW>(n, b, nb, i0, i1);
    const int64_t nq = (i1 - i0) / VW;
    for (int64_t q = threadIdx.x; q < nq; q += KT) {
        const int64_t i = i0 + VW * q;
        const KVec<TW, VW> wv = ldv<TW, VW>(w + i);
        double acc[VW];
#pragma unroll
        for (int e = 0; e < VW; ++e) acc[e] = double(wv.v[e]);
        subtract_rows<T, VW>(V, ld, nv, hs, i, acc);
        T out[VW];
#pragma unroll
        for (int e = 0; e < VW; ++e) out[e] = to_store<T>(acc[e] * sc);
        stv<T, VW>(v_out + i, out);
    }
    const int64_t i = i0 + VW * nq + threadIdx.x;
    if (VW > 1 && i < i1) {
        double acc[1] = {double(w[i])};
        subtract_rows<T, 1>(V, ld, nv, hs, i, acc);
        v_out[i] = to_store<T>(acc[0] * sc);
    }
}

// state layout (doubles): [0] |w|^2 before projection, [1] |w'|^2 after;
// flag (int) = 1 when the second pass is skipped.
__global__ void k_reorth_test(const double *state, int *flag) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *flag = (state[1] >= REORTH * state[0]) ? 1 : 0;
}

__global__ void k_set_flag(int *flag, int v) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *flag = v;
}

// v_out = w / |w|, |w|^2 the sum of the nrm2 partials (every block adds them,
// in the same order).  The last block has no rows: it sets hcol[nv] = |w| and,
// when state is given, folds Hessenberg column j into the Givens factorisation.
template <typename T>
__global__ __launch_bounds__(KT) void k_normalize(const T *__restrict__ w, T *__restrict__ v_out,
                                                  int64_t n, const double *__restrict__ nrm2,
                                                  int nparts, double *__restrict__ hcol, int nv,
                                                  int j, int m, double *state) {
    __shared__ double sh[KW];
    double v = 0.0;
#pragma unroll
    for (int u = 0; u < KNB / KT; ++u) {
        const int q = threadIdx.x + KT * u;
        v += keep_if(nrm2[min(q, nparts - 1)], q < nparts);
    }
    const double beta = sqrt(block_sum1(v, sh));
    const double s = beta > 0.0 ? 1.0 / beta : 0.0;
    const int nb = gridDim.x - 1;
    if (int(blockIdx.x) == nb) {
        if (threadIdx.x == 0) hcol[nv] = beta;
        if (!state) return;
        __shared__ double hc[KMAXV + 1];
        for (int t = threadIdx.x; t <= j; t += KT) hc[t] = hcol[t];
        __syncthreads();
        givens_column(hc, beta, j, m, state);
        return;
    }
    int64_t i = int64_t(blockIdx.x) * KT + threadIdx.x;
    for (; i < n; i += int64_t(nb) * KT) v_out[i] = T(double(w[i]) * s);
}

// x += sum_j y_j V_j  (y on the device)
template <typename TV, typename TX>
__global__ __launch_bounds__(KT) void k_combine(const TV *__restrict__ V, int64_t ld, int nv,
                                                const double *__restrict__ y,
                                                TX *__restrict__ x, int64_t n, int accumulate) {
    __shared__ double ys[KMAXV];
    for (int j = threadIdx.x; j < nv; j += KT) ys[j] = y[j];
    __syncthreads();
    int64_t i = int64_t(blockIdx.x) * KT + threadIdx.x;
    for (; i < n; i += int64_t(gridDim.x) * KT) {
        double acc = accumulate ? double(x[i]) : 0.0;
        for (int j = 0; j < nv; ++j) acc += double(V[int64_t(j) * ld + i]) * ys[j];
        x[i] = to_store<TX>(acc);
    }
}

// y = a x + b y with x and y of different storage types
template <typename TX, typename TY>
__global__ void k_axpby_mixed(int64_t n, double a, const TX *__restrict__ x, double b,
                              TY *__restrict__ y) {
    int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    for (; i < n; i += int64_t(gridDim.x) * blockDim.x)
        y[i] = to_store<TY>(a * double(x[i]) + (b == 0.0 ? 0.0 : b * double(y[i])));
}

// y = a x + b y (device scalars optional)
template <typename T>
__global__ void k_axpby(int64_t n, double a, const T *__restrict__ x, double b,
                        T *__restrict__ y) {
    int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    for (; i < n; i += int64_t(gridDim.x) * blockDim.x)
        y[i] = T(a * double(x[i]) + (b == 0.0 ? 0.0 : b * double(y[i])));
}

// ---- least-squares state of one GMRES restart cycle of m steps, on the
// device (doubles): cs[m], sn[m], g[m + 1], R[m * m] (column j at R + j m),
// H[(m + 1) * m] (raw Hessenberg, column j at H + j (m + 1)), est[m].
struct GState {
    double *cs, *sn, *g, *R, *H, *est;
    __device__ GState(double *s, int m)
        : cs(s), sn(s + m), g(s + 2 * m), R(s + 3 * m + 1), H(s + 3 * m + 1 + m * m),
          est(s + 3 * m + 1 + m * m + (m + 1) * m) {}
};

__global__ void k_gmres_begin(int m, double beta, double *state) {
    GState s(state, m);
    for (int i = threadIdx.x; i <= m; i += blockDim.x) s.g[i] = (i == 0) ? beta : 0.0;
}

// Fold Hessenberg column j (hcol[0..j+1]) into the QR factorisation: apply
// the previous rotations, form rotation j, update g; est[j] = |g[j + 1]|
// is the residual norm of the minimiser over the first j + 1 directions.
__global__ void k_gmres_givens(int j, int m, const double *__restrict__ hcol, double *state) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    GState s(state, m);
    double *Rj = s.R + int64_t(j) * m;
    double *Hj = s.H + int64_t(j) * (m + 1);
    for (int i = 0; i <= j + 1; ++i) Hj[i] = hcol[i];
    for (int i = 0; i <= j; ++i) Rj[i] = hcol[i];
    const double hj1 = hcol[j + 1];
    for (int i = 0; i < j; ++i) {
        const double a = Rj[i], b = Rj[i + 1];
        Rj[i] = s.cs[i] * a + s.sn[i] * b;
        Rj[i + 1] = -s.sn[i] * a + s.cs[i] * b;
    }
    const double den = hypot(Rj[j], hj1);
    const double c = den != 0.0 ? Rj[j] / den : 1.0;
    const double sn = den != 0.0 ? hj1 / den : 0.0;
    s.cs[j] = c;
    s.sn[j] = sn;
    Rj[j] = den;
    const double gj = s.g[j];
    s.g[j + 1] = -sn * gj;
    s.g[j] = c * gj;
    s.est[j] = fabs(s.g[j + 1]);
}

// y = R_k^{-1} g_k (back substitution over the first k columns), one
// wavefront: lane l holds rows l, l + 64, .. and takes the columns from the
// last to the first, the next one (contiguous in R) loading meanwhile.  Row by
// row on one thread it was 110 us at k = 50, each term waiting for a load:
// 14 us now.
template <int ROWS>
__device__ inline void back_substitute(int k, int m, const GState &s, double *y, int lane) {
    double acc[ROWS], col[ROWS], nxt[ROWS];
    const auto load = [&](int l, double (&c)[ROWS]) {
        const double *R = s.R + int64_t(max(l, 0)) * m;
#pragma unroll
        for (int q = 0; q < ROWS; ++q) c[q] = R[min(lane + 64 * q, max(l, 0))];
    };
#pragma unroll
    for (int q = 0; q < ROWS; ++q) acc[q] = s.g[min(lane + 64 * q, k - 1)];
    load(k - 1, col);
    for (int l = k - 1; l >= 0; --l) {
        load(l - 1, nxt);
        double num = acc[0], d = col[0];
#pragma unroll
        for (int q = 1; q < ROWS; ++q)
            if (l >> 6 == q) {
                num = acc[q];
                d = col[q];
            }
        num = __shfl(num, l & 63);
        d = __shfl(d, l & 63);
        const double yl = d != 0.0 ? num / d : 0.0;
        if (lane == 0) y[l] = yl;
#pragma unroll
        for (int q = 0; q < ROWS; ++q) {
            if (lane + 64 * q < l) acc[q] -= col[q] * yl;
            col[q] = nxt[q];
        }
    }
}

__global__ __launch_bounds__(64) void k_gmres_solve(int k, int m, const double *state,
                                                    double *__restrict__ y) {
    GState s(const_cast<double *>(state), m);
    if (k <= 64) back_substitute<1>(k, m, s, y, threadIdx.x);
    else back_substitute<KMAXV / 64>(k, m, s, y, threadIdx.x);
}

template <typename S, typename D>
__global__ void k_convert(int64_t n, const S *__restrict__ s, D *__restrict__ d) {
    int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    for (; i < n; i += int64_t(gridDim.x) * blockDim.x) d[i] = D(s[i]);
}

}  // namespace rtx

using namespace rtx;

extern "C" int rtx_arnoldi_workspace(int max_vecs, int64_t *n_doubles) {
    RTX_CHECK(n_doubles && max_vecs >= 1 && max_vecs < KMAXV,
              "rtx_arnoldi_workspace: max_vecs must be in [1, %d)", KMAXV);
    // dot partials ((KMAXV + 1) rows, the last one also holding the second-pass
    // coefficients), norm partials, and a small state block (norms + flag)
    *n_doubles = int64_t(KMAXV + 2) * KNB + WORK_TAIL;
    return RTX_OK;
}

template <typename T>
static bool aligned16(const T *p) {
    return (reinterpret_cast<uintptr_t>(p) & 15) == 0;
}

// Values per load that the basis and w allow (rows of nv > 1 vectors start
// ld apart).
template <typename T, typename TW>
static int vec_width(const T *V, int64_t ld, int nv, const TW *w) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(V) | (nv > 1 ? uintptr_t(ld) * sizeof(T) : 0);
    if (!aligned16(w)) return 1;
    if (at % 16 == 0) return kvec<T>();
    return sizeof(T) == 2 && at % 8 == 0 ? 4 : 1;
}

// f(std::integral_constant<int, VW>) for the width vec_width gave.
template <typename T, typename F>
static void with_width(int vw, F f) {
    if (vw == kvec<T>()) return f(std::integral_constant<int, kvec<T>()>());
    if constexpr (sizeof(T) == 2)
        if (vw == 4) return f(std::integral_constant<int, 4>());
    f(std::integral_constant<int, 1>());
}

template <typename T, typename TW>
static void launch_mdot(int vw, int nb, hipStream_t st, const T *V, int64_t ld, int nv,
                        const TW *w, int64_t n, double *part, int with_ww, const int *flag) {
    const int grid = (nb + 7) / 8 * 8 * ((nv + KCH - 1) / KCH);
    with_width<T>(vw, [&](auto v) {
        k_mdot<T, decltype(v)::value, TW><<<grid, KT, 0, st>>>(V, ld, nv, w, n, nb, part, with_ww,
                                                               flag);
    });
}

static void launch_reduce(const double *part, int nb, int nj, double *out, int accumulate,
                          const int *flag, hipStream_t st) {
    k_reduce<<<(nj + KW - 1) / KW, KT, 0, st>>>(part, nb, nj, out, accumulate, flag);
}

template <typename T>
static void launch_update(int vw, int nb, hipStream_t st, const T *V, int64_t ld, int nv,
                          const double *h, T *w, int64_t n, double *part, const int *flag) {
    with_width<T>(vw, [&](auto v) {
        k_update<T, decltype(v)::value><<<nb, KT, 0, st>>>(V, ld, nv, h, w, n, part, flag);
    });
}

// Classical Gram-Schmidt, one pass, with the norm from the dot products, in
// three launches: dots, their reduction, the update writing the normalised
// vector (and the Givens update).  Widths count V_out's row too.
template <typename T, typename TW>
static int arnoldi_pyth(const T *d_V, int64_t ld, int nv, int64_t n, const TW *d_w, double *d_hcol,
                        double *part, double *hd, hipStream_t st, int gj, int gm,
                        double *d_state) {
    T *V_out = const_cast<T *>(d_V) + int64_t(nv) * ld;
    const int vw = vec_width(d_V, ld, nv + 1, d_w), nb = row_blocks(n, vw);
    launch_mdot(vw, nb, st, d_V, ld, nv, d_w, n, part, 1, nullptr);
    launch_reduce(part, nb, nv + 1, hd, 0, nullptr, st);
    with_width<T>(vw, [&](auto v) {
        k_update_pyth<T, decltype(v)::value, TW><<<nb + 1, KT, 0, st>>>(
            d_V, ld, nv, hd, d_w, V_out, n, d_hcol, gj, gm, d_state);
    });
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

// One Arnoldi step; with d_state, the final normalisation also folds the
// new Hessenberg column j into the least-squares state (rtx_gmres_givens).
template <typename T>
static int arnoldi_step(const T *d_V, int64_t ld, int nv, int64_t n, T *d_w, double *d_hcol,
                        double *d_work, int refine, void *stream, int gj = -1, int gm = 0,
                        double *d_state = nullptr) {
    RTX_CHECK(d_V && d_w && d_hcol && d_work, "rtx_arnoldi_step: null argument");
    RTX_CHECK(refine >= 0 && refine <= 2, "rtx_arnoldi_step: refine must be 0, 1 or 2");
    RTX_CHECK(nv >= 1 && nv < KMAXV - 1, "rtx_arnoldi_step: nv=%d outside [1, %d)", nv,
              KMAXV - 1);
    RTX_CHECK(n >= 1 && ld >= n, "rtx_arnoldi_step: bad n/ld");
    hipStream_t st = static_cast<hipStream_t>(stream);
    double *part = d_work;                                  // (nv + 1) * KNB
    double *part2 = d_work + int64_t(KMAXV + 1) * KNB;      // KNB
    double *state = part2 + KNB;                            // [ww0, ww1, h2...]
    int *flag = reinterpret_cast<int *>(state + 4);
    T *V_out = const_cast<T *>(d_V) + int64_t(nv) * ld;
    // FP32 basis (the inner solves of mixed refinement)
    if constexpr (std::is_same<T, float>::value)
        if (refine == 0)
            return arnoldi_pyth(d_V, ld, nv, n, d_w, d_hcol, part, part2, st, gj, gm,
                                d_state);
    const int vw = vec_width(d_V, ld, nv, d_w), nb = row_blocks(n, vw);
    auto normalize = [&](const double *nrm2, int nparts) {
        const int blocks = int(std::min<int64_t>(2048, (n + KT - 1) / KT));
        k_normalize<T><<<blocks + 1, KT, 0, st>>>(d_w, V_out, n, nrm2, nparts, d_hcol, nv, gj, gm,
                                                  d_state);
    };
    // pass 1: h = V^T w, |w|^2
    launch_mdot(vw, nb, st, d_V, ld, nv, d_w, n, part, refine == 1 ? 1 : 0, nullptr);
    launch_reduce(part, nb, nv, d_hcol, 0, nullptr, st);
    if (refine == 1) launch_reduce(part + int64_t(nv) * nb, nb, 1, state + 0, 0, nullptr, st);
    // w -= V h, |w'|^2
    launch_update<T>(vw, nb, st, d_V, ld, nv, d_hcol, d_w, n, part2, nullptr);
    if (refine == 0) {     // classical Gram-Schmidt, one pass (PETSc's default)
        normalize(part2, nb);
        RTX_HIP(hipGetLastError());
        return RTX_OK;
    }
    launch_reduce(part2, nb, 1, state + 1, 0, nullptr, st);
    if (refine == 1)
        k_reorth_test<<<1, 1, 0, st>>>(state, flag);
    else
        k_set_flag<<<1, 1, 0, st>>>(flag, 0);
    // optional pass 2 (skipped on the device when flag == 1)
    launch_mdot(vw, nb, st, d_V, ld, nv, d_w, n, part, 0, flag);
    // accumulate the correction into hcol, keep it separately for the update
    double *hcorr = part + int64_t(KMAXV) * KNB;            // nv doubles, after the partials
    launch_reduce(part, nb, nv, hcorr, 0, flag, st);
    launch_update<T>(vw, nb, st, d_V, ld, nv, hcorr, d_w, n, part2, flag);
    launch_reduce(part2, nb, 1, state + 1, 0, flag, st);
    launch_reduce(hcorr, 1, nv, d_hcol, 1, flag, st);       // hcol += hcorr
    normalize(state + 1, 1);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

// Arnoldi step on an FP16 basis with an FP32 w (the inner solves of mixed
// refinement): classical Gram-Schmidt, one pass, the norm from the dot
// products (accumulated in FP64), in the FP32 basis's three launches; the
// new basis vector is rounded to FP16 once, after the normalisation.
static int arnoldi_step_h(const _Float16 *d_V, int64_t ld, int nv, int64_t n, const float *d_w,
                          double *d_hcol, double *d_work, int refine, void *stream, int gj,
                          int gm, double *d_state) {
    RTX_CHECK(d_V && d_w && d_hcol && d_work, "rtx_gmres_arnoldi: null argument");
    RTX_CHECK(refine == 0, "rtx_gmres_arnoldi: an FP16 basis takes one pass (refine 0)");
    RTX_CHECK(nv >= 1 && nv < KMAXV - 1, "rtx_gmres_arnoldi: nv=%d outside [1, %d)", nv,
              KMAXV - 1);
    RTX_CHECK(n >= 1 && ld >= n, "rtx_gmres_arnoldi: bad n/ld");
    hipStream_t st = static_cast<hipStream_t>(stream);
    double *part = d_work;
    double *hd = d_work + int64_t(KMAXV + 1) * KNB;
    return arnoldi_pyth(d_V, ld, nv, n, d_w, d_hcol, part, hd, st, gj, gm, d_state);
}

/* One Arnoldi step: orthogonalise w against V_0..V_{nv-1} (columns of length n,
   stride ld) by classical Gram-Schmidt; refine 0: one pass, 1: a second pass
   when the norm dropped by more than the "twice is enough" factor, 2: always
   two passes; normalise into V_nv and write the Hessenberg column
   h_0..h_{nv-1}, h_nv = |w| to d_hcol (device, nv + 1 doubles).  w is
   overwritten.  Everything is enqueued on `stream`; no host sync. */
extern "C" int rtx_arnoldi_step(const double *d_V, int64_t ld, int nv, int64_t n, double *d_w,
                                double *d_hcol, double *d_work, int refine, void *stream) {
    return arnoldi_step<double>(d_V, ld, nv, n, d_w, d_hcol, d_work, refine, stream);
}

/* Arnoldi step j of a GMRES cycle of m steps fused with its Givens update:
   rtx_arnoldi_step (FP64 basis, basis_precision 0, FP32, 1, or FP16 with an
   FP32 w, 2, one pass only) on nv = j + 1 vectors, then
   rtx_gmres_givens(j, m, d_hcol, d_state) folded into the final
   normalisation.  No counterpart in the reference (PETSc
   keeps the least-squares problem on the host). */
extern "C" int rtx_gmres_arnoldi(int basis_precision, const void *d_V, int64_t ld, int64_t n,
                                 void *d_w, double *d_hcol, double *d_work, int refine, int j,
                                 int m, double *d_state, void *stream) {
    RTX_CHECK(d_state && m >= 1 && m < KMAXV - 1 && j >= 0 && j < m,
              "rtx_gmres_arnoldi: bad argument (j=%d, m=%d)", j, m);
    RTX_CHECK(basis_precision >= 0 && basis_precision <= 2,
              "rtx_gmres_arnoldi: basis_precision must be 0 (FP64), 1 (FP32) or 2 (FP16)");
    if (basis_precision == 2)
        return arnoldi_step_h(static_cast<const _Float16 *>(d_V), ld, j + 1, n,
                              static_cast<const float *>(d_w), d_hcol, d_work, refine, stream, j,
                              m, d_state);
    if (basis_precision == 0)
        return arnoldi_step<double>(static_cast<const double *>(d_V), ld, j + 1, n,
                                    static_cast<double *>(d_w), d_hcol, d_work, refine, stream,
                                    j, m, d_state);
    return arnoldi_step<float>(static_cast<const float *>(d_V), ld, j + 1, n,
                               static_cast<float *>(d_w), d_hcol, d_work, refine, stream, j, m,
                               d_state);
}

/* ---- rtx_gmres_arnoldi without a workspace argument.  Its reduction
   partials, norms and re-orthogonalisation flag live in a file-scope device
   array instead, so a caller that cannot allocate (code being captured into
   a HIP graph, a serving loop) passes only its inputs and outputs.  The
   array has the workspace layout of rtx_arnoldi_workspace (every step
   writes each partial before it reads it, so nothing needs clearing
   between calls).  One copy per device, held until the process ends;
   calls that overlap on one device share it and race. */
constexpr int64_t STATIC_WORK_DOUBLES = int64_t(KMAXV + 2) * KNB + WORK_TAIL;   // 2.1 MB
static __device__ __align__(256) double scratch[STATIC_WORK_DOUBLES];

constexpr int MAX_DEVICES = 64;
static std::mutex scratch_mutex;
static double *scratch_ptr[MAX_DEVICES];     // device address of `scratch`, per device

// Device address of `scratch` on the current device (looked up once per
// device with that device current); null with the error set on failure.
static double *static_workspace() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) {
        set_error("rtx_gmres_arnoldi_static: no usable current device (%d)", dev);
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(scratch_mutex);
    if (!scratch_ptr[dev]) {
        void *ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            set_error("rtx_gmres_arnoldi_static: hipGetSymbolAddress failed on device %d: %s",
                      dev, hipGetErrorString(e));
            return nullptr;
        }
        scratch_ptr[dev] = static_cast<double *>(ptr);
    }
    return scratch_ptr[dev];
}

extern "C" int rtx_gmres_arnoldi_static(int basis_precision, const void *d_V, int64_t ld,
                                        int64_t n, void *d_w, double *d_hcol, int refine,
                                        int j, int m, double *d_state, void *stream) {
    RTX_CHECK(m >= 1 && m < KMAXV - 1 && j >= 0 && j < m,
              "rtx_gmres_arnoldi_static: cycle length m=%d (step j=%d) outside the static "
              "workspace's limit m < %d",
              m, j, KMAXV - 1);
    double *work = static_workspace();
    if (!work) return RTX_ERR_HIP;
    return rtx_gmres_arnoldi(basis_precision, d_V, ld, n, d_w, d_hcol, work, refine, j, m,
                             d_state, stream);
}

/* The same step on an FP32 basis (dot products, norms and the Hessenberg
   column accumulated in FP64). */
extern "C" int rtx_arnoldi_step_f32(const float *d_V, int64_t ld, int nv, int64_t n, float *d_w,
                                    double *d_hcol, double *d_work, int refine, void *stream) {
    return arnoldi_step<float>(d_V, ld, nv, n, d_w, d_hcol, d_work, refine, stream);
}

extern "C" int rtx_gmres_state_size(int m, int64_t *n_doubles) {
    RTX_CHECK(n_doubles && m >= 1 && m < KMAXV - 1, "rtx_gmres_state_size: m outside [1, %d)",
              KMAXV - 1);
    *n_doubles = 3 * int64_t(m) + 1 + int64_t(m) * m + int64_t(m + 1) * m + m;
    return RTX_OK;
}

extern "C" int rtx_gmres_begin(int m, double beta, double *d_state, void *stream) {
    RTX_CHECK(d_state && m >= 1 && m < KMAXV - 1, "rtx_gmres_begin: bad argument");
    k_gmres_begin<<<1, 256, 0, static_cast<hipStream_t>(stream)>>>(m, beta, d_state);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

extern "C" int rtx_gmres_givens(int j, int m, const double *d_hcol, double *d_state,
                                void *stream) {
    RTX_CHECK(d_hcol && d_state && m >= 1 && m < KMAXV - 1 && j >= 0 && j < m,
              "rtx_gmres_givens: bad argument (j=%d, m=%d)", j, m);
    k_gmres_givens<<<1, 64, 0, static_cast<hipStream_t>(stream)>>>(j, m, d_hcol, d_state);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

extern "C" int rtx_gmres_solve(int k, int m, const double *d_state, double *d_y, void *stream) {
    RTX_CHECK(d_state && d_y && m >= 1 && m < KMAXV - 1 && k >= 1 && k <= m,
              "rtx_gmres_solve: bad argument (k=%d, m=%d)", k, m);
    k_gmres_solve<<<1, 64, 0, static_cast<hipStream_t>(stream)>>>(k, m, d_state, d_y);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

/* d_out[j] = V_j . w for j < nv (device), workspace as for rtx_arnoldi_step. */
extern "C" int rtx_mdot(const double *d_V, int64_t ld, int nv, int64_t n, const double *d_w,
                        double *d_out, double *d_work, void *stream) {
    RTX_CHECK(d_V && d_w && d_out && d_work && nv >= 1 && nv < KMAXV, "rtx_mdot: bad argument");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int vw = vec_width(d_V, ld, nv, d_w), nb = row_blocks(n, vw);
    launch_mdot(vw, nb, st, d_V, ld, nv, d_w, n, d_work, 0, nullptr);
    launch_reduce(d_work, nb, nv, d_out, 0, nullptr, st);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

/* d_x (+)= sum_j y_j V_j with y on the device. */
extern "C" int rtx_combine(const double *d_V, int64_t ld, int nv, const double *d_y, int64_t n,
                           double *d_x, int accumulate, void *stream) {
    RTX_CHECK(d_V && d_y && d_x && nv >= 1 && nv < KMAXV, "rtx_combine: bad argument");
    k_combine<double, double><<<2048, KT, 0, static_cast<hipStream_t>(stream)>>>(
        d_V, ld, nv, d_y, d_x, n, accumulate);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

/* d_x (+)= sum_j y_j V_j for an FP32 basis; d_x is FP64 (x_precision 0) or
   FP32 (x_precision 1); accumulation in FP64. */
extern "C" int rtx_combine_f32(const float *d_V, int64_t ld, int nv, const double *d_y,
                               int64_t n, void *d_x, int x_precision, int accumulate,
                               void *stream) {
    RTX_CHECK(d_V && d_y && d_x && nv >= 1 && nv < KMAXV && (x_precision == 0 || x_precision == 1),
              "rtx_combine_f32: bad argument");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (x_precision == 0)
        k_combine<float, double><<<2048, KT, 0, st>>>(d_V, ld, nv, d_y, (double *)d_x, n,
                                                      accumulate);
    else
        k_combine<float, float><<<2048, KT, 0, st>>>(d_V, ld, nv, d_y, (float *)d_x, n,
                                                     accumulate);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

/* d_x (+)= sum_j y_j V_j for an FP16 basis (device, IEEE binary16); d_x is
   FP64 (x_precision 0) or FP32 (x_precision 1); accumulation in FP64. */
extern "C" int rtx_combine_f16(const void *d_V, int64_t ld, int nv, const double *d_y,
                               int64_t n, void *d_x, int x_precision, int accumulate,
                               void *stream) {
    RTX_CHECK(d_V && d_y && d_x && nv >= 1 && nv < KMAXV && (x_precision == 0 || x_precision == 1),
              "rtx_combine_f16: bad argument");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const _Float16 *V = static_cast<const _Float16 *>(d_V);
    if (x_precision == 0)
        k_combine<_Float16, double><<<2048, KT, 0, st>>>(V, ld, nv, d_y, (double *)d_x, n,
                                                         accumulate);
    else
        k_combine<_Float16, float><<<2048, KT, 0, st>>>(V, ld, nv, d_y, (float *)d_x, n,
                                                        accumulate);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

/* y = a x + b y with x FP32 and y FP64 (direction 0), x FP64 and y FP32
   (direction 1), or x FP64 and y FP16 (direction 2). */
extern "C" int rtx_axpby_mixed(int direction, int64_t n, double a, const void *d_x, double b,
                               void *d_y, void *stream) {
    RTX_CHECK(d_x && d_y && n >= 0 && direction >= 0 && direction <= 2,
              "rtx_axpby_mixed: bad argument");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (direction == 0)
        k_axpby_mixed<float, double><<<2048, 256, 0, st>>>(n, a, (const float *)d_x, b,
                                                           (double *)d_y);
    else if (direction == 2)
        k_axpby_mixed<double, _Float16><<<2048, 256, 0, st>>>(n, a, (const double *)d_x, b,
                                                              (_Float16 *)d_y);
    else
        k_axpby_mixed<double, float><<<2048, 256, 0, st>>>(n, a, (const double *)d_x, b,
                                                           (float *)d_y);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

/* y = a x + b y for FP64 (precision 0) or FP32 (precision 1) vectors. */
extern "C" int rtx_axpby(int precision, int64_t n, double a, const void *d_x, double b,
                         void *d_y, void *stream) {
    RTX_CHECK(d_x && d_y && n >= 0, "rtx_axpby: bad argument");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (precision == RTX_PREC_F64)
        k_axpby<double><<<2048, 256, 0, st>>>(n, a, (const double *)d_x, b, (double *)d_y);
    else
        k_axpby<float><<<2048, 256, 0, st>>>(n, a, (const float *)d_x, b, (float *)d_y);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

/* Precision conversion FP64 <-> FP32 (direction 0: f64 -> f32, 1: f32 -> f64). */
extern "C" int rtx_convert(int direction, int64_t n, const void *d_src, void *d_dst,
                           void *stream) {
    RTX_CHECK(d_src && d_dst && n >= 0, "rtx_convert: bad argument");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (direction == 0)
        k_convert<double, float><<<2048, 256, 0, st>>>(n, (const double *)d_src, (float *)d_dst);
    else
        k_convert<float, double><<<2048, 256, 0, st>>>(n, (const float *)d_src, (double *)d_dst);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}
