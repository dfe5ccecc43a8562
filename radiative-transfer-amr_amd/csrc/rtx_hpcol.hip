// Matrix-free DG transport operator for uneven-order hp meshes: two kernels.
//
// A column's DOFs are contiguous in the reference's global order (columns by
// key, cells by key, then beta = nth ny i + nth j + a inside a cell).
//
//   k_hp_flux  the upwind face coupling (boundary_convection_matrix.py:
//              348-524).  One wavefront per cell, no LDS: for every link the
//              neighbour's trace is contracted with E^theta over the
//              neighbour's angles, then with E^s over its face nodes, both on
//              the matrix cores with operands read from memory; the links of
//              a face add up in the accumulators.  The sums of the cell's
//              inflow faces are stored at their DOFs of y.  Cells whose
//              neighbours have the same nodes and angles are left out.
//   k_hpcol    everything else, one workgroup of 512 threads per column:
//              x of the column -> LDS (angle-major); each
//              wavefront owns 16 output angles R and every node: it
//              accumulates the scattering sum_A x[s, A] G^T[A, R] on the
//              matrix cores (scattering_matrix.py:142-237), then adds mass
//              (mass_matrix.py:140-173), interior convection
//              (interior_convection_matrix.py:161-243), the outflow faces
//              (boundary_convection_matrix.py:284-346) and the sums that
//              k_hp_flux left in y, or, where the neighbours are alike, their
//              values of x times the (then diagonal) coupling; stores y.
//
// The two share no workspace: y itself carries the face sums from one to the
// other (with accumulation a node that has some is therefore rounded twice, in
// FP32 up to 1.5 times the error of one rounding).  The plan's side stream and its two events are shared by all applies, so
// a plan serves one stream at a time.
//
// The nodes are the rows of the scattering product in an order of our own: a
// lane's accumulators are whole lines of nodes (x-lines q = lane group,
// lane group + 4, ..), so the derivative along x reads a line once for all of
// its outputs, with the derivative matrix in scalar registers, and the
// derivative along y reads each row of nodes once per line.  On an hp mesh of
// 8.3 M DOF that is 28 LDS instructions per 64 outputs in FP64 and 21 in mixed
// precision; evaluated output by output, with the face coupling in LDS, it was
// 71 and 70, and the LDS pipe was what bounded the column.
//
// Every output has one owner and a fixed order of additions, so results are
// bit-reproducible; x is read from HBM once (plus the neighbours' face
// traces), G once, y written once (plus the face sums).  Columns are grouped
// by LDS need into two classes (one launch each) sized so that the first runs
// two workgroups per CU.  Arithmetic: FP64 (v_mfma_f64_16x16x4f64), FP32
// (v_mfma_f32_16x16x4f32) or mixed (FP32 transport terms, BF16 scattering
// operands on v_mfma_f32_16x16x16bf16_1k with FP32 accumulation); columns that
// hp_wide names keep FP64 arithmetic in the last two.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "rtx_internal.h"

namespace rtx {

constexpr int HP_THREADS = 512;
constexpr int HP_WAVES = HP_THREADS / 64;
constexpr int HP_NM = RTX_NMAX;
constexpr int HP_XCD = 8;
constexpr int HP_NMIN = 3;        // node counts compiled for the column kernel
constexpr int HP_WD = HP_NM + HP_NM * HP_NM;   // one n's entry of the line tables

typedef double hp_d4 __attribute__((ext_vector_type(4)));
typedef float hp_f4 __attribute__((ext_vector_type(4)));
typedef short hp_s4 __attribute__((ext_vector_type(4)));

__device__ inline bool hp_on_bdry(int bd, int i, int j, int nx, int ny) {
    return ((bd & 1) && i == nx - 1) || ((bd & 2) && j == ny - 1) || ((bd & 4) && i == 0) ||
           ((bd & 8) && j == 0);
}

// floor(v / n) for 0 <= v < 2^16 and 1 <= n <= 100, by a float product: (v + 0.5)
// / n stays 0.5 / n away from an integer, and the product is off by at most
// 2^-22 of itself, 2^-6 / n.
__device__ inline int hp_div(int v, float rcp) { return int((float(v) + 0.5f) * rcp); }

__device__ inline uint16_t hp_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return uint16_t(u >> 16);
}

// 16 x 16 x 4 products.  A operand: row lane % 16, k = lane / 16; B operand:
// k = lane / 16, column lane % 16; D: column lane % 16, row(lane / 16, v).
// A D is the next product's B operand as it stands, with k = row(lane / 16, s)
// in step s.
template <typename A> struct HpMma;
template <> struct HpMma<double> {
    typedef hp_d4 v4;
    __device__ static v4 step(double a, double b, v4 c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    __host__ __device__ static int row(int lg, int v) { return lg + 4 * v; }
    // lane group and register that hold D row r
    __host__ __device__ static int group(int r) { return r & 3; }
    __host__ __device__ static int reg(int r) { return r >> 2; }
};
template <> struct HpMma<float> {
    typedef hp_f4 v4;
    __device__ static v4 step(float a, float b, v4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __host__ __device__ static int row(int lg, int v) { return 4 * lg + v; }
    __host__ __device__ static int group(int r) { return r >> 2; }
    __host__ __device__ static int reg(int r) { return r & 3; }
};

// XCD-aware index: block b runs on XCD b % 8, and XCD j takes the j-th
// contiguous run of the (key-ordered) work, so neighbouring columns are mostly
// read through the same L2.  -1 past the end.
__device__ inline int hp_xcd(int n) {
    const int per = (n + HP_XCD - 1) / HP_XCD;
    const int i = (blockIdx.x % HP_XCD) * per + blockIdx.x / HP_XCD;
    return (int(blockIdx.x / HP_XCD) < per && i < n) ? i : -1;
}

// ---- the upwind face coupling

constexpr int HF_WAVES = 4;       // cells per workgroup

// One link's operands in matrix-core layout: the neighbour's trace, E^theta
// and E^s.  Indices past the sizes read the last entry; the trace is zero
// there (one mask serves both products: the rows past the face's nodes that
// the first leaves are zero too), and rows and columns past this cell's sizes
// reach no stored value.  Offsets are 32-bit from uniform bases.
template <typename A>
struct HpLink {
    A tv[3], ev[3], sv[4];
    int F, n1, nt1;
};

template <typename T, typename A>
__device__ __forceinline__ HpLink<A> hp_load_link(const DevMesh &m, const int4 rec, uint32_t N,
                                                  uint32_t nt, int restrict_, uint32_t l16,
                                                  uint32_t lg, const T *x) {
    const uint32_t w = rec.y, n1 = (w >> 2) & 15, nt1 = (w >> 6) & 15, stride = (w >> 10) & 255;
    HpLink<A> o;
    o.F = w & 3;
    o.n1 = n1;
    o.nt1 = nt1;
    const uint32_t row = min(l16, n1 - 1);
    // masked inflow nodes of the neighbour count as zero
    bool live = l16 < n1;
    if (restrict_) live = live && !((w >> (18 + row)) & 1);
    const T *tr = x + rec.x;
    const double *Et = m.Eth_pool + rec.w, *Es = m.Es_pool + rec.z;
    const uint32_t r = min(l16, nt - 1), m0 = min(l16, N - 1);
#pragma unroll
    for (int s = 0; s < 3; ++s) {
        const uint32_t a = 4 * s + lg, ac = min(a, nt1 - 1);
        o.tv[s] = keep_if(A(tr[row * stride + ac]), live && a < nt1);
        o.ev[s] = A(Et[ac * nt + r]);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
        o.sv[s] = A(Es[min(uint32_t(HpMma<A>::row(lg, s)), n1 - 1) * N + m0]);
    return o;
}

// Bound by instructions and latency (cell record -> link record -> operands,
// then short matrix chains): records of one load each instead of a walk
// through the mesh tables, no LDS, no branches around loads, and registers
// for 8 wavefronts per SIMD to cover the chains.  An hp mesh's 34,279 cells
// (86,793 links) in FP64: 42 us; loading the next link's operands while the
// current one is multiplied costs two wavefronts per SIMD and measures the
// same.  In FP32 the links of 1,024 columns of 7 x 7 nodes take 9.4 us.
template <typename T, typename A>
__global__ __launch_bounds__(64 * HF_WAVES)
__attribute__((amdgpu_waves_per_eu(8)))
void k_hp_flux(DevMesh m, const HpCell *__restrict__ cells, const int4 *__restrict__ links,
               int ncells, int restrict_, int accumulate, const T *__restrict__ x,
               T *__restrict__ y) {
    typedef HpMma<A> Mma;
    typedef typename Mma::v4 v4;
    const int blk = hp_xcd((ncells + HF_WAVES - 1) / HF_WAVES);
    const int lane = threadIdx.x & 63, l16 = lane & 15, lg = lane >> 4;
    const int ci = blk * HF_WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (blk < 0 || ci >= ncells) return;
    // the cell's scalars are uniform over the wavefront
    const HpCell cl = cells[ci];
    const int nl = cl.w & 255, nt = (cl.w >> 12) & 15, nx = (cl.w >> 8) & 15, ny = (cl.w >> 24) & 15;
    const int bd = restrict_ ? (cl.w >> 16) & 15 : 0, lf = (cl.w >> 20) & 15;
    if (nl == 0) return;
    const v4 zero = v4{0, 0, 0, 0};
    v4 cur = zero;
    // A face shares its first node (m0 = 0) with one neighbouring face and its
    // last with another; the later of the two in face order stores the sum.
    // c0, c1: the values that an earlier face leaves at face F's first and
    // last node, [F] (faces 1, 2, 3)
    A c0[4] = {A(0), A(0), A(0), A(0)}, c1[4] = {A(0), A(0), A(0), A(0)};
    for (int i = 0; i < nl; ++i) {           // ascending faces
        const int4 rec = links[cl.l0 + i];
        const int N = (rec.y & 1) ? nx : ny;             // nodes of this face
        const HpLink<A> lk = hp_load_link<T, A>(m, rec, N, nt, restrict_, l16, lg, x);
        // inn[m1, r] = sum_a tr[m1, a] E^theta[a, r], then
        // sum_m1 E^s[m1, m0] inn[m1, r] onto the face's sums
        v4 inn = zero;
#pragma unroll
        for (int s = 0; s < 3; ++s)
            if (4 * s < lk.nt1) inn = Mma::step(lk.tv[s], lk.ev[s], inn);
#pragma unroll
        for (int s = 0; s < 4; ++s)
            if (Mma::row(0, s) < lk.n1) cur = Mma::step(lk.sv[s], inn[s], cur);
        if (i + 1 == nl || (links[cl.l0 + i + 1].y & 3) != lk.F) {
            const int F = lk.F;
            cur *= (F & 1) ? A(cl.fy) : A(cl.fx);
            // the faces at the first and last node: for an x-face the y-faces
            // 3 and 1, for a y-face the x-faces 2 and 0
            const int f0 = (F & 1) ? 2 : 3, f1 = (F & 1) ? 0 : 1;
            const int rgN = Mma::reg(N - 1);
            const A first = __shfl(cur[0], l16);
            const A last = __shfl(rgN == 0 ? cur[0] : rgN == 1 ? cur[1] : rgN == 2 ? cur[2] : cur[3],
                                  Mma::group(N - 1) * 16 + l16);
            // left for a later face f: at its last node if this is face 0 (an
            // x-face's p = N - 1) or face 1, at its first if face 2
            if (F == 0) { c1[1] = last; c1[3] = first; }
            if (F == 1) c1[2] = first;
            if (F == 2) c0[3] = first;
            const A add0 = F == 3 ? c0[3] : A(0);
            const A add1 = F == 1 ? c1[1] : F == 2 ? c1[2] : F == 3 ? c1[3] : A(0);
            const bool skip0 = ((bd >> f0) & 1) || (((lf >> f0) & 1) && f0 > F);
            const bool skip1 = ((bd >> f1) & 1) || (((lf >> f1) & 1) && f1 > F);
            const int first_s = F == 0 ? (nx - 1) * ny : F == 1 ? ny - 1 : 0;    // its first node
            const int ms = (F & 1) ? ny * nt : nt;
            T *yf = y + cl.off + first_s * nt + l16;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if (Mma::row(0, v) >= N) continue;           // uniform
                const int m0 = Mma::row(lg, v);
                const bool at0 = m0 == 0, at1 = m0 == N - 1;
                const A val = cur[v] + (at0 ? add0 : A(0)) + (at1 ? add1 : A(0));
                if (m0 < N && l16 < nt && !(at0 && skip0) && !(at1 && skip1)) {
                    T *yp = yf + m0 * ms;
                    *yp = accumulate ? T(A(*yp) + val) : T(val);
                }
            }
            cur = zero;
        }
    }
}

// ---- the column kernel

// Row stride (elements) of a node-major copy: at least na rounded up to the
// K step, and congruent to c modulo M, so that the 16 rows x K lanes of one
// matrix-core operand read fall on distinct banks (BF16 quads, 16 x 2 per
// half-wave: stride / 8 odd, c = 8, M = 16).
__host__ __device__ inline int hp_stride(int na, int kstep, int c, int M) {
    const int n = (na + kstep - 1) / kstep * kstep;
    return n + ((c - n) % M + M) % M;
}

struct HpLayout {           // dynamic LDS of one column, in bytes from the base
    int xs, xb, vo, cx, cy, pk, fl, src, total;
    int S, NA, XSB;         // angle-major row (node) stride, padded angle rows, BF16 stride
};

// Angle-major copy: NA rows (the column's angles, padded to the K step with
// zero rows) of S = nsp rounded up to odd entries, so that lanes on
// consecutive angles or nodes read distinct banks; mixed adds the node-major
// BF16 copy.  Then three values and two words per angle, and two more where
// alike neighbours are read directly.  A: LDS element type.
template <typename A, int PREC>
__host__ __device__ inline HpLayout hp_layout(int nsp, int na, bool alike) {
    HpLayout L;
    const int ea = int(sizeof(A));
    const int kstep = (PREC == RTX_PREC_MIXED) ? 16 : 4;
    L.S = nsp | 1;
    L.NA = (na + kstep - 1) / kstep * kstep;
    L.XSB = (PREC == RTX_PREC_MIXED) ? hp_stride(na, 16, 8, 16) : 0;
    int o = 0;
    L.xs = o;
    o += L.NA * L.S * ea;
    o = (o + 15) & ~15;
    L.xb = o;
    o += nsp * L.XSB * 2;
    o = (o + 15) & ~15;
    L.vo = o;
    o += na * ea;
    L.cx = o;
    o += na * ea;
    L.cy = o;
    o += na * ea;
    L.pk = o;
    o += na * 4;
    L.fl = o;
    o += na * 4;
    L.src = (o + 7) & ~7;
    o = L.src + (alike ? na * 8 : 0);
    L.total = (o + 15) & ~15;
    return L;
}

template <typename A>
struct HpShared {
    __attribute__((aligned(16))) A nf[2 * HP_NM * HP_NM];   // mass and scattering factor of each node
    A wd[HP_WD];                                // weights, then w_i l'_p(xi_i) (N x N)
};

// Operand row i of node tile t of the scattering product: register e = 4 t + v
// of lane group g holds node p = e % N of line q = g + 4 (l0 + e / N).  Rows
// past the lines read a valid node; their outputs are not stored.
template <typename A, int N>
__device__ inline int hp_node(int t, int i, int l0, int ny) {
    const int e = 4 * t + HpMma<A>::reg(i), q = HpMma<A>::group(i) + 4 * (l0 + e / N);
    return (e % N) * ny + (q < ny ? q : ny - 1);
}

// What bounds a column: latency in its phases and the LDS pipe in the lines.
// FP64, N = 6, 88 angles, two workgroups per CU, cycles: tables and first G
// rows 7,900, x to LDS 4,200, a wavefront's 16 angles 9,700 (matrix) + 6,600
// (lines), those of the second round 15,100.  Times of the two kernels
// together, against one kernel with the contraction's operands in LDS that
// evaluated output by output: hp mesh of 34,279 cells FP64 283 -> 226 us, 9,150
// cells mixed 87 -> 45 us, 1,024 columns of 7 x 7 nodes FP32 52 -> 35 us (29
// with alike neighbours read directly).
//
// RECT: N nodes along x, the number along y read at run time.  The lines have
// their compiled length; only the sums along y and the divisions by the node
// count are left to run time, and one item takes one line per lane group.  A
// kernel apart: in one with the other columns its scalar registers slow those
// down by 2 to 5 %.  Always in FP64 arithmetic (see hp_wide), on FP64 or FP32
// vectors.  Against the generic kernels, alike neighbours read directly: 1,024
// columns of 8 x 6 nodes and 56 angles FP64 96 -> 38 us, FP32 87 -> 36 us; 4,096
// of 4 x 5 nodes and 64 angles 185 -> 94 and 168 -> 97 us; 256 of 3 x 5 nodes and
// 16 angles 16 -> 8 us.  With hanging nodes, 856 columns of 8 x 6 nodes and 56
// angles: 84 -> 47 and 76 -> 45 us.
template <typename T, typename A, int PREC, int N, bool RECT, bool ALIKE>
__device__ __forceinline__ void hp_column(const DevMesh &m, const HpTables &h, uint32_t ops,
                                          int accumulate, HpShared<A> &sh, unsigned char *lds,
                                          const int32_t *hd, const T *__restrict__ x,
                                          T *__restrict__ y) {
    const int NY = RECT ? hd[5] : N;
    const int NSP = N * NY;
    // x-lines: NL per lane group, LI of them in one item (16 output angles x
    // 4 LI lines).  FP64 takes one: with all of them its accumulators leave
    // too few of the 128 registers of 4 wavefronts per SIMD for the lines
    // (252 spilled, against 2), and two or three times the items spread
    // better over the wavefronts; G is then read from L2 once per item.
    constexpr int NL = (N + 3) / 4;
    constexpr int LI = sizeof(A) == 8 || RECT ? 1 : NL;
    const int NI = RECT ? (NY + 3) / 4 : NL / LI;
    constexpr int MT = (N * LI + 3) / 4;         // node tiles
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lg = lane >> 4;
    const bool restrict_ = (ops & RTX_OP_RESTRICT) != 0;
    const bool bconv = (ops & RTX_OP_BCONV) != 0;
    const int na = hd[3], cdof = hd[4], ga0 = hd[7], sp0 = hd[13], c = hd[14];
    const int ncd = NSP * na;
    const double dx = m.col_geom[4 * c + 2] - m.col_geom[4 * c + 0];
    const double dy = m.col_geom[4 * c + 3] - m.col_geom[4 * c + 1];
    const HpLayout Lo = hp_layout<A, PREC>(NSP, na, ALIKE);
    const int S = Lo.S, XSB = Lo.XSB;
    A *xs = reinterpret_cast<A *>(lds + Lo.xs);
    uint16_t *xb = reinterpret_cast<uint16_t *>(lds + Lo.xb);
    A *vo = reinterpret_cast<A *>(lds + Lo.vo);
    A *fcx = reinterpret_cast<A *>(lds + Lo.cx);
    A *fcy = reinterpret_cast<A *>(lds + Lo.cy);
    int *pk = reinterpret_cast<int *>(lds + Lo.pk);
    int *fl = reinterpret_cast<int *>(lds + Lo.fl);
    int2 *sr = reinterpret_cast<int2 *>(lds + Lo.src);

    // ---- the first G rows of this wavefront's first 16 output angles, in
    // flight through the staging phases.  PD load groups of four K steps (one
    // of 16 in mixed precision; four groups in FP32 are 1 to 2 % slower); lanes
    // past the last angle, and rows past it, read valid addresses: those angle
    // rows of the copy are zero, and those lanes' outputs are not stored.
    constexpr int PD = 2;
    typedef typename std::conditional<PREC == RTX_PREC_MIXED, uint16_t, A>::type GT;
    const GT *Gc = PREC == RTX_PREC_MIXED ? (const GT *)(m.G_bf16 + m.col_G_off[c])
                   : PREC == RTX_PREC_F64 ? (const GT *)(m.G + m.col_G_off[c])
                                          : (const GT *)(m.G_f + m.col_G_off[c]);
    struct Group { GT g[4]; };
    const auto gload = [&](int Rc, int kb) {
        Group o;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int Ak = kb + (PREC == RTX_PREC_MIXED ? 4 * lg + u : 4 * u + lg);
            o.g[u] = Gc[size_t(Ak < na ? Ak : na - 1) * na + Rc];
        }
        return o;
    };
    Group gq[PD];
    const bool scat = (ops & RTX_OP_SCAT) != 0;
    if (scat) {
        const int R = wave / NI * 16 + l16;
#pragma unroll
        for (int d = 0; d < PD; ++d) gq[d] = gload(R < na ? R : na - 1, 16 * d);
    }
    // ---- x of the column and its tables.  The first batch of x is loaded
    // while the angles' tables go to LDS.
    // x values per thread and pass: a column of 96 angles in one (for 48 angles
    // the FP64 hp mesh of 2.0 M DOF takes 93.5 us against 90, for 160 its and
    // the 7 x 7 columns 2 to 5 % more)
    constexpr int XM = (N * N * 96 + HP_THREADS - 1) / HP_THREADS, XU = RECT || XM > 16 ? 16 : XM;
    A vv[XU];
#pragma unroll
    for (int u = 0; u < XU; ++u) {
        const int t = tid + u * HP_THREADS;
        vv[u] = (t < ncd) ? A(x[cdof + t]) : A(0);
    }
    // per angle the mass factor and the fluxes along x and y, rounded once
    for (int a = tid; a < na; a += HP_THREADS) {
        const double w = h.ang_dth[ga0 + a] * m.ang_trig[3 * (ga0 + a) + 2];
        vo[a] = A(dx * dy * 0.125 * w);
        fcx[a] = A(dy * 0.25 * w * m.ang_trig[3 * (ga0 + a)]);
        fcy[a] = A(dx * 0.25 * w * m.ang_trig[3 * (ga0 + a) + 1]);
        pk[a] = m.ang_pack[ga0 + a];
        fl[a] = h.ang_flag[ga0 + a];
        if constexpr (ALIKE) sr[a] = h.ang_src[ga0 + a];
    }
    const double *wd = h.wd + NY * HP_WD;
    for (int t = tid; t < HP_NM + NY * NY; t += HP_THREADS) sh.wd[t] = A(wd[t]);
    if (tid < NSP) {
        const int i = tid / NY, j = tid - i * NY;
        const double w2 = h.wd[N * HP_WD + i] * wd[j];
        sh.nf[2 * tid] = A(w2 * m.kappa[sp0 + tid]);
        sh.nf[2 * tid + 1] = A(dx * dy * m.sigma[sp0 + tid] * w2);
    }
    __syncthreads();
    // DOF t of the column belongs to the cell of angle t / NSP (a cell's DOFs
    // start at NSP times its first angle)
    for (int t0 = tid; t0 < ncd; t0 += XU * HP_THREADS) {
        if (t0 != tid) {
#pragma unroll
            for (int u = 0; u < XU; ++u) {
                const int t = t0 + u * HP_THREADS;
                vv[u] = (t < ncd) ? A(x[cdof + t]) : A(0);
            }
        }
#pragma unroll
        for (int u = 0; u < XU; ++u) {
            const int t = t0 + u * HP_THREADS;
            if (t >= ncd) break;
            A v = vv[u];
            const int ta = RECT ? hp_div(t, 1.0f / float(NSP)) : t / (N * N), w = pk[ta];
            const int nt = (w >> 20) & 31, ao = ta - (w >> 25);
            const int lt = t - NSP * ao;
            const int s = hp_div(lt, 1.0f / float(nt)), a = lt - s * nt;
            const int bd = restrict_ ? (fl[ta] & 15) : 0;
            if (bd) {
                const int i = RECT ? hp_div(s, 1.0f / float(NY)) : s / N;
                if (hp_on_bdry(bd, i, s - i * NY, N, NY)) v = A(0);
            }
            xs[(ao + a) * S + s] = v;
            if constexpr (PREC == RTX_PREC_MIXED) xb[s * XSB + ao + a] = hp_bf16(float(v));
        }
    }
    // zero the padding: angle rows [na, NA) and (mixed) columns [na, XSB)
    for (int t = tid; t < (Lo.NA - na) * S; t += HP_THREADS) xs[na * S + t] = A(0);
    if constexpr (PREC == RTX_PREC_MIXED) {
        for (int t = tid; t < NSP * (XSB - na); t += HP_THREADS) {
            const int s = t / (XSB - na), a = na + t % (XSB - na);
            xb[s * XSB + a] = 0;
        }
    }
    __syncthreads();

    // ---- 16 output angles per wavefront, every node
    typedef typename HpMma<A>::v4 acc4;
    typedef const A __attribute__((address_space(4))) *CPtr;
    // the derivative matrix along x in scalar registers
    const CPtr wdc = (CPtr)(uintptr_t)((sizeof(A) == 8 ? (const void *)(h.wd + N * HP_WD)
                                                       : (const void *)(h.wd_f + N * HP_WD)));
    const int NRT = (na + 15) / 16;
    auto item = [&](int it) {
        const int rt = it / NI, lb = it - rt * NI;
        const int R = rt * 16 + l16;
        const int Rc = R < na ? R : na - 1;
        acc4 acc[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = acc4{0, 0, 0, 0};
        if (scat) {
            int arow[MT], li = l16;
            asm volatile("" : "+v"(li));
#pragma unroll
            for (int t = 0; t < MT; ++t) arow[t] = hp_node<A, N>(t, li, lb, NY);
            for (int kb = 0; kb < na; kb += 16) {
                const Group cur = gq[0];
#pragma unroll
                for (int d = 0; d + 1 < PD; ++d) gq[d] = gq[d + 1];
                gq[PD - 1] = gload(Rc, kb + 16 * PD);
                if constexpr (PREC != RTX_PREC_MIXED) {
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        if (kb + 4 * u < na) {            // uniform across the wave
                            const A *xk = xs + (kb + 4 * u + lg) * S;
#pragma unroll
                            for (int t = 0; t < MT; ++t)
                                acc[t] = HpMma<A>::step(xk[arow[t]], cur.g[u], acc[t]);
                        }
                    }
                } else {
                    const hp_s4 bv = {short(cur.g[0]), short(cur.g[1]), short(cur.g[2]), short(cur.g[3])};
#pragma unroll
                    for (int t = 0; t < MT; ++t) {
                        const hp_s4 av = *reinterpret_cast<const hp_s4 *>(xb + arow[t] * XSB + 4 * lg + kb);
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, bv, acc[t], 0, 0, 0);
                    }
                }
            }
        }
        if (R >= na) return;
        // the output angle's cell and constants
        const int w = pk[R], nt = (w >> 20) & 31, f = fl[R];
        const int bd = restrict_ ? (f & 15) : 0, quad = ((f >> 4) & 7) - 1;
        const int lf = bconv ? (f >> 8) & 15 : 0;
        const A vol = (ops & RTX_OP_MASS) ? vo[R] : A(0), gx = fcx[R], gy = fcy[R];
        const A cx = (ops & RTX_OP_ICONV) ? gx : A(0), cy = (ops & RTX_OP_ICONV) ? gy : A(0);
        // outflow factors of the faces +x, +y, -x, -y (quadrant Q flows out of
        // faces Q and Q + 1)
        const bool ob = bconv && quad >= 0;
        const A ox1 = ob && (quad == 0 || quad == 3) ? gx : A(0);
        const A ox0 = ob && (quad == 1 || quad == 2) ? -gx : A(0);
        const A oy1 = ob && quad < 2 ? gy : A(0);
        const A oy0 = ob && quad >= 2 ? -gy : A(0);
        // ALIKE: inflow from alike neighbours: the outflow factors of the
        // opposite faces, and the neighbours' first face nodes (-1: none)
        int2 src = make_int2(-1, -1);
        if constexpr (ALIKE)
            if (bconv) src = sr[R];
        const bool xlow = quad == 0 || quad == 3;   // inflow at p = 0
        const A ix = -(ox1 + ox0), iy = -(oy1 + oy0);
        // their masked end nodes: x first, x last, y first, y last
        const int mk = restrict_ ? f >> 12 : 0;
        T *yb = y + cdof;
        const int yo = (w & 0xfffff) + (w >> 25);                  // + s nt: node s
        const A *xr = xs + R * S;                                  // angle row R of the copy
#pragma unroll
        for (int l = 0; l < LI; ++l) {
            int q = lg + 4 * (lb + l);
            // opaque: addresses and factors of the line are computed here, not
            // hoisted out of the items and lines to be held (and spilled)
            asm volatile("" : "+v"(q));
            if (q >= NY) continue;
            // faces of the line's nodes (bit F: face F); the end nodes also
            // lie on face 2 (p = 0) or 0 (p = N - 1)
            const int qf = (q == NY - 1 ? 2 : 0) | (q == 0 ? 8 : 0);
            auto faces = [&](int p) { return qf | (p == 0 ? 4 : 0) | (p == N - 1 ? 1 : 0); };
            // the inflow-face sums that k_hp_flux left in y, or the value of
            // the alike y-neighbour; one node ahead
            const bool yin = src.y >= 0 && q == (quad < 2 ? 0 : NY - 1);
            auto face_sum = [&](int p) {
                A v = A(0);
                const bool dead = (p == 0 && (mk & 4)) || (p == N - 1 && (mk & 8));
                if (faces(p) & lf) v = A(yb[yo + (p * NY + q) * nt]);
                if (yin && !dead) v = iy * A(x[uint32_t(src.y + p * NY * nt)]);
                return v;
            };
            A fs = face_sum(0);
            A lx[N];
#pragma unroll
            for (int i = 0; i < N; ++i) lx[i] = xr[i * NY + q];
            const A *wy = sh.wd + HP_NM + q * NY;
            const A wq = sh.wd[q];
            // and of the alike x-neighbour
            A xin = A(0);
            if (src.x >= 0 && !(q == 0 && (mk & 1)) && !(q == NY - 1 && (mk & 2)))
                xin = wq * ix * A(x[uint32_t(src.x + q * nt)]);
            // y-faces' outflow factor of this line, times w_p below
            const A oy = q == NY - 1 ? oy1 : (q == 0 ? oy0 : A(0));
            // one output's reads at a time, and none kept for the next line:
            // hoisted, they spill
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int p = 0; p < N; ++p) {
                const int s = p * NY + q;
                const A *ly = xr + p * NY;
                const A fn = p + 1 < N ? face_sum(p + 1) : A(0);
                A sx = A(0), sy = A(0);
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    sx += wdc[HP_NM + p * N + i] * lx[i];
                    if constexpr (!RECT) sy += wy[i] * ly[i];
                }
                if constexpr (RECT) {
                    // four at a time; past the last node that node again
                    // with a zero factor
#pragma unroll
                    for (int jb = 0; jb < HP_NM; jb += 4)
                        if (jb < NY) {                    // uniform
#pragma unroll
                            for (int j = jb; j < jb + 4; ++j) {
                                const int jc = j < NY ? j : NY - 1;
                                sy += keep_if(wy[jc], j < NY) * ly[jc];
                            }
                        }
                }
                const A wp = wdc[p], xv = lx[p];
                A val = vol * sh.nf[2 * s] * xv - (cx * wq * sx + cy * wp * sy);
                if (p == N - 1) val += ox1 * wq * xv;
                if (p == 0) val += ox0 * wq * xv;
                if (p == 0) val += xlow ? xin : A(0);
                if (p == N - 1) val += xlow ? A(0) : xin;
                val += oy * wp * xv;
                val += yin ? wp * fs : fs;
                fs = fn;
                if (scat) val -= sh.nf[2 * s + 1] * A(acc[(l * N + p) / 4][(l * N + p) % 4]);
                const int on = faces(p), o = yo + s * nt;
                if (accumulate) {
                    // (face sums were added to y by k_hp_flux)
                    if (!(on & bd)) yb[o] = T((on & lf) ? val : A(yb[o]) + val);
                } else {
                    yb[o] = T((on & bd) ? A(0) : val);
                }
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    // the first item apart from the others: in one loop, the G rows loaded
    // ahead for it would hold registers through every item's lines
    if (wave < NRT * NI) item(wave);
    for (int it = wave + HP_WAVES; it < NRT * NI; it += HP_WAVES) {
        if (scat) {
            const int R = it / NI * 16 + l16;
#pragma unroll
            for (int d = 0; d < PD; ++d) gq[d] = gload(R < na ? R : na - 1, 16 * d);
        }
        item(it);
    }
}

template <typename T, typename A, int PREC, bool RECT, bool ALIKE>
__global__ __launch_bounds__(HP_THREADS) __attribute__((amdgpu_waves_per_eu(4)))
void k_hpcol(DevMesh m, HpTables h, uint32_t ops, int accumulate,
             const int32_t *__restrict__ hdr, int ncols, const T *__restrict__ x,
             T *__restrict__ y) {
    extern __shared__ __align__(16) unsigned char hp_lds[];
    __shared__ HpShared<A> sh;
    const int ci = hp_xcd(ncols);
    if (ci < 0) return;
    const int32_t *hd = hdr + size_t(ci) * HP_HDR;
    // compiled per node count along x
    switch (hd[2]) {
#define HP_CASE(NN)                                                                   \
    case NN:                                                                          \
        hp_column<T, A, PREC, NN, RECT, ALIKE>(m, h, ops, accumulate, sh, hp_lds, hd, \
                                               x, y);                                 \
        break;
        HP_CASE(3) HP_CASE(4) HP_CASE(5) HP_CASE(6) HP_CASE(7) HP_CASE(8) HP_CASE(9) HP_CASE(10)
#undef HP_CASE
        default: break;
    }
}

// ---- host side

// Bytes of dynamic LDS a column needs (FP64 or FP32 storage, mixed adds the
// BF16 copy).
static size_t hp_bytes(int nsp, int na, int prec, bool alike) {
    if (prec == RTX_PREC_F64) return size_t(hp_layout<double, RTX_PREC_F64>(nsp, na, alike).total);
    if (prec == RTX_PREC_F32) return size_t(hp_layout<float, RTX_PREC_F32>(nsp, na, alike).total);
    return size_t(hp_layout<float, RTX_PREC_MIXED>(nsp, na, alike).total);
}

// Static LDS of k_hpcol (the tables above), for the capacity check.
constexpr size_t HP_STATIC_BYTES = sizeof(HpShared<double>) + 64;

// Whether FP32 and mixed precision apply column c in FP64 arithmetic (T float,
// A double, on the RECT kernel): columns of unlike orders, and square ones that
// with their couplings hold more FP64 values than a CU's LDS less 11 KB of
// tables, or more than 192 links or 4,096 inflow-face values.  Those have
// always run like that in reduced precision (on the generic kernels, with FP64
// transport terms), and what a caller gets there is not to depend on the kernel:
// relative error 2.5e-8 (generic 3.6e-8), against 1e-7 in FP32 arithmetic and
// 2e-5 with BF16 scattering.  (FP32 arithmetic took 30 us where this takes 36,
// 1,024 columns of 8 x 6 nodes and 56 angles.)
static bool hp_wide(const rtx_mesh_desc *d, int c) {
    constexpr size_t LDS_VALUES = 152712;
    const int k0 = d->col_cell_start[c], k1 = d->col_cell_start[c + 1];
    const int nx = d->col_nx[c], ny = d->col_ny[c], na = d->col_nang[c];
    if (nx != ny || d->link_start[k1] - d->link_start[k0] > 192) return true;
    // values of the inflow faces, of the traces contracted over their angles,
    // and of the distinct E^s blocks
    int sums = 0, inner = 0, nes = 0;
    std::vector<int32_t> seen;
    for (int k = k0; k < k1; ++k) {
        int lf = 0;
        for (int l = d->link_start[k]; l < d->link_start[k + 1]; ++l) {
            const int c1 = d->cell_col[d->link_src[l]], odd = d->link_face[l] & 1;
            const int n1 = odd ? d->col_nx[c1] : d->col_ny[c1];
            lf |= 1 << d->link_face[l];
            inner += n1 * d->cell_nth[k];
            if (std::find(seen.begin(), seen.end(), d->link_Es_off[l]) == seen.end()) {
                seen.push_back(d->link_Es_off[l]);
                nes += nx * n1;
            }
        }
        sums += __builtin_popcount(lf) * nx * d->cell_nth[k];
    }
    const size_t own = std::max((na + 3) / 4 * 4 * (nx * ny | 1), d->col_ntrace[c]);
    const size_t bytes = (8 * own + 15) / 16 * 16 + 8 * size_t(std::max(sums, inner) + nes) + 28 * na;
    return sums > 4096 || (bytes + 15) / 16 * 16 > LDS_VALUES;
}

// Whether the RECT kernel needs long for column c: its wavefronts' rounds of
// items (16 angles, a line per lane group) times an item's work, the matrix steps
// (angles x node tiles / 4) and the lines' products at half the weight.
static bool hp_long(const rtx_mesh_desc *d, int c) {
    const int nx = d->col_nx[c], ny = d->col_ny[c], na = d->col_nang[c];
    const int items = (na + 15) / 16 * ((ny + 3) / 4);
    const int work = na * ((nx + 3) / 4) / 2 + nx * (nx + ny);
    return (items + HP_WAVES - 1) / HP_WAVES * work > 500;
}

// Whether cell k's links all join it to cells with the same nodes and angles,
// through an inflow face each.  E^s and E^theta are then diagonal (weights;
// weights x direction) up to the rounding of the node positions, and the
// column kernel reads the neighbours' values directly.  src: the x- and the
// y-neighbour's first face node (-1: none); masked: its masked end nodes
// (bits: x first, x last, y first, y last).
bool alike_cell(const rtx_mesh_desc *d, int k, int32_t *src, int32_t *masked) {
    const int c = d->cell_col[k], nx = d->col_nx[c], ny = d->col_ny[c], nt = d->cell_nth[k];
    const int quad = d->cell_quad[k];
    src[0] = src[1] = -1;
    *masked = 0;
    if (quad < 0) return false;
    const auto diagonal = [](const double *E, int n, auto diag) {
        for (int a = 0; a < n; ++a)
            for (int b = 0; b < n; ++b)
                if (!(std::fabs(E[a * n + b] - (a == b ? diag(a) : 0.0)) <= 1e-13)) return false;
        return true;
    };
    for (int l = d->link_start[k]; l < d->link_start[k + 1]; ++l) {
        const int s = d->link_src[l], F = d->link_face[l], c1 = d->cell_col[s], odd = F & 1;
        if ((F != ((quad + 2) & 3) && F != ((quad + 3) & 3)) || src[odd] >= 0) return false;
        if (d->col_nx[c1] != nx || d->col_ny[c1] != ny || d->cell_nth[s] != nt) return false;
        const int n = odd ? nx : ny;
        const double *trig = d->ang_trig + 3 * (d->col_ang_start[c] + d->cell_ang_off[k]);
        if (!diagonal(d->Es_pool + d->link_Es_off[l], n,
                      [&](int a) { return d->lgl_w[n * HP_NM + a]; }) ||
            !diagonal(d->Eth_pool + d->link_Eth_off[l], nt, [&](int a) {
                return trig[3 * a + 2] * trig[3 * a + odd] * (F < 2 ? 1.0 : -1.0);
            }))
            return false;
        // the neighbour's opposite face: its first node and masked ends (the
        // masked faces next to it; never the face itself, which has links)
        const int bd = d->cell_bdry[s] & 15, node = F == 2 ? (nx - 1) * ny : F == 3 ? ny - 1 : 0;
        if (bd >> ((F + 2) & 3) & 1) return false;
        src[odd] = d->cell_dof_off[s] + node * nt;
        *masked |= ((bd >> (odd ? 2 : 3) & 1) | (bd >> (odd ? 0 : 1) & 1) << 1) << 2 * odd;
    }
    return true;
}

int hpcol_build(rtx_plan *p, const rtx_mesh_desc *d) {
    const int nc = d->ncol;
    p->hp_ok = false;
    std::vector<int32_t> ang_flag(std::max<int64_t>(d->nang, 1), 0);
    std::vector<double> ang_dth(std::max<int64_t>(d->nang, 1), 0.0);
    std::vector<int32_t> ang_src(2 * std::max<int64_t>(d->nang, 1), -1);
    int max_lds = 0;
    RTX_HIP(hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, p->device));
    const size_t cap = size_t(max_lds) > HP_STATIC_BYTES ? size_t(max_lds) - HP_STATIC_BYTES : 0;
    // a column whose workgroup (dynamic + static LDS) fits half of a CU's
    // 160 KB runs two workgroups per CU (class 0), the others one (class 1)
    const size_t half = 80 * 1024 > HP_STATIC_BYTES ? 80 * 1024 - HP_STATIC_BYTES : 0;
    std::vector<int32_t> hdr[3][HP_NCLS], wide[2][HP_NCLS], over, links;
    std::vector<HpCell> cells, wide_cells;
    p->hp_ncols = 0;
    // Neighbours are read directly where at least half of the cells have alike
    // ones.  The kernel that does so holds more registers: with no such cell it
    // takes 3 to 6 % longer (an hp mesh in FP64, 208 -> 221 us), with nothing else
    // it saves the face kernel (1,024 columns of 5 x 5 nodes and 40 angles FP64 29
    // -> 21 us, FP32 25 -> 20).  That mesh with columns p-refined: 69 % alike 29.4
    // -> 26.7 and 25.7 -> 24.6 us, 50 % 29.8 -> 28.2 and 25.9 -> 26.0, 36 % 29.9 ->
    // 29.2 and 26.1 -> 27.7, 28 % 30.1 -> 30.4 and 26.3 -> 28.5.
    std::vector<int32_t> cell_src(size_t(2) * d->ncell), cell_mask(d->ncell);
    std::vector<char> direct(d->ncell);
    int64_t ndirect = 0;
    for (int k = 0; k < d->ncell; ++k) {
        direct[k] = alike_cell(d, k, &cell_src[size_t(2) * k], &cell_mask[k]);
        ndirect += direct[k];
    }
    p->hp_alike = 2 * ndirect >= d->ncell;
    if (!p->hp_alike) std::fill(direct.begin(), direct.end(), char(0));
    // A workgroup works a column off alone, so few columns that need long leave
    // the chip idle, and the generic kernels spread them better.  Where they
    // are at most three for every four CUs, the default path leaves the long
    // ones of the columns that hp_wide names to the generic kernels.  Generic
    // against column kernel: 16 columns of 10 x 9 nodes and 80 angles (work 620)
    // FP32 32 / 36 us, of 8 x 7 nodes and 112 angles (464) 33 / 30 us; 16 of 8 x 7
    // nodes and 256 angles FP64 50 / 79 us, 64 of them 61 / 79, 160 115 / 90; of
    // 6 x 5 nodes and 192 angles in FP32 160 columns 51 / 54 us, 193 53 / 52.
    std::vector<char> in_f64(nc), late(nc);
    int nlate = 0;
    for (int c = 0; c < nc; ++c) {
        in_f64[c] = hp_wide(d, c);
        late[c] = in_f64[c] && hp_long(d, c);
        nlate += late[c];
    }
    if (4 * nlate > 3 * p->n_cu) std::fill(late.begin(), late.end(), char(0));
    // late columns last, so that each list begins with the default path's part
    std::vector<int32_t> order;
    for (int l = 0; l < 2; ++l)
        for (int c = 0; c < nc; ++c)
            if (late[c] == l) order.push_back(c);
    std::vector<int32_t> deferred;
    for (const int c : order) {
        const int k0 = d->col_cell_start[c], k1 = d->col_cell_start[c + 1];
        const int nsp = d->col_nx[c] * d->col_ny[c], na = d->col_nang[c];
        // per angle: its cell's masked faces, quadrant + 1 and the faces that
        // carry links, and the cell's width
        int64_t a = d->col_ang_start[c];
        for (int k = k0; k < k1; ++k) {
            int lf = 0;
            if (!direct[k])
                for (int l = d->link_start[k]; l < d->link_start[k + 1]; ++l)
                    lf |= 1 << d->link_face[l];
            for (int r = 0; r < d->cell_nth[k]; ++r, ++a) {
                ang_flag[a] = (d->cell_bdry[k] & 15) | (d->cell_quad[k] + 1) << 4 | lf << 8;
                ang_dth[a] = d->cell_geom[2 * k + 1] - d->cell_geom[2 * k];
                if (!direct[k]) continue;
                ang_flag[a] |= cell_mask[k] << 12;
                for (int e = 0; e < 2; ++e) {
                    const int32_t src = cell_src[size_t(2) * k + e];
                    ang_src[2 * a + e] = src < 0 ? -1 : src + r;
                }
            }
        }
        const int32_t h[HP_HDR] = {k0, k1 - k0, d->col_nx[c], na, d->cell_dof_off[k0],
                                   d->col_ny[c], 0,
                                   d->col_ang_start[c], 0, 0, 0, 0, 0, d->col_sp_off[c], c, 0};
        // HP_NMIN..RTX_NMAX nodes per direction (the compiled node counts)
        bool ok = (k1 - k0) <= HP_MAX_CELLS && std::min(d->col_nx[c], d->col_ny[c]) >= HP_NMIN &&
                  na <= 4096 && k1 > k0;
        for (int k = k0; k < k1; ++k) ok = ok && d->link_start[k + 1] - d->link_start[k] < 256;
        size_t need[3];
        for (int pr = 0; pr < 3; ++pr) {
            need[pr] = hp_bytes(nsp, na, pr, p->hp_alike);
            ok = ok && need[pr] <= cap;
        }
        if (!ok) {
            over.push_back(c);
            continue;
        }
        ++p->hp_ncols;
        if (late[c]) deferred.push_back(c);
        const double dx = d->col_geom[4 * c + 2] - d->col_geom[4 * c];
        const double dy = d->col_geom[4 * c + 3] - d->col_geom[4 * c + 1];
        for (int k = k0; k < k1; ++k) {
            if (direct[k]) continue;
            const double dth = d->cell_geom[2 * k + 1] - d->cell_geom[2 * k];
            HpCell cl;
            cl.fx = dy * 0.25 * dth;
            cl.fy = dx * 0.25 * dth;
            cl.off = d->cell_dof_off[k];
            cl.l0 = int32_t(links.size() / 4);
            int lf = 0, nl = 0;
            for (int F = 0; F < 4; ++F)
                for (int l = d->link_start[k]; l < d->link_start[k + 1]; ++l) {
                    if (d->link_face[l] != F) continue;
                    const int w1 = d->link_meta[4 * l + 1];
                    const int nx1 = (w1 >> 2) & 15, ny1 = (w1 >> 6) & 15, nt1 = (w1 >> 10) & 15;
                    const int bd1 = (w1 >> 14) & 15, n1 = (F & 1) ? nx1 : ny1;
                    // the trace's first DOF, stride and masked nodes
                    const int fixed = F < 2 ? 0 : (F == 2 ? nx1 : ny1) - 1;
                    const int first = (F & 1) ? fixed * nt1 : fixed * ny1 * nt1;
                    const int stride = (F & 1) ? ny1 * nt1 : nt1;
                    int mk = 0;
                    for (int m1 = 0; m1 < n1; ++m1) {
                        const int i1 = (F & 1) ? m1 : fixed, j1 = (F & 1) ? fixed : m1;
                        if (((bd1 & 1) && i1 == nx1 - 1) || ((bd1 & 2) && j1 == ny1 - 1) ||
                            ((bd1 & 4) && i1 == 0) || ((bd1 & 8) && j1 == 0))
                            mk |= 1 << m1;
                    }
                    const int32_t rec[4] = {d->link_meta[4 * l] + first,
                                            F | n1 << 2 | nt1 << 6 | stride << 10 | mk << 18,
                                            d->link_Es_off[l], d->link_Eth_off[l]};
                    links.insert(links.end(), rec, rec + 4);
                    lf |= 1 << F;
                    ++nl;
                }
            cl.w = nl | d->col_nx[c] << 8 | d->cell_nth[k] << 12 | (d->cell_bdry[k] & 15) << 16 |
                   lf << 20 | d->col_ny[c] << 24;
            (in_f64[c] ? wide_cells : cells).push_back(cl);
            if (!late[c]) ++p->hp_n_cells[0];
        }
        const auto take = [&](std::vector<int32_t> *lists, HpClass *classes, size_t bytes) {
            const int cls = bytes <= half ? 0 : 1;
            lists[cls].insert(lists[cls].end(), h, h + HP_HDR);
            classes[cls].bytes = std::max(classes[cls].bytes, bytes);
            if (!late[c]) ++classes[cls].n[0];
        };
        if (d->col_nx[c] == d->col_ny[c]) take(hdr[RTX_PREC_F64], p->hp_cls[RTX_PREC_F64], need[RTX_PREC_F64]);
        else take(wide[0], p->hp_wide[0], need[RTX_PREC_F64]);
        if (in_f64[c]) {
            take(wide[1], p->hp_wide[1], need[RTX_PREC_F64]);
        } else {
            take(hdr[RTX_PREC_F32], p->hp_cls[RTX_PREC_F32], need[RTX_PREC_F32]);
            take(hdr[RTX_PREC_MIXED], p->hp_cls[RTX_PREC_MIXED], need[RTX_PREC_MIXED]);
        }
    }
    p->hp_n_narrow = int(cells.size());
    cells.insert(cells.end(), wide_cells.begin(), wide_cells.end());
    // generic kernels: the columns the kernel cannot take, and in the default
    // path those left to them
    std::vector<int32_t> gcells[2], gitems[2];
    for (int f = 0; f < 2; ++f) {
        std::vector<int32_t> cols(over);
        if (f == 0) cols.insert(cols.end(), deferred.begin(), deferred.end());
        std::sort(cols.begin(), cols.end());
        for (int c : cols)
            for (int k = d->col_cell_start[c]; k < d->col_cell_start[c + 1]; ++k)
                gcells[f].push_back(k);
        gitems[f] = scatter_items(p, cols);
    }
    // weights and w_i l'_p(xi_i) per node count
    std::vector<double> wd(size_t(HP_NM + 1) * HP_WD, 0.0);
    for (int n = 1; n <= HP_NM; ++n)
        for (int i = 0; i < n; ++i) {
            wd[size_t(n) * HP_WD + i] = d->lgl_w[n * HP_NM + i];
            for (int pp = 0; pp < n; ++pp)
                wd[size_t(n) * HP_WD + HP_NM + pp * n + i] =
                    d->lgl_w[n * HP_NM + i] * d->lgl_D[(size_t(n) * HP_NM + pp) * HP_NM + i];
        }
    const std::vector<float> wd_f(wd.begin(), wd.end());
    size_t total = ang_flag.size() + ang_src.size() + links.size() + wd_f.size() + 96;
    for (int f = 0; f < 2; ++f) total += gcells[f].size() + gitems[f].size();
    for (int k = 0; k < HP_NCLS; ++k) {
        for (const auto &lists : hdr) total += lists[k].size();
        for (const auto &lists : wide) total += lists[k].size();
    }
    RTX_HIP(hipMalloc(&p->hp_alloc, total * sizeof(int32_t)));
    RTX_HIP(hipMalloc(&p->hp_es, (wd.size() + ang_dth.size()) * sizeof(double) +
                                    cells.size() * sizeof(HpCell) + 64));
    char *base = static_cast<char *>(p->hp_alloc);
    auto put = [&](const void *v, size_t bytes) -> const void * {
        if (bytes == 0) return nullptr;
        const void *ptr = base;
        (void)hipMemcpy(base, v, bytes, hipMemcpyHostToDevice);
        base += (bytes + 15) & ~size_t(15);
        return ptr;
    };
    auto put_i = [&](const std::vector<int32_t> &v) {
        return static_cast<const int32_t *>(put(v.data(), v.size() * sizeof(int32_t)));
    };
    p->hp.ang_flag = put_i(ang_flag);
    p->hp.ang_src = reinterpret_cast<const int2 *>(put_i(ang_src));
    p->hp.links = reinterpret_cast<const int4 *>(put_i(links));
    const auto put_class = [&](HpClass &hc, const std::vector<int32_t> &list) {
        hc.hdr = put_i(list);
        hc.n[1] = int(list.size() / HP_HDR);
    };
    for (int k = 0; k < HP_NCLS; ++k) {
        for (int pr = 0; pr < 3; ++pr) put_class(p->hp_cls[pr][k], hdr[pr][k]);
        for (int w = 0; w < 2; ++w) put_class(p->hp_wide[w][k], wide[w][k]);
    }
    for (int f = 0; f < 2; ++f) {
        p->hp_gen_cells[f] = put_i(gcells[f]);
        p->hp_n_gen_cells[f] = int(gcells[f].size());
        p->hp_gen_items[f] = put_i(gitems[f]);
        p->hp_n_gen_items[f] = int(gitems[f].size() / 2);
    }
    p->hp.wd_f = static_cast<const float *>(put(wd_f.data(), wd_f.size() * sizeof(float)));
    base = static_cast<char *>(p->hp_es);
    p->hp.wd = static_cast<const double *>(put(wd.data(), wd.size() * sizeof(double)));
    p->hp.ang_dth = static_cast<const double *>(put(ang_dth.data(), ang_dth.size() * sizeof(double)));
    p->hp.cells = static_cast<const HpCell *>(put(cells.data(), cells.size() * sizeof(HpCell)));
    p->hp_n_cells[1] = int(cells.size());
    RTX_HIP(hipGetLastError());
    p->hp_ok = p->hp_ncols > 0;
    // side stream (default priority) and fork / join events of the class launches
    if (p->hp_ok) {
        RTX_HIP(hipStreamCreateWithFlags(&p->hp_side, hipStreamNonBlocking));
        RTX_HIP(hipEventCreateWithFlags(&p->hp_fork, hipEventDisableTiming));
        RTX_HIP(hipEventCreateWithFlags(&p->hp_join, hipEventDisableTiming));
    }
    // the default apply of a mesh that is not one uniform order bin
    // (rtx_autotune may move it back to the generic kernels)
    p->hp_default = p->hp_ok && !p->uni_ok;
    return RTX_OK;
}

template <typename T, typename A>
static int launch_hp_flux(const rtx_plan *p, uint32_t ops, int c0, int n, const T *x, T *y,
                          hipStream_t st, int accumulate) {
    if (n == 0) return RTX_OK;
    const int nblk = (n + HF_WAVES - 1) / HF_WAVES;
    k_hp_flux<T, A><<<(nblk + HP_XCD - 1) / HP_XCD * HP_XCD, 64 * HF_WAVES, 0, st>>>(
        p->m, p->hp.cells + c0, p->hp.links, n, (ops & RTX_OP_RESTRICT) ? 1 : 0, accumulate, x, y);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

template <typename T, typename A, int PREC>
static int launch_hp(const rtx_plan *p, uint32_t ops, const void *dx, void *dy, hipStream_t st,
                     int accumulate, int all) {
    const T *x = static_cast<const T *>(dx);
    T *y = static_cast<T *>(dy);
    if (ops & RTX_OP_BCONV) {
        const int nn = PREC == RTX_PREC_F64 ? 0 : p->hp_n_narrow;
        int rc = launch_hp_flux<T, A>(p, ops, 0, nn, x, y, st, accumulate);
        if (rc) return rc;
        rc = launch_hp_flux<T, double>(p, ops, nn, p->hp_n_cells[all] - nn, x, y, st, accumulate);
        if (rc) return rc;
    }
    auto launch_class = [&](auto kern, const HpClass &hc, hipStream_t s) -> int {
        const int n = hc.n[all];
        if (n == 0) return RTX_OK;
        const int per = (n + HP_XCD - 1) / HP_XCD;
        RTX_HIP(hipFuncSetAttribute((const void *)kern,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, int(hc.bytes)));
        kern<<<per * HP_XCD, HP_THREADS, hc.bytes, s>>>(p->m, p->hp, ops, accumulate, hc.hdr, n, x,
                                                        y);
        RTX_HIP(hipGetLastError());
        return RTX_OK;
    };
    // the columns of the RECT kernel, in FP64 arithmetic whatever the precision
    for (const HpClass &hc : p->hp_wide[PREC == RTX_PREC_F64 ? 0 : 1]) {
        const int rc = p->hp_alike
                           ? launch_class(k_hpcol<T, double, RTX_PREC_F64, true, true>, hc, st)
                           : launch_class(k_hpcol<T, double, RTX_PREC_F64, true, false>, hc, st);
        if (rc) return rc;
    }
    auto launch = [&](const HpClass &hc, hipStream_t s) -> int {
        return p->hp_alike ? launch_class(k_hpcol<T, A, PREC, false, true>, hc, s)
                           : launch_class(k_hpcol<T, A, PREC, false, false>, hc, s);
    };
    const HpClass *hc = p->hp_cls[PREC];
    if (hc[0].n[all] == 0 || hc[1].n[all] == 0 || !p->hp_side)
        return launch(hc[0].n[all] ? hc[0] : hc[1], st);
    // The classes write disjoint outputs, so the large-column class runs on
    // the caller's stream and the other on the plan's side stream at the same
    // time (the side stream waits for the work queued before, and the
    // caller's stream for the side stream): the few large columns then share
    // the GPU with the small ones instead of leaving CUs idle in their tail.
    RTX_HIP(hipEventRecord(p->hp_fork, st));
    RTX_HIP(hipStreamWaitEvent(p->hp_side, p->hp_fork, 0));
    int rc = launch(hc[1], st);
    if (rc) return rc;
    rc = launch(hc[0], p->hp_side);
    if (rc) return rc;
    RTX_HIP(hipEventRecord(p->hp_join, p->hp_side));
    RTX_HIP(hipStreamWaitEvent(st, p->hp_join, 0));
    return RTX_OK;
}

// The column kernels on their columns: all they can take (all = 1) or the
// default path's (0).
int launch_hpcol(rtx_plan *p, uint32_t ops, int prec, const void *dx, void *dy, hipStream_t st,
                 int accumulate, int all) {
    if (prec == RTX_PREC_F64)
        return launch_hp<double, double, RTX_PREC_F64>(p, ops, dx, dy, st, accumulate, all);
    if (prec == RTX_PREC_F32)
        return launch_hp<float, float, RTX_PREC_F32>(p, ops, dx, dy, st, accumulate, all);
    return launch_hp<float, float, RTX_PREC_MIXED>(p, ops, dx, dy, st, accumulate, all);
}

}  // namespace rtx
