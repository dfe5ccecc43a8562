// Order-binned fused apply for uniform column bins.
//
// When every column has nx = ny = N, every cell nth = NTH angular nodes and
// every column NC cells with one shared angular mesh (one G^T block), the
// per-column work has compile-time shape: NSP = N^2 spatial nodes,
// NA = NC NTH angles, NCD = NSP NA DOFs.  The same terms as rtx_fused.hip
// (same reference formulas), specialised: no searches, constant divisions,
// batched register prefetch of the column and the MFMA B operands, and
// XCD-aware (column, part) blocks: each XCD owns a contiguous run of columns.
//
// Two kernels: k_uniform adds the cell-local terms by lines of nodes into an
// output tile in LDS (1, 2 or 4 parts per column) and takes the inflow from
// the neighbours' values directly; k_uniform_e computes every term of an
// output in the scattering MFMA's accumulator layout, with no output tile, so
// more columns are resident per CU (the FP64 default), and stages the
// neighbours' traces in LDS (read by the output lanes instead, they are
// scattered loads: 27 -> 30 us for 1,024 columns of 5 x 5 x 80).
#include <type_traits>

#include "rtx_internal.h"

namespace rtx {

namespace {

typedef double u_dbl4 __attribute__((ext_vector_type(4)));
typedef float u_flt4 __attribute__((ext_vector_type(4)));
typedef short u_sht4 __attribute__((ext_vector_type(4)));

constexpr int UNM = RTX_NMAX;
constexpr int UXCD = 8;

// Faces of the cell that spatial node (i, j) lies on, as cell_bdry bits:
// 1 right (i = n - 1), 2 top (j = n - 1), 4 left (i = 0), 8 bottom (j = 0).
// A node is a masked boundary node of a cell with boundary bits bd exactly
// when bd & u_node_faces(i, j, n) != 0.
__device__ inline int u_node_faces(int i, int j, int n) {
    return (i == n - 1 ? 1 : 0) | (j == n - 1 ? 2 : 0) | (i == 0 ? 4 : 0) | (j == 0 ? 8 : 0);
}

__device__ inline uint16_t u_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return uint16_t(u >> 16);
}

// LDS row stride (in elements) of an [node][angle] tile with na angles per
// node row.  With an odd angle count per cell (nth), a stride congruent to
// nth mod 16 puts the rows of consecutive nodes of one cell at consecutive
// addresses modulo 16, so lanes walking a cell's (node, angle) DOFs in order
// hit distinct banks; the stride stays odd, so lanes on 16 consecutive nodes
// at one angle (the MFMA operand reads) do too.  Even nth: the next odd
// count.
constexpr int u_pad(int na, int nth) {
    if (nth % 2 == 0) return na | 1;
    int v = na;
    while (v % 16 != nth % 16) ++v;
    return v;
}

// Inflow through a face from the neighbour's node at the same place.  Both
// columns have the same nodes and angles there, so the coupling matrices
// E^s and E^theta are diagonal (weights, weights x direction) and the flux at
// a node is the outflow term's product with the neighbour's value and the
// opposite direction: no traces to stage, no contraction.  flux: side / 4 x
// width x angle weight x direction of the axis (rounded once, from FP64: in
// FP32 the error of the coupling is then below that of the contraction); high:
// the outflow face opposite lies at the axis' upper end; w: node weight.
template <typename A>
__device__ inline A u_inflow(A flux, bool high, A w, A xn) {
    return (high ? -flux : flux) * w * xn;
}

// Outflow faces quad and quad + 1 of a cell: the x-face (F even), the y-face,
// and the node rows they lie on.
struct UFaces {
    int Fx, Fy;
    bool yfirst;
    __device__ explicit UFaces(int quad) : yfirst((quad & 1) != 0) {
        Fx = yfirst ? ((quad + 1) & 3) : quad;
        Fy = yfirst ? quad : ((quad + 1) & 3);
    }
};

// BF16 copy of the column for the MIXED scattering MFMA: rows padded to
// whole 16-node tiles, columns to whole 16-angle k-steps, both with zeros;
// row stride na16 + 4 (a multiple of 4 elements, so one 8-byte read per
// operand; 2 dwords mod 32 banks apart per row, so 16 rows hit distinct
// banks).  Byte offset of the copy: the FP32 column and output tiles,
// rounded up to 16 bytes.
constexpr int u_bf_stride(int na) { return (na + 15) / 16 * 16 + 4; }
constexpr size_t u_bf_off(size_t tiles_bytes) { return (tiles_bytes + 15) / 16 * 16; }
constexpr size_t u_bf_bytes(int nsp, int na) {
    return size_t((nsp + 15) / 16 * 16) * u_bf_stride(na) * 2;
}

// Threads per workgroup: one wavefront per 16-wide output-angle tile of the
// part, at least four.
template <int NTH, int NC, int H>
constexpr int u_threads() {
    return ((NC / H) * NTH + 15) / 16 > 4 ? 512 : 256;
}

// Bound by LDS traffic and latency; what counts is how many columns a CU
// holds.  The bounds below hold three (FP64) or four workgroups of eight
// wavefronts, at most 80 or 64 registers, so the neighbours' values are loaded
// where the scattering's operands are not live.  With the traces and the face
// contraction in LDS and no bound (columns of 5 x 5 x 80): 4,096 columns mixed
// 51.7 -> 43.2 us, FP32 64 -> 60 us, FP64 97 -> 89 us; 1,024 columns mixed
// 16.2 -> 14.7 us.
template <typename T, typename A, int PREC, int N, int NTH, int NC, int H,
          int UTHREADS = u_threads<NTH, NC, H>()>
__global__ __launch_bounds__(UTHREADS, PREC == RTX_PREC_F64 ? 6 : 8)
void k_uniform(DevMesh m, uint32_t ops, int accumulate, const int4 *__restrict__ src,
               const T *__restrict__ x, T *__restrict__ y) {
    constexpr int NSP = N * N, NA = NC * NTH, NCD = NSP * NA, CD = NSP * NTH;
    constexpr int OC = NC / H;                 // cells per part
    constexpr int NOA = OC * NTH;
    constexpr int MT = (NSP + 15) / 16;
    constexpr int NTILE = (NOA + 15) / 16;     // output-angle tiles of the part
    constexpr int NKS = (NA + 3) / 4;          // f64/f32 k-steps
    constexpr int NKB = (NA + 15) / 16;        // bf16 k-steps
    // DOF passes t = t0 + u XS over a column (cell-major, CD DOFs per cell):
    // a pass covers CPP whole cells and a thread keeps one in-cell position
    // in every pass, so its (node, angle) indices are computed once; threads
    // past CPP CD idle (t0 = NCD)
    static_assert(CD <= UTHREADS, "a cell fits the workgroup");
    constexpr int CPP = UTHREADS / CD;
    constexpr int XS = CPP * CD;
    constexpr int XU = (NCD + XS - 1) / XS;
    constexpr int YU = (OC + CPP - 1) / CPP;   // passes over the part's outputs
    // LDS rows per spatial node, angle-contiguous, strides from u_pad
    constexpr int NAP = u_pad(NA, NTH), NOAP = u_pad(NOA, NTH);
    static_assert(NTILE <= UTHREADS / 64, "one output-angle tile per wavefront");
    static_assert(NC % H == 0, "parts must split the cells evenly");
    extern __shared__ __align__(16) unsigned char u_lds[];
    A *xs = reinterpret_cast<A *>(u_lds);      // [NSP][NAP]: column x, angle A of node s
    A *ys = xs + NSP * NAP;                    // [NSP][NOAP]: part outputs
    // MIXED: [MT 16][NAPB] BF16 copy of the column (MFMA A operands)
    constexpr bool XB = PREC == RTX_PREC_MIXED;
    constexpr int NAPB = u_bf_stride(NA);
    constexpr size_t XB_OFF = u_bf_off(size_t(NSP * NAP + NSP * NOAP) * sizeof(A));
    uint16_t *xb = reinterpret_cast<uint16_t *>(u_lds + XB_OFF);
    __shared__ A cth[NA], sth[NA], cw[NA];
    __shared__ A flx[NA], fly[NA];             // x- and y-flux of each angle (u_inflow)
    __shared__ A kap[NSP], sgw[NSP];
    __shared__ A wx_[N], WD[N * N];
    __shared__ A dth_[NC];
    __shared__ int cbd[NC], cqd[NC];
    __shared__ int nfc[NSP];                   // u_node_faces of each spatial node
    // per part cell, the neighbours' first face nodes (-1: none) and masked ends
    __shared__ int4 nbr[OC];

    // workgroups go to the XCDs round-robin (b mod 8); XCD j takes the
    // contiguous columns [j cpx, (j + 1) cpx) in order, all parts of a column
    // together, so a column's neighbours in index order (its y-neighbours,
    // and its x-neighbours inside the run) are read through the same L2
    const int b = blockIdx.x;
    const int cpx = (m.ncol + UXCD - 1) / UXCD;
    const int slot = b / UXCD;
    const int h = slot % H, c = (b % UXCD) * cpx + slot / H;
    if (c >= m.ncol) return;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    // the plan admits a uniform bin only when columns are laid out
    // contiguously in index order, so no table lookup precedes the x loads
    const int k0 = c * NC;
    const int cdof = c * NCD;
    const int kk_lo = h * OC;
    const int own0 = kk_lo * CD;
    const bool restrict_ = (ops & RTX_OP_RESTRICT) != 0;
    const bool bconv = (ops & RTX_OP_BCONV) != 0;
    const double dx = m.col_geom[4 * c + 2] - m.col_geom[4 * c + 0];
    const double dy = m.col_geom[4 * c + 3] - m.col_geom[4 * c + 1];
    const int ga0 = c * NA;

    // ---- batched loads issued before any use
    typedef typename std::conditional<PREC == RTX_PREC_F64, double, float>::type EB;
    EB bpre[(PREC == RTX_PREC_MIXED) ? 1 : NKS];
    const int l16 = lane & 15, lg = lane >> 4;
    const int Rl = wave * 16 + l16;            // part-local output angle of this lane
    const bool rok = (wave < NTILE) && (Rl < NOA);
    const int R = kk_lo * NTH + Rl;
    // FP64 runs the scattering MFMA before the vector phases (phase 2) and
    // loads its B operands (G) at the end of phase 1, so that they do not
    // hold registers while the column is prefetched (72 VGPRs, 7 waves per
    // SIMD); FP32 and BF16 load them here with the column
    constexpr bool MFMA_FIRST = PREC == RTX_PREC_F64;
    auto load_b = [&]() {
        if constexpr (PREC != RTX_PREC_MIXED) {
            const EB *Gp = (PREC == RTX_PREC_F64) ? (const EB *)(m.G + m.col_G_off[c])
                                                  : (const EB *)(m.G_f + m.col_G_off[c]);
            const bool scat = (ops & RTX_OP_SCAT) != 0;
            if constexpr (NA % 4 == 0 && NOA % 16 == 0) {
                // every lane of a scattering wave has an in-range operand and
                // the other waves never read them: one wave-uniform branch,
                // no per-lane masks or zero fills
                if (scat && wave < NTILE) {
                    const EB *Gl = Gp + size_t(lg) * NA + R;
#pragma unroll
                    for (int u = 0; u < NKS; ++u) bpre[u] = Gl[size_t(u) * 4 * NA];
                }
            } else {
#pragma unroll
                for (int u = 0; u < NKS; ++u) {
                    const int Ak = u * 4 + lg;
                    bpre[u] = (scat && rok && Ak < NA) ? Gp[size_t(Ak) * NA + R] : EB(0);
                }
            }
        }
    };
    if constexpr (!MFMA_FIRST) load_b();
    const int t0 = tid < XS ? tid : NCD;
    A xv[XU];
#pragma unroll
    for (int u = 0; u < XU; ++u) {
        const int t = t0 + u * XS;
        xv[u] = (t < NCD) ? A(x[cdof + t]) : A(0);
    }
    double r_c = 0, r_s = 0, r_w = 0, r_ag = 0, r_kap = 0, r_sig = 0, r_wd = 0, r_g = 0;
    int r_bd = 0, r_q = -1;
    int4 r_nbr = make_int4(-1, -1, 0, 0);
    if (tid < NA) {
        r_c = m.ang_trig[3 * (ga0 + tid)];
        r_s = m.ang_trig[3 * (ga0 + tid) + 1];
        r_w = m.ang_trig[3 * (ga0 + tid) + 2];
        const int k = k0 + tid / NTH;
        r_ag = m.cell_geom[2 * k + 1] - m.cell_geom[2 * k];
    }
    if (tid < NSP) {
        r_kap = m.kappa[c * NSP + tid];
        r_sig = m.sigma[c * NSP + tid];
    }
    if (tid < N * N) {
        const int p = tid / N, i = tid % N;
        r_wd = m.lgl_w[N * UNM + i] * m.lgl_D[(size_t(N) * UNM + p) * UNM + i];
    }
    if (tid < NC) {
        const int k = k0 + tid;
        r_bd = m.cell_bdry[k];
        r_q = m.cell_quad[k];
        r_g = m.cell_geom[2 * k + 1] - m.cell_geom[2 * k];
    }
    if (bconv && tid < OC) r_nbr = src[k0 + kk_lo + tid];
    if (tid < NA) {
        cth[tid] = A(r_c);
        sth[tid] = A(r_s);
        cw[tid] = A(r_w);
        flx[tid] = A(dy * 0.25 * r_ag * r_w * r_c);
        fly[tid] = A(dx * 0.25 * r_ag * r_w * r_s);
    }
    if (tid < NSP) {
        kap[tid] = A(r_kap);
        sgw[tid] = A(dx * dy * m.lgl_w[N * UNM + tid / N] * m.lgl_w[N * UNM + tid % N] * r_sig);
    }
    if (tid < N * N) WD[tid] = A(r_wd);
    if (tid < N) wx_[tid] = A(m.lgl_w[N * UNM + tid]);
    if (tid < NSP) nfc[tid] = u_node_faces(tid / N, tid % N, N);
    if (tid < NC) {
        cbd[tid] = restrict_ ? r_bd : 0;
        cqd[tid] = r_q;
        dth_[tid] = A(r_g);
    }
    if (tid < OC) nbr[tid] = r_nbr;
    __syncthreads();

    // ---- the neighbours' values of this thread's outputs, in flight until the
    // write-back: after the scattering in FP64 and before it in FP32, where its
    // operands hold registers (loaded with the column they spill), with the
    // column in mixed precision
    const int le = tid % CD, sne = le / NTH, ae = le % NTH, ie = sne / N, je = sne % N;
    A xi[YU], yi[YU];
    auto load_inflow = [&]() {
        int ax[YU], ay[YU];
#pragma unroll
        for (int u = 0; u < YU; ++u) {
            const int kl = tid / CD + u * CPP;
            ax[u] = ay[u] = -1;
            if (tid < XS && kl < OC) {
                const int4 nb = nbr[kl];
                const UFaces f(cqd[kk_lo + kl]);
                const int mk = restrict_ ? nb.z : 0;
                if (ie == (f.Fx == 0 ? 0 : N - 1) && nb.x >= 0 &&
                    !(je == 0 && (mk & 1)) && !(je == N - 1 && (mk & 2)))
                    ax[u] = nb.x + je * NTH + ae;
                if (je == (f.Fy == 1 ? 0 : N - 1) && nb.y >= 0 &&
                    !(ie == 0 && (mk & 4)) && !(ie == N - 1 && (mk & 8)))
                    ay[u] = nb.y + ie * N * NTH + ae;
            }
        }
#pragma unroll
        for (int u = 0; u < YU; ++u) {
            xi[u] = ax[u] >= 0 ? A(x[ax[u]]) : A(0);
            yi[u] = ay[u] >= 0 ? A(x[ay[u]]) : A(0);
        }
    };
    if constexpr (XB) load_inflow();

    // ---- phase 1: column input (masked)
    {
        const int lt0 = t0 % CD, sn0 = lt0 / NTH, a0 = lt0 % NTH, nf0 = nfc[sn0 < NSP ? sn0 : 0];
#pragma unroll
        for (int u = 0; u < XU; ++u) {
            const int t = t0 + u * XS;
            if (t < NCD) {
                A v = xv[u];
                const int kk = t0 / CD + u * CPP;
                if (cbd[kk] & nf0) v = A(0);   // cbd is 0 without RESTRICT
                xs[sn0 * NAP + kk * NTH + a0] = v;
                if constexpr (XB) xb[sn0 * NAPB + kk * NTH + a0] = u_bf16(float(v));
            }
        }
    }
    if constexpr (XB) {
        // zero the BF16 tile's padding: angles [NA, NKB 16) of the NSP
        // nodes, then every angle of the rows [NSP, MT 16)
        constexpr int PC = NKB * 16 - NA, PR = (MT * 16 - NSP) * NKB * 16;
        if constexpr (PC > 0)
            for (int e = tid; e < NSP * PC; e += UTHREADS) xb[(e / PC) * NAPB + NA + e % PC] = 0;
        for (int e = tid; e < PR; e += UTHREADS)
            xb[(NSP + e / (NKB * 16)) * NAPB + e % (NKB * 16)] = 0;
    }
    if constexpr (MFMA_FIRST) load_b();
    __syncthreads();

    // ---- scattering for the part's output angles on MFMA, into registers,
    // subtracted from the outputs in phase 3.  In FP64 it is issued here,
    // before phase 2, so the matrix pipe runs while the cell-local terms go
    // through the vector units (measured faster); in FP32 and BF16, whose MFMA
    // work is short and whose operand conversion competes with phase 2, it
    // runs after it (measured faster).
    typedef typename std::conditional<PREC == RTX_PREC_F64, u_dbl4, u_flt4>::type acc4;
    constexpr bool EARLY = MFMA_FIRST;
    acc4 sacc[MT];
    const bool scat_w = (ops & RTX_OP_SCAT) && wave < NTILE;
#pragma unroll
    for (int t = 0; t < MT; ++t) sacc[t] = acc4{0, 0, 0, 0};
    auto scatter = [&]() {
        if constexpr (PREC == RTX_PREC_F64 || PREC == RTX_PREC_F32) {
            // two accumulator chains per tile (even / odd k-steps) halve the
            // dependent MFMA chain
            constexpr bool TWO = !EARLY;
            acc4 acc2[MT];
#pragma unroll
            for (int t = 0; t < MT; ++t) acc2[t] = acc4{0, 0, 0, 0};
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                const int Ak = ks * 4 + lg;
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    const int s = t * 16 + l16;
                    const EB a = (Ak < NA && s < NSP) ? EB(xs[s * NAP + Ak]) : EB(0);
                    acc4 &dst = (TWO && (ks & 1)) ? acc2[t] : sacc[t];
                    if constexpr (PREC == RTX_PREC_F64)
                        dst = __builtin_amdgcn_mfma_f64_16x16x4f64(a, bpre[ks], dst, 0, 0, 0);
                    else
                        dst = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bpre[ks], dst, 0, 0, 0);
                }
            }
            if constexpr (TWO) {
#pragma unroll
                for (int t = 0; t < MT; ++t) sacc[t] += acc2[t];
            }
        } else {   // MIXED: BF16 operands, FP32 accumulation
            const uint16_t *G = m.G_bf16 + m.col_G_off[c];
            u_sht4 bv[NKB];
#pragma unroll
            for (int ks = 0; ks < NKB; ++ks)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int Ak = ks * 16 + 4 * lg + u;
                    bv[ks][u] = (rok && Ak < NA) ? short(G[size_t(Ak) * NA + R]) : short(0);
                }
#pragma unroll
            for (int ks = 0; ks < NKB; ++ks) {
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    const int s = t * 16 + l16;
                    // four consecutive angles of node s, zero past NA or NSP
                    const u_sht4 av = *reinterpret_cast<const u_sht4 *>(xb + s * NAPB + ks * 16 + 4 * lg);
                    sacc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, bv[ks], sacc[t], 0, 0, 0);
                }
            }
        }
    };
    if (EARLY && scat_w) scatter();
    if constexpr (EARLY) load_inflow();

    // ---- phase 2: cell-local terms on the part's DOFs, by lines of nodes:
    // pass x: one (cell, q, angle) line per thread reads x[0..N-1][q] once
    // and writes mass, outflow faces and the x-derivative term of all N
    // nodes; pass y: one (cell, p, angle) line adds the y-derivative term
    {
        constexpr int NLINE = OC * N * NTH;
        const A cm = A(dx * dy * 0.125);
        for (int e = tid; e < NLINE; e += UTHREADS) {
            // line (q, part angle oa): consecutive lanes read and write
            // consecutive angles of one node row
            const int q = e / NOA, oa0 = e % NOA, kl = oa0 / NTH, r = oa0 % NTH;
            const int kk = kk_lo + kl, ca = kk * NTH + r, oa = kl * NTH + r;
            const A dth = dth_[kk], wr = cw[ca], c_ = cth[ca], s_ = sth[ca];
            const int quad = cqd[kk];
            A xl[N];
#pragma unroll
            for (int i = 0; i < N; ++i) xl[i] = xs[(i * N + q) * NAP + ca];
            const A cx = A(dy * 0.25) * dth * wx_[q] * wr * c_;
            // outflow faces quad and quad + 1 of the line's cell: one x-face
            // (F even) and one y-face (F odd), added in that face order, each
            // term's products in the order of the per-node formula
            // A((F odd ? dx : dy) / 4) dth (F odd ? w_p : w_q) w_r Theta_F x.
            // The x-face adds a per-line constant at one end node; the
            // y-face adds to every node when q is its end (yon).
            const bool obc = bconv && quad >= 0;
            const bool yfirst = (quad & 1) != 0;
            const int Fx = yfirst ? ((quad + 1) & 3) : quad, Fy = yfirst ? quad : ((quad + 1) & 3);
            const A xtf = Fx == 0 ? c_ : -c_, ytf = Fy == 1 ? s_ : -s_;
            const A xb = A(dy * 0.25) * dth * wx_[q] * wr * xtf;
            const A yb = A(dx * 0.25) * dth;
            const int xtg = Fx == 0 ? N - 1 : 0;
            const bool yon = q == (Fy == 1 ? N - 1 : 0);
#pragma unroll
            for (int pp = 0; pp < N; ++pp) {
                A acc = A(0);
                const A xn = xl[pp];
                if (ops & RTX_OP_MASS) acc += cm * dth * wx_[pp] * wx_[q] * wr * kap[pp * N + q] * xn;
                if (ops & RTX_OP_QUADW) acc += cm * dth * wx_[pp] * wx_[q] * wr * xn;
                if (ops & RTX_OP_ICONV) {
                    A sx = A(0);
#pragma unroll
                    for (int i = 0; i < N; ++i) sx += WD[pp * N + i] * xl[i];
                    acc -= cx * sx;
                }
                if (obc) {
                    const A yt = yb * wx_[pp] * wr * ytf * xn;
                    if (yfirst && yon) acc += yt;
                    if (pp == xtg) acc += xb * xn;
                    if (!yfirst && yon) acc += yt;
                }
                ys[(pp * N + q) * NOAP + oa] = acc;
            }
        }
        if (ops & RTX_OP_ICONV) {
            __syncthreads();
            for (int e = tid; e < NLINE; e += UTHREADS) {
                const int pp = e / NOA, oa0 = e % NOA, kl = oa0 / NTH, r = oa0 % NTH;
                const int kk = kk_lo + kl, ca = kk * NTH + r, oa = kl * NTH + r;
                A xl[N];
#pragma unroll
                for (int j = 0; j < N; ++j) xl[j] = xs[(pp * N + j) * NAP + ca];
                const A cy = A(dx * 0.25) * dth_[kk] * wx_[pp] * cw[ca] * sth[ca];
#pragma unroll
                for (int q = 0; q < N; ++q) {
                    A sy = A(0);
#pragma unroll
                    for (int j = 0; j < N; ++j) sy += WD[q * N + j] * xl[j];
                    ys[(pp * N + q) * NOAP + oa] -= cy * sy;
                }
            }
        }
    }
    __syncthreads();

    // ---- phase 3: the scattering, subtracted from the outputs
    if constexpr (!EARLY && !XB) load_inflow();
    if (!EARLY && scat_w) scatter();
    if (scat_w && rok) {
#pragma unroll
        for (int t = 0; t < MT; ++t) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int s = t * 16 + ((PREC == RTX_PREC_F64) ? (lg + 4 * v) : (4 * lg + v));
                if (s < NSP) ys[s * NOAP + Rl] -= sgw[s] * A(sacc[t][v]);
            }
        }
    }
    __syncthreads();

    // ---- phase 4: the inflow through the x-face, then the y-face, and the
    // write-back of the part's DOFs by whole-cell passes as in phase 1
    if (tid >= XS) return;
#pragma unroll
    for (int u = 0; u < YU; ++u) {
        const int kl = tid / CD + u * CPP;
        if (kl >= OC) break;
        const int kk = kk_lo + kl, ca = kk * NTH + ae, t = own0 + kl * CD + le;
        const bool masked = (cbd[kk] & nfc[sne]) != 0;
        A v = ys[sne * NOAP + kl * NTH + ae];
        if (bconv) {
            const UFaces f(cqd[kk]);
            if (ie == (f.Fx == 0 ? 0 : N - 1)) v += u_inflow(flx[ca], f.Fx == 0, wx_[je], xi[u]);
            if (je == (f.Fy == 1 ? 0 : N - 1)) v += u_inflow(fly[ca], f.Fy == 1, wx_[ie], yi[u]);
        }
        if (masked) v = A(0);
        if (accumulate) {
            if (!masked) y[cdof + t] = T(A(y[cdof + t]) + v);
        } else {
            y[cdof + t] = T(v);
        }
    }
}

// Waves of the output-layout kernel: one per 16-wide output-angle tile, at
// least four (the loads and the trace and flux passes use every thread).
template <int NTH, int NC>
constexpr int ue_waves() {
    return (NC * NTH + 15) / 16 > 4 ? (NC * NTH + 15) / 16 : 4;
}

// The same operator on one whole column per workgroup, with every term of an
// output computed where the scattering MFMA leaves it: lane (l16, lg) of wave
// w owns output angle R = 16 w + l16 and the nodes of its accumulator rows,
// and adds to the MFMA result the mass, convection, outflow and inflow-face
// terms of those (node, angle) outputs in the order k_uniform adds them.  The
// two agree to rounding: here the inflow is the neighbours' traces contracted
// with E^s and E^theta, there its diagonal alone.  No output tile in LDS: the
// column tile, the traces and the flux slots are all the LDS it needs, so more
// columns are resident per CU (5 x 5 x 80: 34 KB, four per CU, 1,024 columns in
// one round).  The outputs go through the dead column tile for a coalesced
// store.
template <typename T, typename A, int PREC, int N, int NTH, int NC,
          int ETHREADS = 64 * ue_waves<NTH, NC>()>
// at least as many waves per SIMD as the workgroup has waves: four columns
// per CU (5 x 5 x 80: 5 waves per SIMD, at most 102 VGPRs)
__global__ __launch_bounds__(ETHREADS, ETHREADS / 64) void k_uniform_e(DevMesh m, uint32_t ops, int accumulate,
                                                        const T *__restrict__ x,
                                                        T *__restrict__ y, int nlink_lds) {
    constexpr int NSP = N * N, NA = NC * NTH, NCD = NSP * NA, CD = NSP * NTH;
    constexpr int MT = (NSP + 15) / 16;
    constexpr int NTILE = (NA + 15) / 16;
    constexpr int NKS = (NA + 3) / 4;
    constexpr int NKB = (NA + 15) / 16;
    constexpr int MAXL = 4 * NC;
    constexpr int TRL = N * NTH;
    constexpr int CPP = CD <= ETHREADS ? ETHREADS / CD : 0;
    constexpr int XS = CPP ? CPP * CD : ETHREADS;
    constexpr int XU = (NCD + XS - 1) / XS;
    constexpr int LPP = ETHREADS / TRL;
    constexpr int TS = LPP * TRL;
    constexpr int NAP = u_pad(NA, NTH);
    static_assert(NTILE <= ETHREADS / 64, "one output-angle tile per wavefront");
    static_assert(NSP * NAP >= NCD, "the column tile stages the outputs");
    extern __shared__ __align__(16) unsigned char u_lds[];
    A *xs = reinterpret_cast<A *>(u_lds);      // [NSP][NAP]: column x, angle A of node s
    constexpr bool XB = PREC == RTX_PREC_MIXED;
    constexpr int NAPB = u_bf_stride(NA);
    constexpr size_t XB_OFF = u_bf_off(size_t(NSP * NAP) * sizeof(A));
    uint16_t *xb = reinterpret_cast<uint16_t *>(u_lds + XB_OFF);
    A *tr = XB ? reinterpret_cast<A *>(u_lds + XB_OFF + u_bf_bytes(NSP, NA)) : xs + NSP * NAP;
    A *fl = tr + nlink_lds * TRL;
    __shared__ A cth[NA], sth[NA], cw[NA];
    __shared__ A kap[NSP], sgw[NSP];
    __shared__ A wx_[N], WD[N * N];
    __shared__ A dth_[NC];
    __shared__ int cbd[NC], cqd[NC];
    __shared__ int nfc[NSP];
    __shared__ int l_src[MAXL], l_meta[MAXL], l_es[MAXL], l_et[MAXL];
    __shared__ int cfx[NC], cfy[NC];

    // XCD j takes the contiguous columns [j cpx, (j + 1) cpx)
    const int b = blockIdx.x;
    const int cpx = (m.ncol + UXCD - 1) / UXCD;
    const int c = (b % UXCD) * cpx + b / UXCD;
    if (c >= m.ncol) return;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int k0 = c * NC;
    const int cdof = c * NCD;
    const int L0 = m.link_start[k0];
    const int nl = m.link_start[k0 + NC] - L0;
    const bool restrict_ = (ops & RTX_OP_RESTRICT) != 0;
    const bool bconv = (ops & RTX_OP_BCONV) != 0;
    const double dx = m.col_geom[4 * c + 2] - m.col_geom[4 * c + 0];
    const double dy = m.col_geom[4 * c + 3] - m.col_geom[4 * c + 1];
    const int ga0 = c * NA;

    // ---- batched loads issued before any use
    typedef typename std::conditional<PREC == RTX_PREC_F64, double, float>::type EB;
    EB bpre[(PREC == RTX_PREC_MIXED) ? 1 : NKS];
    const int l16 = lane & 15, lg = lane >> 4;
    const int R = wave * 16 + l16;             // output angle of this lane
    const bool rok = (wave < NTILE) && (R < NA);
    constexpr bool MFMA_FIRST = PREC == RTX_PREC_F64;
    auto load_b = [&]() {
        if constexpr (PREC != RTX_PREC_MIXED) {
            const EB *Gp = (PREC == RTX_PREC_F64) ? (const EB *)(m.G + m.col_G_off[c])
                                                  : (const EB *)(m.G_f + m.col_G_off[c]);
            const bool scat = (ops & RTX_OP_SCAT) != 0;
            if constexpr (NA % 16 == 0) {
                if (scat && wave < NTILE) {
                    const EB *Gl = Gp + size_t(lg) * NA + R;
#pragma unroll
                    for (int u = 0; u < NKS; ++u) bpre[u] = Gl[size_t(u) * 4 * NA];
                }
            } else {
#pragma unroll
                for (int u = 0; u < NKS; ++u) {
                    const int Ak = u * 4 + lg;
                    bpre[u] = (scat && rok && Ak < NA) ? Gp[size_t(Ak) * NA + R] : EB(0);
                }
            }
        }
    };
    if constexpr (!MFMA_FIRST) load_b();
    const int t0 = tid < XS ? tid : NCD;
    A xv[XU];
#pragma unroll
    for (int u = 0; u < XU; ++u) {
        const int t = t0 + u * XS;
        xv[u] = (t < NCD) ? A(x[cdof + t]) : A(0);
    }
    // the tables' loads are unconditional (indices clamped to the last
    // entry; only threads in range store them below), so they all go out
    // before the first wait instead of one branch's loads at a time
    const int tA = tid < NA ? tid : NA - 1, tS = tid < NSP ? tid : NSP - 1;
    const int tD = tid < N * N ? tid : N * N - 1, tC = tid < NC ? tid : NC - 1;
    const double r_c = m.ang_trig[3 * (ga0 + tA)];
    const double r_s = m.ang_trig[3 * (ga0 + tA) + 1];
    const double r_w = m.ang_trig[3 * (ga0 + tA) + 2];
    const double r_kap = m.kappa[c * NSP + tS];
    const double r_sig = m.sigma[c * NSP + tS];
    const double r_wd = m.lgl_w[N * UNM + tD % N] *
                        m.lgl_D[(size_t(N) * UNM + tD / N) * UNM + tD % N];
    const int r_bd = m.cell_bdry[k0 + tC];
    const int r_q = m.cell_quad[k0 + tC];
    const double r_g = m.cell_geom[2 * (k0 + tC) + 1] - m.cell_geom[2 * (k0 + tC)];
    const double r_wp = m.lgl_w[N * UNM + tS / N], r_wq = m.lgl_w[N * UNM + tS % N];
    const double r_wx = m.lgl_w[N * UNM + (tid < N ? tid : N - 1)];
    int r_src = 0, r_meta = 0, r_es = 0, r_et = 0;
    if (bconv && tid < nl) {
        const int l = L0 + tid;
        r_src = m.link_meta[4 * l + 0];
        r_meta = m.link_meta[4 * l + 1];
        r_es = m.link_Es_off[l];
        r_et = m.link_Eth_off[l];
    }
    if (tid < NA) {
        cth[tid] = A(r_c);
        sth[tid] = A(r_s);
        cw[tid] = A(r_w);
    }
    if (tid < NSP) {
        kap[tid] = A(r_kap);
        sgw[tid] = A(dx * dy * r_wp * r_wq * r_sig);
    }
    if (tid < N * N) WD[tid] = A(r_wd);
    if (tid < N) wx_[tid] = A(r_wx);
    if (tid < NSP) nfc[tid] = u_node_faces(tid / N, tid % N, N);
    if (tid < NC) {
        cbd[tid] = restrict_ ? r_bd : 0;
        cqd[tid] = r_q;
        dth_[tid] = A(r_g);
        cfx[tid] = 0;
        cfy[tid] = 0;
    }
    if (bconv && tid < nl) {
        l_src[tid] = r_src;
        l_meta[tid] = r_meta;
        l_es[tid] = r_es;
        l_et[tid] = r_et;
    }
    __syncthreads();
    if (bconv && tid < nl) {
        const int kl = r_meta >> 18, F = r_meta & 3;   // column-local target cell
        const int slots = (tid * TRL) << 4;
        if (F & 1) cfy[kl] = slots | (1 + (F == 1 ? N - 1 : 0));
        else cfx[kl] = slots | (1 + (F == 0 ? N - 1 : 0));
    }

    // ---- phase 1: column input (masked) and the neighbour traces
    {
        const int lt0 = t0 % CD, sn0 = lt0 / NTH, a0 = lt0 % NTH, nf0 = nfc[sn0 < NSP ? sn0 : 0];
#pragma unroll
        for (int u = 0; u < XU; ++u) {
            const int t = t0 + u * XS;
            if (t < NCD) {
                A v = xv[u];
                int kk, sn, a, nf;
                if constexpr (CPP > 0) {
                    kk = t0 / CD + u * CPP;
                    sn = sn0;
                    a = a0;
                    nf = nf0;
                } else {
                    const int lt = t % CD;
                    kk = t / CD;
                    sn = lt / NTH;
                    a = lt % NTH;
                    nf = nfc[sn];
                }
                if (cbd[kk] & nf) v = A(0);
                xs[sn * NAP + kk * NTH + a] = v;
                if constexpr (XB) xb[sn * NAPB + kk * NTH + a] = u_bf16(float(v));
            }
        }
    }
    if constexpr (XB) {
        constexpr int PC = NKB * 16 - NA, PR = (MT * 16 - NSP) * NKB * 16;
        if constexpr (PC > 0)
            for (int e = tid; e < NSP * PC; e += ETHREADS) xb[(e / PC) * NAPB + NA + e % PC] = 0;
        for (int e = tid; e < PR; e += ETHREADS)
            xb[(NSP + e / (NKB * 16)) * NAPB + e % (NKB * 16)] = 0;
    }
    if (bconv) {
        constexpr int TU = (MAXL * TRL + TS - 1) / TS;
        const int e0 = tid < TS ? tid : MAXL * TRL;
        const int le = e0 % TRL, m1 = le / NTH, a = le % NTH;
        int addr[TU];
        bool zero[TU];
        A v[TU];
#pragma unroll
        for (int u = 0; u < TU; ++u) {
            const int li = e0 / TRL + u * LPP;
            addr[u] = -1;
            zero[u] = false;
            if (li < nl) {
                const int w1 = l_meta[li];
                const int F = w1 & 3, bd1 = restrict_ ? ((w1 >> 14) & 15) : 0;
                int i1, j1;
                if (F == 0) { i1 = 0; j1 = m1; }
                else if (F == 2) { i1 = N - 1; j1 = m1; }
                else if (F == 1) { i1 = m1; j1 = 0; }
                else { i1 = m1; j1 = N - 1; }
                addr[u] = l_src[li] + (i1 * N + j1) * NTH + a;
                zero[u] = (bd1 & nfc[i1 * N + j1]) != 0;
            }
        }
#pragma unroll
        for (int u = 0; u < TU; ++u) v[u] = (addr[u] >= 0) ? A(x[addr[u]]) : A(0);
#pragma unroll
        for (int u = 0; u < TU; ++u) {
            const int li = e0 / TRL + u * LPP;
            if (li < nl) tr[li * TRL + le] = zero[u] ? A(0) : v[u];
        }
    }
    if constexpr (MFMA_FIRST) load_b();
    __syncthreads();

    // ---- scattering on MFMA into registers: FP64 issues it first, FP32 and
    // BF16 after the flux pass (as k_uniform)
    typedef typename std::conditional<PREC == RTX_PREC_F64, u_dbl4, u_flt4>::type acc4;
    acc4 sacc[MT];
    const bool scat_w = (ops & RTX_OP_SCAT) && wave < NTILE;
#pragma unroll
    for (int t = 0; t < MT; ++t) sacc[t] = acc4{0, 0, 0, 0};
    auto scatter = [&]() {
        if constexpr (PREC == RTX_PREC_F64 || PREC == RTX_PREC_F32) {
            constexpr bool TWO = !MFMA_FIRST;
            acc4 acc2[MT];
#pragma unroll
            for (int t = 0; t < MT; ++t) acc2[t] = acc4{0, 0, 0, 0};
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                const int Ak = ks * 4 + lg;
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    const int s = t * 16 + l16;
                    const EB a = (Ak < NA && s < NSP) ? EB(xs[s * NAP + Ak]) : EB(0);
                    acc4 &dst = (TWO && (ks & 1)) ? acc2[t] : sacc[t];
                    if constexpr (PREC == RTX_PREC_F64)
                        dst = __builtin_amdgcn_mfma_f64_16x16x4f64(a, bpre[ks], dst, 0, 0, 0);
                    else
                        dst = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bpre[ks], dst, 0, 0, 0);
                }
            }
            if constexpr (TWO) {
#pragma unroll
                for (int t = 0; t < MT; ++t) sacc[t] += acc2[t];
            }
        } else {
            const uint16_t *G = m.G_bf16 + m.col_G_off[c];
            u_sht4 bv[NKB];
#pragma unroll
            for (int ks = 0; ks < NKB; ++ks)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int Ak = ks * 16 + 4 * lg + u;
                    bv[ks][u] = (rok && Ak < NA) ? short(G[size_t(Ak) * NA + R]) : short(0);
                }
#pragma unroll
            for (int ks = 0; ks < NKB; ++ks) {
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    const int s = t * 16 + l16;
                    const u_sht4 av = *reinterpret_cast<const u_sht4 *>(xb + s * NAPB + ks * 16 + 4 * lg);
                    sacc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, bv[ks], sacc[t], 0, 0, 0);
                }
            }
        }
    };
    if (MFMA_FIRST && scat_w) scatter();

    // ---- upwind inflow couplings, one (link, face node, angle) per thread,
    // into a flux slot of its own; a DOF's slots are added below in a fixed
    // order (its cell has at most one x-face and one y-face link)
    if (bconv) {
        const int f0 = tid < TS ? tid : MAXL * TRL;
        const int le = f0 % TRL, m0 = le / NTH, r = le % NTH;
        for (int li = f0 / TRL; li < nl; li += LPP) {
            const int w1 = l_meta[li];
            const int F = w1 & 3, kk = w1 >> 18;      // column-local target cell
            const double *Es = m.Es_pool + l_es[li];
            const double *Et = m.Eth_pool + l_et[li];
            A et[NTH], es[N];
#pragma unroll
            for (int a = 0; a < NTH; ++a) et[a] = A(Et[a * NTH + r]);
#pragma unroll
            for (int a = 0; a < N; ++a) es[a] = A(Es[a * N + m0]);
            const A *trl = tr + li * TRL;
            A acc = A(0);
#pragma unroll 1
            for (int m1 = 0; m1 < N; ++m1) {
                A inner = A(0);
#pragma unroll
                for (int a = 0; a < NTH; ++a) inner += et[a] * trl[m1 * NTH + a];
                acc += es[m1] * inner;
            }
            fl[li * TRL + le] = A(((F & 1) ? dx : dy) * 0.25) * dth_[kk] * acc;
        }
    }
    if (!MFMA_FIRST && scat_w) scatter();
    __syncthreads();

    // ---- every term of this lane's outputs, in k_uniform's order: mass,
    // x-derivative, outflow faces (phase 2 x-lines), y-derivative (y-lines),
    // scattering (phase 3), inflow faces x then y (phase 4)
    A outv[MT][4];
    if (wave < NTILE) {
        const int Rc = rok ? R : NA - 1;
        const int kk = Rc / NTH, r = Rc % NTH;
        const A dth = dth_[kk], wr = cw[Rc], c_ = cth[Rc], s_ = sth[Rc];
        const int quad = cqd[kk];
        const A cm = A(dx * dy * 0.125);
        const bool obc = bconv && quad >= 0;
        const bool yfirst = (quad & 1) != 0;
        const int Fx = yfirst ? ((quad + 1) & 3) : quad, Fy = yfirst ? quad : ((quad + 1) & 3);
        const A xtf = Fx == 0 ? c_ : -c_, ytf = Fy == 1 ? s_ : -s_;
        const A yb = A(dx * 0.25) * dth;
        const int xtg = Fx == 0 ? N - 1 : 0;
        const int fxs = cfx[kk], fys = cfy[kk];
#pragma unroll
        for (int t = 0; t < MT; ++t) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int s = t * 16 + ((PREC == RTX_PREC_F64) ? (lg + 4 * v) : (4 * lg + v));
                A acc = A(0);
                if (s < NSP) {
                    const int pp = s / N, q = s % N;
                    const A xn = xs[s * NAP + Rc];
                    if (ops & RTX_OP_MASS) acc += cm * dth * wx_[pp] * wx_[q] * wr * kap[pp * N + q] * xn;
                    if (ops & RTX_OP_QUADW) acc += cm * dth * wx_[pp] * wx_[q] * wr * xn;
                    if (ops & RTX_OP_ICONV) {
                        const A cx = A(dy * 0.25) * dth * wx_[q] * wr * c_;
                        A sx = A(0);
#pragma unroll
                        for (int i = 0; i < N; ++i) sx += WD[pp * N + i] * xs[(i * N + q) * NAP + Rc];
                        acc -= cx * sx;
                    }
                    if (obc) {
                        const A xbv = A(dy * 0.25) * dth * wx_[q] * wr * xtf;
                        const bool yon = q == (Fy == 1 ? N - 1 : 0);
                        const A yt = yb * wx_[pp] * wr * ytf * xn;
                        if (yfirst && yon) acc += yt;
                        if (pp == xtg) acc += xbv * xn;
                        if (!yfirst && yon) acc += yt;
                    }
                    if (ops & RTX_OP_ICONV) {
                        const A cy = A(dx * 0.25) * dth * wx_[pp] * wr * s_;
                        A sy = A(0);
#pragma unroll
                        for (int j = 0; j < N; ++j) sy += WD[q * N + j] * xs[(pp * N + j) * NAP + Rc];
                        acc -= cy * sy;
                    }
                    if (ops & RTX_OP_SCAT) acc -= sgw[s] * A(sacc[t][v]);
                    if (bconv) {
                        if (pp + 1 == (fxs & 15)) acc += fl[(fxs >> 4) + q * NTH + r];
                        if (q + 1 == (fys & 15)) acc += fl[(fys >> 4) + pp * NTH + r];
                    }
                }
                outv[t][v] = acc;
            }
        }
    }
    __syncthreads();
    // the outputs into the dead column tile in DOF order (cell, node, angle),
    // masked outputs as zero
    if (rok) {
        const int kk = R / NTH, r = R % NTH;
        const int cb = cbd[kk];
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int s = t * 16 + ((PREC == RTX_PREC_F64) ? (lg + 4 * v) : (4 * lg + v));
                if (s < NSP) xs[kk * CD + s * NTH + r] = (cb & nfc[s]) ? A(0) : outv[t][v];
            }
    }
    __syncthreads();
    // ---- coalesced write-back: 16-byte copies when y is overwritten in the
    // tile's type and aligned, else element by element (accumulate adds the
    // unmasked outputs only)
    constexpr int VW = 16 / sizeof(T);
    if constexpr (std::is_same<T, A>::value && NCD % (16 / sizeof(T)) == 0) {
        if (!accumulate && (reinterpret_cast<uintptr_t>(y + cdof) & 15) == 0) {
            typedef T V16 __attribute__((ext_vector_type(VW)));
            const V16 *src = reinterpret_cast<const V16 *>(xs);
            V16 *dst = reinterpret_cast<V16 *>(y + cdof);
            for (int e = tid; e < NCD / VW; e += ETHREADS) dst[e] = src[e];
            return;
        }
    }
    for (int e = tid; e < NCD; e += ETHREADS) {
        const int kk = e / CD, lt = e % CD, sn = lt / NTH;
        const bool masked = (cbd[kk] & nfc[sn]) != 0;
        const A v = masked ? A(0) : xs[e];
        if (accumulate) {
            if (!masked) y[cdof + e] = T(A(y[cdof + e]) + v);
        } else {
            y[cdof + e] = T(v);
        }
    }
}

template <typename T, typename A, int PREC, int N, int NTH, int NC>
int launch_e(rtx_plan *p, uint32_t ops, const void *dx, void *dy, hipStream_t st, int acc) {
    constexpr int NSP = N * N, NA = NC * NTH;
    constexpr int NAP = u_pad(NA, NTH);
    constexpr int MAXL = 4 * NC, TRL = N * NTH;
    RTX_CHECK(p->max_col_links <= MAXL, "uniform apply: %d links in a column (max %d)",
              p->max_col_links, MAXL);
    constexpr bool XB = PREC == RTX_PREC_MIXED;
    const size_t tiles = XB ? u_bf_off(size_t(NSP * NAP) * sizeof(A)) + u_bf_bytes(NSP, NA)
                            : size_t(NSP * NAP) * sizeof(A);
    const size_t lds = tiles + size_t(2 * p->max_col_links * TRL) * sizeof(A);
    auto kern = k_uniform_e<T, A, PREC, N, NTH, NC>;
    RTX_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                int(lds)));
    const int nblocks = ((p->m.ncol + UXCD - 1) / UXCD) * UXCD;
    kern<<<nblocks, 64 * ue_waves<NTH, NC>(), lds, st>>>(p->m, ops, acc, (const T *)dx, (T *)dy,
                                                         p->max_col_links);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

template <typename T, typename A, int PREC, int N, int NTH, int NC, int H>
int launch_one(rtx_plan *p, uint32_t ops, const void *dx, void *dy, hipStream_t st, int acc) {
    constexpr int NSP = N * N, NA = NC * NTH;
    constexpr int NAP = u_pad(NA, NTH), NOAP = u_pad((NC / H) * NTH, NTH);
    constexpr bool XB = PREC == RTX_PREC_MIXED;
    const size_t tiles = XB ? u_bf_off(size_t(NSP * NAP + NSP * NOAP) * sizeof(A)) + u_bf_bytes(NSP, NA)
                            : size_t(NSP * NAP + NSP * NOAP) * sizeof(A);
    const size_t lds = tiles;
    auto kern = k_uniform<T, A, PREC, N, NTH, NC, H>;
    RTX_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                int(lds)));
    const int nblocks = ((p->m.ncol + UXCD - 1) / UXCD) * UXCD * H;   // 8 cpx H
    kern<<<nblocks, u_threads<NTH, NC, H>(), lds, st>>>(p->m, ops, acc, p->uni_src, (const T *)dx,
                                                        (T *)dy);
    RTX_HIP(hipGetLastError());
    return RTX_OK;
}

// A part count H is valid for a shape when it divides the cells and the
// part's output angles fit one 16-wide tile per wavefront of the largest
// workgroup.
template <int NTH, int NC, int H>
constexpr bool u_valid() {
    return NC % H == 0 && ((NC / H) * NTH + 15) / 16 <= 512 / 64;
}

template <int N, int NTH, int NC, int H>
int launch_h(rtx_plan *p, uint32_t ops, int prec, const void *dx, void *dy, hipStream_t st,
             int acc) {
    if constexpr (u_valid<NTH, NC, H>()) {
        if (prec == RTX_PREC_F64)
            return launch_one<double, double, RTX_PREC_F64, N, NTH, NC, H>(p, ops, dx, dy, st, acc);
        if (prec == RTX_PREC_F32)
            return launch_one<float, float, RTX_PREC_F32, N, NTH, NC, H>(p, ops, dx, dy, st, acc);
        return launch_one<float, float, RTX_PREC_MIXED, N, NTH, NC, H>(p, ops, dx, dy, st, acc);
    } else {
        set_error("uniform apply: %d parts are not valid for this shape", H);
        return RTX_ERR_ARG;
    }
}

// Every column of the plan resident at once in the output-layout kernel
// (four workgroups per CU).
inline bool uniform_one_round(const rtx_plan *p) { return p->m.ncol <= 4 * p->n_cu; }

template <int N, int NTH, int NC>
int launch_shape(rtx_plan *p, uint32_t ops, int prec, const void *dx, void *dy, hipStream_t st,
                 int acc) {
    // default: FP64 runs the output-layout kernel when every column is
    // resident at once (four workgroups per CU; 1,024 columns of 5 x 5 x 80:
    // 26.4 us against 27.3 us), else the line-pass kernel, whose eight-wave
    // workgroups pipeline better over several rounds (4,096 columns: 89 us
    // against 109 us); FP32 and mixed run the line-pass kernel (1,024 columns
    // mixed: 14.7 us against 15.7 us).  A part count set by
    // rtx_set_uniform_parts or rtx_autotune selects the line-pass kernel
    // with that many parts.
    int H = p->uni_H;
    if (H == 0 && prec == RTX_PREC_F64 && uniform_one_round(p))
        return launch_e<double, double, RTX_PREC_F64, N, NTH, NC>(p, ops, dx, dy, st, acc);
    if (H == 0) H = u_valid<NTH, NC, 1>() ? 1 : (u_valid<NTH, NC, 2>() ? 2 : 4);
    if (H == 1) return launch_h<N, NTH, NC, 1>(p, ops, prec, dx, dy, st, acc);
    if (H == 2) return launch_h<N, NTH, NC, 2>(p, ops, prec, dx, dy, st, acc);
    return launch_h<N, NTH, NC, 4>(p, ops, prec, dx, dy, st, acc);
}

template <int N, int NTH, int NC>
int valid_parts_mask() {
    return (u_valid<NTH, NC, 1>() ? 1 : 0) | (u_valid<NTH, NC, 2>() ? 2 : 0) |
           (u_valid<NTH, NC, 4>() ? 4 : 0);
}

}  // namespace

// Shapes compiled into the library: (nodes per spatial direction, angular
// nodes per cell, cells per column).
int launch_uniform(rtx_plan *p, uint32_t ops, int prec, const void *dx, void *dy, hipStream_t st,
                   int acc) {
    const int N = p->uni_n, NTH = p->uni_nth, NC = p->uni_ncells;
#define RTX_SHAPE(a, b, c_) \
    if (N == a && NTH == b && NC == c_) return launch_shape<a, b, c_>(p, ops, prec, dx, dy, st, acc);
    RTX_SHAPE(5, 5, 16)
    RTX_SHAPE(4, 4, 16)
    RTX_SHAPE(4, 4, 4)
    RTX_SHAPE(3, 3, 8)
    RTX_SHAPE(5, 5, 8)
    RTX_SHAPE(4, 4, 8)
    RTX_SHAPE(3, 3, 4)
#undef RTX_SHAPE
    return 1;   // not compiled: caller falls back
}

int uniform_default_parts(const rtx_plan *p) {
    if (p->uni_H) return p->uni_H;
    const int mask = uniform_valid_parts(p);
    return (mask & 1) ? 1 : ((mask & 2) ? 2 : 4);
}

int uniform_valid_parts(const rtx_plan *p) {
    const int N = p->uni_n, NTH = p->uni_nth, NC = p->uni_ncells;
#define RTX_SHAPE(a, b, c_) \
    if (N == a && NTH == b && NC == c_) return valid_parts_mask<a, b, c_>();
    RTX_SHAPE(5, 5, 16)
    RTX_SHAPE(4, 4, 16)
    RTX_SHAPE(4, 4, 4)
    RTX_SHAPE(3, 3, 8)
    RTX_SHAPE(5, 5, 8)
    RTX_SHAPE(4, 4, 8)
    RTX_SHAPE(3, 3, 4)
#undef RTX_SHAPE
    return 0;
}

bool uniform_shape_compiled(int N, int NTH, int NC) {
    const int shapes[][3] = {{5, 5, 16}, {4, 4, 16}, {4, 4, 4}, {3, 3, 8},
                             {5, 5, 8},  {4, 4, 8},  {3, 3, 4}};
    for (auto &s : shapes)
        if (s[0] == N && s[1] == NTH && s[2] == NC) return true;
    return false;
}

}  // namespace rtx
