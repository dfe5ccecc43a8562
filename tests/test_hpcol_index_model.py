"""CPU model of the hp column kernels (``csrc/rtx_hpcol.hip``), test-only.

Restates what the host prepares (the packed cell and link records of the face
kernel, the flags and alike neighbours of the angles, the lists) and what
k_hp_flux and k_hpcol do with it: which face stores a corner node that two
faces share, the masked nodes, the angle-major LDS copy, the nodes that a
lane's matrix accumulators hold, the items of the wavefronts and the output
addresses.  Every index is checked against its buffer, every stored value is
stored once and every value read was stored, and the result is compared with
the oracle's assembled operator.
"""
import numpy as np
import pytest

from oracle import assemble as asm
from rtx import problems

NM = 10
WAVES, THREADS = 8, 512
MAX_CELLS = 64
STATIC_F64 = (2 * NM * NM + NM + NM * NM) * 8 + 64
CAP = 160 * 1024 - STATIC_F64


class F64:
    """v_mfma_f64_16x16x4f64: rows of an accumulator, and where row r is."""
    row = staticmethod(lambda lg, v: lg + 4 * v)
    group = staticmethod(lambda r: r & 3)
    reg = staticmethod(lambda r: r >> 2)


class F32:
    """The FP32 and BF16 shapes."""
    row = staticmethod(lambda lg, v: 4 * lg + v)
    group = staticmethod(lambda r: r >> 2)
    reg = staticmethod(lambda r: r & 3)


def hp_stride(na, kstep, c, M):
    n = (na + kstep - 1) // kstep * kstep
    return n + ((c - n) % M + M) % M


def hp_layout(nsp, na, prec, alike):
    """(S, NA, XSB, total bytes) of a column's dynamic LDS."""
    ea, kstep = (8 if prec == "f64" else 4), (16 if prec == "mixed" else 4)
    S, NA = nsp | 1, (na + kstep - 1) // kstep * kstep
    XSB = hp_stride(na, 16, 8, 16) if prec == "mixed" else 0
    o = (NA * S * ea + 15) & ~15
    o = (o + nsp * XSB * 2 + 15) & ~15
    o += 3 * na * ea + 2 * na * 4
    o = ((o + 7) & ~7) + (8 * na if alike else 0)
    return S, NA, XSB, (o + 15) & ~15


def on_bdry(bd, i, j, nx, ny):
    return bool(((bd & 1) and i == nx - 1) or ((bd & 2) and j == ny - 1) or
                ((bd & 4) and i == 0) or ((bd & 8) and j == 0))


def links_of(T, k):
    return range(int(T.link_start[k]), int(T.link_start[k + 1]))


def alike_cell(T, k):
    """(alike, first face nodes of the x- and y-neighbour, masked ends)."""
    c, quad = int(T.cell_col[k]), int(T.cell_quad[k])
    nx, ny, nt = int(T.col_nx[c]), int(T.col_ny[c]), int(T.cell_nth[k])
    src, masked = [-1, -1], 0
    if quad < 0:
        return False, src, masked
    a0 = int(T.col_ang_start[c]) + int(T.cell_ang_off[k])
    trig = T.ang_trig[3 * a0:3 * (a0 + nt)].reshape(nt, 3)
    for l in links_of(T, k):
        s, F = int(T.link_src[l]), int(T.link_face[l])
        c1, odd = int(T.cell_col[s]), F & 1
        if F not in ((quad + 2) & 3, (quad + 3) & 3) or src[odd] >= 0:
            return False, src, masked
        if (T.col_nx[c1], T.col_ny[c1], T.cell_nth[s]) != (nx, ny, nt):
            return False, src, masked
        n = nx if odd else ny
        es, et = int(T.link_Es_off[l]), int(T.link_Eth_off[l])
        Es, Et = T.Es_pool[es:es + n * n].reshape(n, n), T.Eth_pool[et:et + nt * nt].reshape(nt, nt)
        want = trig[:, 2] * trig[:, odd] * (1.0 if F < 2 else -1.0)
        if np.abs(Es - np.diag(T.lgl_w[n * NM:n * NM + n])).max() > 1e-13 or \
                np.abs(Et - np.diag(want)).max() > 1e-13:
            return False, src, masked
        bd = int(T.cell_bdry[s]) & 15
        if bd >> ((F + 2) & 3) & 1:
            return False, src, masked
        node = {2: (nx - 1) * ny, 3: ny - 1}.get(F, 0)
        src[odd] = int(T.cell_dof_off[s]) + node * nt
        masked |= ((bd >> (2 if odd else 3) & 1) | (bd >> (0 if odd else 1) & 1) << 1) << 2 * odd
    return True, src, masked


class Tables:
    """What hpcol_build prepares."""

    def __init__(self, T):
        self.T = T
        cells = [alike_cell(T, k) for k in range(T.ncell)]
        self.alike = 2 * sum(c[0] for c in cells) >= T.ncell
        self.direct = [self.alike and c[0] for c in cells]
        self.flag, self.src = [], []
        for k in range(T.ncell):
            lf = 0
            if not self.direct[k]:
                for l in links_of(T, k):
                    lf |= 1 << int(T.link_face[l])
            w = (int(T.cell_bdry[k]) & 15) | (int(T.cell_quad[k]) + 1) << 4 | lf << 8
            for r in range(int(T.cell_nth[k])):
                self.flag.append(w | (cells[k][2] << 12 if self.direct[k] else 0))
                self.src.append([s + r if self.direct[k] and s >= 0 else -1 for s in cells[k][1]])
        self.cells, self.links = [], []
        for k in range(T.ncell):
            if not self.direct[k]:
                self._records(k)

    def _records(self, k):
        T, c = self.T, int(self.T.cell_col[k])
        dx, dy = T.col_geom[c, 2] - T.col_geom[c, 0], T.col_geom[c, 3] - T.col_geom[c, 1]
        dth = T.cell_geom[k, 1] - T.cell_geom[k, 0]
        l0, lf, nl = len(self.links), 0, 0
        for F in range(4):
            for l in links_of(T, k):
                if int(T.link_face[l]) != F:
                    continue
                w1 = int(T.link_meta[4 * l + 1])
                nx1, ny1, nt1, bd1 = (w1 >> 2) & 15, (w1 >> 6) & 15, (w1 >> 10) & 15, (w1 >> 14) & 15
                n1 = nx1 if F & 1 else ny1
                fixed = 0 if F < 2 else (nx1 if F == 2 else ny1) - 1
                first = fixed * nt1 if F & 1 else fixed * ny1 * nt1
                stride = ny1 * nt1 if F & 1 else nt1
                mk = 0
                for m1 in range(n1):
                    i1, j1 = (m1, fixed) if F & 1 else (fixed, m1)
                    mk |= on_bdry(bd1, i1, j1, nx1, ny1) << m1
                rec1 = F | n1 << 2 | nt1 << 6 | stride << 10 | mk << 18
                assert stride < 256 and 0 <= rec1 < 2 ** 31
                self.links.append((int(T.link_meta[4 * l]) + first, rec1, int(T.link_Es_off[l]),
                                   int(T.link_Eth_off[l])))
                lf |= 1 << F
                nl += 1
        assert nl < 256
        w = nl | int(T.col_nx[c]) << 8 | int(T.cell_nth[k]) << 12 | \
            (int(T.cell_bdry[k]) & 15) << 16 | lf << 20 | int(T.col_ny[c]) << 24
        self.cells.append((dy * 0.25 * dth, dx * 0.25 * dth, int(T.cell_dof_off[k]), l0, w))


def flux_model(H, M, x, y, restrict, accumulate):
    """k_hp_flux: the inflow-face sums into y; returns which DOFs were stored."""
    T, stored = H.T, np.zeros(H.T.ndof, bool)
    for fx, fy, off, l0, w in H.cells:
        nl, nx, nt = w & 255, (w >> 8) & 15, (w >> 12) & 15
        bd, lf, ny = ((w >> 16) & 15) if restrict else 0, (w >> 20) & 15, (w >> 24) & 15
        c0, c1 = [np.zeros(nt) for _ in range(4)], [np.zeros(nt) for _ in range(4)]
        cur = None
        for i in range(nl):
            a, w1, es, et = H.links[l0 + i]
            F, n1, nt1, stride = w1 & 3, (w1 >> 2) & 15, (w1 >> 6) & 15, (w1 >> 10) & 255
            N = nx if F & 1 else ny
            at = a + np.arange(n1)[:, None] * stride + np.arange(nt1)
            assert at.min() >= 0 and at.max() < T.ndof and nt1 <= 12 and max(n1, N, nt) <= 16
            tr = x[at]
            if restrict:
                tr = np.where(((w1 >> (18 + np.arange(n1))) & 1)[:, None], 0.0, tr)
            assert es + n1 * N <= T.Es_pool.size and et + nt1 * nt <= T.Eth_pool.size
            # the K steps taken cover every face node of the neighbour
            rows = {M.row(lg, s) for s in range(4) if M.row(0, s) < n1 for lg in range(4)}
            assert set(range(n1)) <= rows
            inn = tr @ T.Eth_pool[et:et + nt1 * nt].reshape(nt1, nt)
            f = T.Es_pool[es:es + n1 * N].reshape(n1, N).T @ inn
            cur = f if cur is None else cur + f
            if i + 1 < nl and H.links[l0 + i + 1][1] & 3 == F:
                continue
            cur = cur * (fy if F & 1 else fx)
            f0, f1 = (2, 0) if F & 1 else (3, 1)
            assert (M.group(N - 1), M.reg(N - 1)) in [(g, v) for g in range(4) for v in range(4)
                                                      if M.row(g, v) == N - 1]
            first, last = cur[0].copy(), cur[N - 1].copy()
            if F == 0:
                c1[1], c1[3] = last, first
            if F == 1:
                c1[2] = first
            if F == 2:
                c0[3] = first
            cur[0] += c0[3] if F == 3 else 0.0
            cur[N - 1] += c1[F] if F else 0.0
            skip = {0: (bd >> f0) & 1 or ((lf >> f0) & 1 and f0 > F),
                    N - 1: (bd >> f1) & 1 or ((lf >> f1) & 1 and f1 > F)}
            base = off + {0: (nx - 1) * ny, 1: ny - 1}.get(F, 0) * nt
            for m0 in range(N):
                if skip.get(m0):
                    continue
                d = base + m0 * (ny if F & 1 else 1) * nt + np.arange(nt)
                assert off <= d[0] and d[-1] < off + nx * ny * nt and not stored[d].any()
                y[d] = y[d] + cur[m0] if accumulate else cur[m0]
                stored[d] = True
            cur = None
    return stored


def column_model(H, c, kappa, sigma, G, G_off, x, y, stored, restrict, accumulate):
    """k_hpcol on column c."""
    T = H.T
    k0, k1 = int(T.col_cell_start[c]), int(T.col_cell_start[c + 1])
    N, NY = int(T.col_nx[c]), int(T.col_ny[c])
    nsp, na = N * NY, int(T.col_nang[c])
    assert k1 - k0 <= MAX_CELLS and min(N, NY) >= 3
    cdof, ga0, sp0 = int(T.cell_dof_off[k0]), int(T.col_ang_start[c]), int(T.col_sp_off[c])
    S, NA, _, _ = hp_layout(nsp, na, "f64", H.alike)
    dx, dy = T.col_geom[c, 2] - T.col_geom[c, 0], T.col_geom[c, 3] - T.col_geom[c, 1]
    pack = [int(v) for v in T.ang_pack[ga0:ga0 + na]]
    flag = H.flag[ga0:ga0 + na]
    # x -> LDS: DOF t belongs to the cell of angle t // nsp
    xs = np.full(NA * S, np.nan)
    for t in range(nsp * na):
        ta = t // nsp
        w = pack[ta]
        nt, ao = (w >> 20) & 31, ta - (w >> 25)
        s, a = divmod(t - nsp * ao, nt)
        assert 0 <= s < nsp and ao + a < na and np.isnan(xs[(ao + a) * S + s])
        bd = flag[ta] & 15 if restrict else 0
        xs[(ao + a) * S + s] = 0.0 if on_bdry(bd, s // NY, s % NY, N, NY) else x[cdof + t]
    X = xs.reshape(NA, S)[:na, :nsp]
    assert not np.isnan(X).any()
    g0 = int(G_off[c])
    scat = G[g0:g0 + na * na].reshape(na, na).T @ X              # [R, s]
    w1 = {n: T.lgl_w[n * NM:n * NM + n] for n in (N, NY)}
    wd = {n: np.array([[w1[n][i] * T.lgl_D[(n * NM + p) * NM + i] for i in range(n)]
                       for p in range(n)]) for n in (N, NY)}
    dth_of = np.repeat(T.cell_geom[k0:k1, 1] - T.cell_geom[k0:k1, 0], T.cell_nth[k0:k1])
    for R in range(na):
        w, f, dth = pack[R], flag[R], dth_of[R]
        nt, bd, quad = (w >> 20) & 31, (f & 15) if restrict else 0, ((f >> 4) & 7) - 1
        lf, mk = (f >> 8) & 15, (f >> 12) if restrict else 0
        cR, sR, wR = T.ang_trig[3 * (ga0 + R):3 * (ga0 + R) + 3]
        fx, fy = dy * 0.25 * dth, dx * 0.25 * dth
        ox1 = fx * wR * cR if quad in (0, 3) else 0.0
        ox0 = -fx * wR * cR if quad in (1, 2) else 0.0
        oy1 = fy * wR * sR if quad in (0, 1) else 0.0
        oy0 = -fy * wR * sR if quad in (2, 3) else 0.0
        sx_, sy_ = H.src[ga0 + R] if H.alike else (-1, -1)
        yo = cdof + (w & 0xfffff) + (w >> 25)
        xr = X[R].reshape(N, NY)
        for q in range(NY):
            qf = (2 if q == NY - 1 else 0) | (8 if q == 0 else 0)
            yin = sy_ >= 0 and q == (0 if quad < 2 else NY - 1)
            xin = 0.0
            if sx_ >= 0 and not (q == 0 and mk & 1) and not (q == NY - 1 and mk & 2):
                assert sx_ + q * nt < T.ndof
                xin = w1[NY][q] * -(ox1 + ox0) * x[sx_ + q * nt]
            oy = oy1 if q == NY - 1 else (oy0 if q == 0 else 0.0)
            for p in range(N):
                s = p * NY + q
                on = qf | (4 if p == 0 else 0) | (1 if p == N - 1 else 0)
                o = yo + s * nt
                assert cdof <= o < cdof + nsp * na
                fs = 0.0
                if on & lf:
                    assert stored[o] or on & bd
                    fs = y[o]
                if yin:
                    dead = (p == 0 and mk & 4) or (p == N - 1 and mk & 8)
                    assert sy_ + p * NY * nt < T.ndof
                    fs = 0.0 if dead else -(oy1 + oy0) * x[sy_ + p * NY * nt]
                wq, wp, xv = w1[NY][q], w1[N][p], xr[p, q]
                val = dx * dy * 0.125 * dth * wR * wp * wq * kappa[sp0 + s] * xv
                val -= fx * wR * cR * wq * (wd[N][p] @ xr[:, q]) + fy * wR * sR * wp * (wd[NY][q] @ xr[p])
                val += (ox1 * wq * xv if p == N - 1 else 0.0) + (ox0 * wq * xv if p == 0 else 0.0)
                val += xin if p == (0 if quad in (0, 3) else N - 1) else 0.0
                val += oy * wp * xv + (wp * fs if yin else fs)
                val -= dx * dy * wp * wq * sigma[sp0 + s] * scat[R, s]
                if accumulate:
                    if not on & bd:
                        y[o] = val if on & lf else y[o] + val
                else:
                    y[o] = 0.0 if on & bd else val


def edge_mesh(case):
    if case.startswith("random_hp"):
        return problems.random_hp_mesh(int(case[-1]), base_spt=1, base_ang=2, extra_spt=1,
                                       extra_ang=1, p_col=0.5, p_cell=0.5)
    if case == "periodic_x":
        mesh = problems.uniform_mesh([1.0, 1.0], [4, 4, 3], 2, 2, pbcs=(True, False))
        mesh.ref_col(sorted(mesh.cols)[0], kind="spt", form="h")
        return mesh
    if case == "unlike":
        mesh = problems.uniform_mesh([1.0, 1.3], [4, 3, 3], 2, 2)
        keys = sorted(mesh.cols)
        mesh.ref_col(keys[0], kind="spt", form="p")
        mesh.ref_cell(keys[-1], sorted(mesh.cols[keys[-1]].cells)[0], "p")
        return mesh
    if case == "half_circles":        # a cell spans several quadrants: four inflow faces
        mesh = problems.uniform_mesh([1.0, 1.0], [3, 4, 4], 1, 1)
        mesh.ref_col(sorted(mesh.cols)[0], "spt", "p")
        return mesh
    return problems.uniform_mesh([1.0, 1.0], [4, 3, 3], 2, 2)


@pytest.mark.parametrize("restrict", [True, False], ids=["interior", "whole"])
@pytest.mark.parametrize("case", ["random_hp_1", "random_hp_2", "periodic_x", "unlike", "alike",
                                  "half_circles"])
def test_hp_kernels_model_matches_oracle(case, restrict):
    from rtx.plan import MeshTables
    mesh = edge_mesh(case)
    wl = problems.two_scatterers()
    T = MeshTables(mesh)
    H = Tables(T)
    assert H.alike == (case in ("alike", "unlike", "periodic_x"))
    assert any(H.direct) == H.alike and all(H.direct) == (case == "alike")
    G, G_off = T.G_pool(wl.Phi)
    kappa, sigma = T.eval_spatial(wl.kappa), T.eval_spatial(wl.sigma)
    rng = np.random.default_rng(3)
    x, y0 = rng.uniform(-1, 1, T.ndof), rng.uniform(-1, 1, T.ndof)
    V = asm.assemble(mesh, wl.kappa, wl.sigma, wl.Phi, drop=False)
    A = (V["BC"] - V["IC"] + V["M"] + V["S"]).tocsr()
    mask = asm.intr_mask(mesh) if restrict else np.ones(T.ndof)
    ref = mask * (A @ (mask * x))
    for M, accumulate in ((F64, False), (F32, True)):
        y = y0.copy() if accumulate else np.full(T.ndof, np.nan)
        stored = flux_model(H, M, x, y, restrict, accumulate)
        for c in range(T.ncol):
            column_model(H, c, kappa, sigma, G, G_off, x, y, stored, restrict, accumulate)
        want = y0 + ref if accumulate else ref
        assert not np.isnan(y).any()                 # every output written
        assert np.linalg.norm(y - want) / np.linalg.norm(want) < 1e-12


@pytest.mark.parametrize("N", range(3, 11))
def test_accumulators_hold_whole_lines(N):
    """Row i of node tile t is the node that lane group and register of that
    accumulator row stand for: register e of lane group g holds node e % N of
    line g + 4 (l0 + e / N), which is where a lane's lines read it.  The items
    of the wavefronts cover every line of every 16 angles once."""
    NL = (N + 3) // 4
    for M, LI, NY in [(F64, 1, N), (F32, NL, N)] + [(F64, 1, ny) for ny in range(3, 11)]:
        MT = (N * LI + 3) // 4
        NI = (NY + 3) // 4 if LI == 1 else 1
        lines = []
        for l0 in range(NI):
            held = {}
            for t in range(MT):
                for i in range(16):
                    e, q = 4 * t + M.reg(i), M.group(i) + 4 * (l0 + (4 * t + M.reg(i)) // N)
                    node = (e % N) * NY + (q if q < NY else NY - 1)
                    assert 0 <= node < N * NY
                    held[t, i] = node
            for lg in range(4):
                for l in range(LI):
                    q = lg + 4 * (l0 + l)
                    if q >= NY:
                        continue
                    lines.append(q)
                    for p in range(N):
                        t, v = divmod(l * N + p, 4)
                        assert t < MT and held[t, M.row(lg, v)] == p * NY + q
        assert sorted(lines) == list(range(NY))
        for na in (1, 16, 17, 88, 160):
            total = (na + 15) // 16 * NI
            taken = [it for w in range(WAVES) for it in range(w, total, WAVES)]
            assert sorted(taken) == list(range(total))


def test_index_division():
    """hp_div: floor(v / n) by a float product, exact for v < 2^16, n <= 100
    (nodes of a column, angles of a cell, nodes of a line)."""
    v = np.arange(1 << 16)
    for n in range(1, 101):
        q = ((v.astype(np.float32) + np.float32(0.5)) * (np.float32(1.0) / np.float32(n)))
        assert np.array_equal(q.astype(np.int64), v // n), n


def test_bf16_stride_spreads_operand_reads_over_banks():
    """The BF16 matrix-core operand reads of a half-wave (16 rows of the
    node-major copy, 2 quads of k) fall on 64 distinct 4-byte banks."""
    for na in range(1, 300):
        XSB = hp_stride(na, 16, 8, 16)
        assert XSB >= (na + 15) // 16 * 16
        words = {(l16 * XSB // 2 + 2 * lg + w) % 64 for l16 in range(16) for lg in range(2)
                 for w in range(2)}
        assert len(words) == 64, na


def wide_bytes(T, c):
    """The FP64 bytes that hp_wide counts: own values or traces, the larger of
    the contracted traces and the inflow-face sums, distinct E^s blocks."""
    k0, k1 = int(T.col_cell_start[c]), int(T.col_cell_start[c + 1])
    nx, ny, na = int(T.col_nx[c]), int(T.col_ny[c]), int(T.col_nang[c])
    sums = inner = nes = 0
    seen = set()
    for k in range(k0, k1):
        faces = set()
        for l in links_of(T, k):
            F, c1 = int(T.link_face[l]), int(T.cell_col[int(T.link_src[l])])
            n1 = int(T.col_nx[c1] if F & 1 else T.col_ny[c1])
            faces.add(F)
            inner += n1 * int(T.cell_nth[k])
            if int(T.link_Es_off[l]) not in seen:
                seen.add(int(T.link_Es_off[l]))
                nes += nx * n1
        sums += len(faces) * nx * int(T.cell_nth[k])
    own = max((na + 3) // 4 * 4 * (nx * ny | 1), int(T.col_ntrace[c]))
    nbytes = (8 * own + 15) // 16 * 16 + 8 * (max(sums, inner) + nes) + 28 * na
    return (nbytes + 15) // 16 * 16, sums


def test_batched_hp_meshes_run_in_their_own_precision():
    """Every column of the two batched uneven-order meshes fits the column
    kernel in all precisions, and none is so large or so linked that reduced
    precision keeps FP64 arithmetic; a 10 x 10 x 10 mesh of 16 angular cells
    has columns that do."""
    from rtx.plan import MeshTables
    for p_col in (0.3, 0.4):
        T = MeshTables(problems.random_hp_mesh(0, p_col=p_col))
        for c in range(T.ncol):
            k0, k1 = T.col_cell_start[c], T.col_cell_start[c + 1]
            nsp, na = int(T.col_nx[c] * T.col_ny[c]), int(T.col_nang[c])
            assert k1 - k0 <= MAX_CELLS and T.col_nx[c] == T.col_ny[c] >= 3
            for prec in ("f64", "f32", "mixed"):
                assert hp_layout(nsp, na, prec, True)[3] <= CAP
            nbytes, sums = wide_bytes(T, c)
            assert nbytes <= 152712 and sums <= 4096
            assert T.link_start[k1] - T.link_start[k0] <= 192
    T = MeshTables(problems.uniform_mesh([1.0, 1.0], [10, 10, 10], 4, 2))
    wide = [wide_bytes(T, c)[0] > 152712 for c in range(T.ncol)]
    assert sum(wide) == 12 and hp_layout(100, 160, "f64", True)[3] <= CAP
