"""The work that users of libmtsp2 have it do, as cases to time and compare.

A user's program holds one context per GPU with the model assembled, and asks
it for
  * the fields of a batch of (frequency, polarization) systems ("solve": the
    mixed-precision batched solver on device buffers, A for the forward
    fields, A^T for the adjoint ones),
  * one system at a time from host arrays, as the reference's Fortran host
    does ("dropin": mt_bicg or mt_qmr),
  * the start of a new model of an inversion ("fields": mt_update_cond, the
    2-D boundary fields and the right-hand sides of every system),
  * what follows the forward solves ("sens": responses, the adjoint sources
    of the residuals and the gradient of the misfit).
Grids, models, frequencies and sites are those of mtsp2.problem (the
repository's workloads), and ragged ones whose cells fill no whole 8x8x8 tile.

The solves run to a relative residual of 1e-13 (QMR to 1e-12):
at the default 1e-7 the fields still differ by 1e-4 from one summation order to
the next, which says nothing about either; the iterations are the same ones.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "modem-gpu_amd"))

import mtsp2                       # noqa: E402
from mtsp2 import problem as P     # noqa: E402

PI, MU0, SIGMA_AIR = P.PI, P.MU0, 1e-10
DEV = "cuda"


def listed():
    def solve(name, nx, ny, nz, nair, nf, adjoint=False):
        return {"name": name, "kind": "solve", "nx": nx, "ny": ny, "nz": nz, "nair": nair,
                "nf": nf, "adjoint": adjoint}

    def dropin(name, nx, ny, nz, nair, solver):
        return {"name": name, "kind": "dropin", "nx": nx, "ny": ny, "nz": nz, "nair": nair,
                "nf": 1, "solver": solver}

    def other(name, kind, nx, ny, nz, nair, nf):
        return {"name": name, "kind": kind, "nx": nx, "ny": ny, "nz": nz, "nair": nair, "nf": nf}

    return [
        # every forward system of the headline workload in one batch
        solve("forward_100x100x60_8f", 100, 100, 60, 10, 8),
        # the adjoint systems of a shard of the 80x80x50 gradient workload
        solve("adjoint_80x80x50_3f", 80, 80, 50, 10, 3, adjoint=True),
        # a regional survey's grid, no side a multiple of the tile
        solve("forward_53x61x37_2f", 53, 61, 37, 9, 2),
        # one frequency of the smallest workload: few workgroups per launch
        solve("forward_40x40x30_1f", 40, 40, 30, 10, 1),
        # one frequency per rank, adjoint, on a small odd grid
        solve("adjoint_27x23x19_1f", 27, 23, 19, 7, 1, adjoint=True),
        # the reference host's cuBiCG call at the size of its CylinderModel grid
        dropin("bicg_48x68x44", 48, 68, 44, 10, "bicg"),
        # the same call on a test-sized grid: launches and host work
        dropin("bicg_22x24x14", 22, 24, 14, 6, "bicg"),
        # the reference's default solver
        dropin("qmr_30x26x20", 30, 26, 20, 6, "qmr"),
        # a new model's boundary fields and right-hand sides, headline workload
        other("fields_100x100x60_8f", "fields", 100, 100, 60, 10, 8),
        # the same for one frequency on a ragged grid
        other("fields_45x33x27_1f", "fields", 45, 33, 27, 8, 1),
        # responses, adjoint sources and gradient of the 80x80x50 workload
        other("sens_80x80x50_12f", "sens", 80, 80, 50, 10, 12),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["solve", "solve", "solve", "dropin", "fields", "sens"])
    c = {"kind": kind, "nair": rng.randint(6, 10)}
    if kind == "dropin":
        c.update(nx=size(20, 56), ny=size(20, 56), nz=size(12, 40), nf=1,
                 solver=rng.choice(["bicg", "bicg", "qmr"]))
        if c["solver"] == "qmr":
            c.update(nx=min(c["nx"], 28), ny=min(c["ny"], 28), nz=min(c["nz"], 18))
        return c
    c.update(nx=size(22, 96), ny=size(22, 96), nz=size(14, 58), nf=size(1, 8))
    if kind == "solve":
        c["adjoint"] = rng.random() < 0.5
    return c


# ------------------------------------------------------------------ inputs
def _grid(case):
    pad = 8 if min(case["nx"], case["ny"]) >= 28 else 6
    return P.make_grid(case["nx"], case["ny"], case["nz"], nair=case["nair"], npad=pad)


def _model(case, grid, seed):
    return P.boxes_model(grid, nbox=max(10, case["nx"] * case["ny"] // 50), seed=seed)


def _freqs(case):
    """The workloads' band, 1e-3 .. 1e2 Hz; a single frequency is 1 Hz."""
    nf = case["nf"]
    return 10.0 ** (-3 + 5 * np.arange(nf) / (nf - 1)) if nf > 1 else np.array([1.0])


def _systems(case):
    om = np.repeat(2 * PI * _freqs(case), 2)
    return om, np.tile(np.array([1, 2], np.int32), case["nf"])


def _sites(grid):
    return P.core_sites(grid, 12, npad=6)


def _adjoint_sources(case, grid, nsys, seed):
    """Right-hand sides of adjoint systems: complex weights on the edges round
    the sites, zero elsewhere (interior-edge order)."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"] + case["nair"]
    ei = P.interior_edges(nx, ny, nz)
    pos = np.full(sum(P.edge_counts(nx, ny, nz)), -1, np.int64)
    pos[ei] = np.arange(len(ei))
    nXe, nYe, _ = P.edge_counts(nx, ny, nz)
    s = _sites(grid)
    i = np.searchsorted(np.cumsum(grid["dx"]), s[:, 0])
    j = np.searchsorted(np.cumsum(grid["dy"]), s[:, 1])
    k = case["nair"]
    at = np.concatenate([i + nx * (j + (ny + 1) * k), i + nx * (j + 1 + (ny + 1) * k),
                         nXe + i + (nx + 1) * (j + ny * k), nXe + i + 1 + (nx + 1) * (j + ny * k),
                         nXe + nYe + i + (nx + 1) * (j + (ny + 1) * k)])
    at = np.unique(pos[at])
    at = at[at >= 0]
    rng = np.random.default_rng(seed + 1000)
    b = np.zeros((nsys, len(ei)), np.complex128)
    b[:, at] = rng.standard_normal((nsys, len(at))) + 1j * rng.standard_normal((nsys, len(at)))
    return b


def _context(case, grid, lc):
    ctx = mtsp2.Context(0)
    ctx.assemble(grid["dx"], grid["dy"], grid["dz"], grid["nzAir"], lc)
    return ctx


def _buf(nsys, n):
    return torch.zeros((nsys, n), dtype=torch.complex128, device=DEV)


def prepare(case, seed):
    grid = _grid(case)
    lc = _model(case, grid, seed)
    kind = case["kind"]
    st = {"kind": kind, "case": case, "grid": grid}
    if kind == "dropin":
        ctx = _context(case, grid, lc)
        om, B, X0 = P.forward_systems(ctx, grid, _freqs(case), pols=(seed % 2,))
        st.update(ctx=ctx, om=float(om[0]), b=B[0], x0=X0[0])
        return st
    om, modes = _systems(case)
    ns = len(om)
    st.update(om=om, modes=modes)
    # the context of a "fields" case holds another model: the call brings the new one
    ctx = _context(case, grid, _model(case, grid, seed + 1) if kind == "fields" else lc)
    st["ctx"] = ctx
    n, ne = ctx.n_int, ctx.n_edge
    if kind == "solve":
        st["x"] = _buf(ns, n)
        if case["adjoint"]:
            st["b"] = torch.from_numpy(_adjoint_sources(case, grid, ns, seed)).to(DEV)
            st["x0"] = _buf(ns, n)
        else:
            e, st["b"], st["x0"] = _buf(ns, ne), _buf(ns, n), _buf(ns, n)
            torch.cuda.synchronize()
            ctx.bc_x0_dev(om, modes, e.data_ptr())
            ctx.rhs_fwd_dev(ns, e.data_ptr(), st["b"].data_ptr(), st["x0"].data_ptr())
    elif kind == "fields":
        st.update(lc=lc, e=_buf(ns, ne), b=_buf(ns, n), x0=_buf(ns, n))
    else:
        # forward fields as the solver returns them (here their 2-D start),
        # adjoint fields of a like decay with depth
        st.update(e=_buf(ns, ne), comb=_buf(ns, ne), s=_buf(ns, n),
                  dm=torch.zeros(case["nx"] * case["ny"] * case["nz"], dtype=torch.float64, device=DEV))
        torch.cuda.synchronize()
        ctx.bc_x0_dev(om, modes, st["e"].data_ptr())
        st["lam"] = torch.from_numpy(_adjoint_fields(case, grid, ns, seed)).to(DEV)
        ctx.receivers_set(grid["dx"], grid["dy"], grid["dz"], grid["nzAir"], _sites(grid))
        rng = np.random.default_rng(seed + 2000)
        st["d"] = rng.standard_normal((case["nf"], 144, 8)) * 1e-3
    torch.cuda.synchronize()
    return st


def _adjoint_fields(case, grid, nsys, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"] + case["nair"]
    rng = np.random.default_rng(seed + 3000)
    z = P.node_depths(grid)
    fall = np.exp(-np.abs(z) / 2e4)
    out = np.empty((nsys, len(P.interior_edges(nx, ny, nz))), np.complex128)
    parts = ((nz - 1, ny - 1, nx), (nz - 1, ny, nx - 1), (nz, ny - 1, nx - 1))
    for s in range(nsys):
        row, a = out[s], 0
        for shp in parts:
            m = shp[0] * shp[1] * shp[2]
            w = (fall[1:-1] if shp[0] == nz - 1 else fall[:-1])[:, None, None]
            v = rng.standard_normal(shp, dtype=np.float32) + 1j * rng.standard_normal(shp, dtype=np.float32)
            row[a:a + m] = (w * v).ravel()
            a += m
    return out


# ------------------------------------------------------------------ one pass
def run(st):
    ctx, kind, case = st["ctx"], st["kind"], st["case"]
    if kind == "dropin":
        f = ctx.qmr if case["solver"] == "qmr" else ctx.bicg
        r = f(st["om"], st["b"], st["x0"], maxit=3000, tol=1e-12 if case["solver"] == "qmr" else 1e-13)
        return {"x": r[0], "failed": r[3]}
    ns = len(st["om"])
    if kind == "solve":
        ctx.dev_copy(st["x"].data_ptr(), st["x0"].data_ptr(), st["x"].numel() * 16)
        r = ctx.solve_batch_dev(st["om"], st["b"].data_ptr(), st["x"].data_ptr(), tol=1e-13, maxit=6000,
                                precision=mtsp2.PREC_MIXED, precond=mtsp2.PC_DILU_RB,
                                op_transpose=int(case["adjoint"]))
        return {"x": st["x"], "status": [s["status"] for s in r]}
    if kind == "fields":
        ctx.update_cond(st["lc"])
        ctx.bc_x0_dev(st["om"], st["modes"], st["e"].data_ptr())
        ctx.rhs_fwd_dev(ns, st["e"].data_ptr(), st["b"].data_ptr(), st["x0"].data_ptr())
        return {"e": st["e"], "b": st["b"], "x0": st["x0"]}
    f_om = st["om"][::2]
    resp = ctx.data_resp(mtsp2.DT_FULL_IMPEDANCE, f_om, st["e"].data_ptr(), 8)
    ctx.lmultT(mtsp2.DT_FULL_IMPEDANCE, f_om, st["e"].data_ptr(), st["d"], st["comb"].data_ptr())
    ctx.rhs_trn_dev(st["om"], st["comb"].data_ptr(), st["s"].data_ptr(), gd_correct=False)
    ctx.gradient_dev(f_om, 2, st["e"].data_ptr(), st["lam"].data_ptr(), st["dm"].data_ptr())
    return {"resp": resp, "s": st["s"], "dm": st["dm"]}


def work(case):
    """Inputs once, outputs once; a solve cannot do without the operator (its
    15 couplings and the diagonal in FP64) and one multiplication by it."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"] + case["nair"]
    n = nx * (ny - 1) * (nz - 1) + (nx - 1) * ny * (nz - 1) + (nx - 1) * (ny - 1) * nz
    ne = sum(P.edge_counts(nx, ny, nz))
    ns, cells = 2 * case["nf"], nx * ny * case["nz"]
    kind = case["kind"]
    if kind == "dropin":
        return {"bytes": 16 * n * 8 + 3 * 16 * n, "flops": 64 * n}
    if kind == "solve":
        return {"bytes": 16 * n * 8 + 3 * 16 * n * ns, "flops": 64 * n * ns}
    if kind == "fields":
        # the banded LU of every slice: b^2 complex multiply-adds per unknown
        lu = case["nf"] * sum(sl * (nh - 1) * (nz - 1) ** 3 * 8 for sl, nh in ((nx, ny), (ny, nx)))
        return {"bytes": 8 * cells + 16 * ns * (ne + 2 * n), "flops": lu}
    return {"bytes": 16 * ns * (ne + n + n) + 8 * cells, "flops": 64 * n * ns}


# ------------------------------------------------- the same in plain torch
def _pad(a, dim):
    shp = list(a.shape)
    shp[dim] = 1
    z = a.new_zeros(shp)
    return torch.cat([z, a, z], dim)


def _dpad(a, dim):
    """Transpose of torch.diff along dim, negated."""
    return torch.diff(_pad(a, dim), dim=dim)


def _mean(w, s, dims):
    """sum(w s) / sum(w) over the cells that touch an edge or node."""
    for d in dims:
        a, b = _pad(w * s, d), _pad(w, d)
        n = a.shape[d]
        num = a.narrow(d, 0, n - 1) + a.narrow(d, 1, n - 1)
        w = b.narrow(d, 0, n - 1) + b.narrow(d, 1, n - 1)
        s = num / w
    return s


class _Operator:
    """CC + GD + i ISIGN omega mu0 sigma V on the staggered grid, from the
    definition: arrays (..., k, j, i), components x, y, z."""

    def __init__(self, grid, lc):
        t = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.float64, device=DEV)  # noqa: E731
        d = [t(grid["dx"]), t(grid["dy"]), t(grid["dz"])]
        half = [_dual(v) for v in d]
        X, Y, Z = (lambda v: v[None, None, :]), (lambda v: v[None, :, None]), (lambda v: v[:, None, None])
        self.n = nx, ny, nz = len(d[0]), len(d[1]), len(d[2])
        ax = (X, Y, Z)
        L, H = [f(v) for f, v in zip(ax, d)], [f(v) for f, v in zip(ax, half)]
        self.L = L
        self.dual = [H[1] * H[2], H[0] * H[2], H[0] * H[1]]
        self.face = [H[0] / (L[1] * L[2]), H[1] / (L[0] * L[2]), H[2] / (L[0] * L[1])]
        self.vnode = H[0] * H[1] * H[2]
        self.lc = t(lc).permute(2, 1, 0).contiguous()
        air = torch.full((grid["nzAir"], ny, nx), SIGMA_AIR, dtype=torch.float64, device=DEV)
        self.air, self.vol = air, (L[0] * L[1] * L[2]).expand(nz, ny, nx)
        self.shape = ((nz + 1, ny + 1, nx), (nz + 1, ny, nx + 1), (nz, ny + 1, nx + 1))
        self.inner = [(slice(1, -1), slice(1, -1), slice(None)), (slice(1, -1), slice(None), slice(1, -1)),
                      (slice(None), slice(1, -1), slice(1, -1))]
        self.set_model(self.lc)

    def set_model(self, lc):
        s = torch.cat([self.air, torch.exp(lc)], 0)
        self.sig = [_mean(self.vol, s, dims) for dims in ((0, 1), (0, 2), (1, 2))]
        sn = _mean(self.vol, s, (0, 1, 2))
        with torch.no_grad():
            wet = [(e >= float(np.float32(1.1)) * SIGMA_AIR).double() for e in self.sig]
            near = torch.zeros_like(sn)
            for c, w in enumerate(wet):
                p = _pad(w, 2 - c)
                m = p.shape[2 - c]
                near += p.narrow(2 - c, 0, m - 1) + p.narrow(2 - c, 1, m - 1)
            inside = torch.zeros_like(sn)
            inside[1:-1, 1:-1, 1:-1] = 1.0
            earth = (near > 0).double() * inside
        self.m_air = (inside - earth) / self.vnode
        self.m_earth = earth / (sn * self.vnode)

    def curlcurl(self, e):
        w = [a * b for a, b in zip(self.L, e)]
        D = lambda a, c: torch.diff(a, dim=c - 3)          # noqa: E731  c: 0 k, 1 j, 2 i
        f = [D(w[2], 1) - D(w[1], 0), D(w[0], 0) - D(w[2], 2), D(w[1], 2) - D(w[0], 1)]
        f = [a * b for a, b in zip(self.face, f)]
        T = lambda a, c: _dpad(a, a.dim() - 3 + c)         # noqa: E731
        return [self.L[0] * (T(f[2], 1) - T(f[1], 0)), self.L[1] * (T(f[0], 0) - T(f[2], 2)),
                self.L[2] * (T(f[1], 2) - T(f[0], 1))]

    def graddiv(self, e):
        out = [0, 0, 0]
        for m, wt in ((self.m_air, None), (self.m_earth, self.sig)):
            u = [a * b if wt is None else a * b * s for a, b, s in zip(self.dual, e, self.sig)]
            div = -m * sum(_dpad(u[c], u[c].dim() - 1 - c) for c in range(3))
            out = [o + a * torch.diff(div, dim=-1 - c) for c, (o, a) in enumerate(zip(out, self.dual))]
        return out

    def apply(self, omega, e):
        """Rows of the interior edges, columns of the interior edges."""
        e = self.mask(e)
        cc, gd = self.curlcurl(e), self.graddiv(e)
        s = 1j * P.ISIGN * omega * MU0
        return self.mask([a + b + s * sg * (ln * du) * x for a, b, sg, ln, du, x in
                          zip(cc, gd, self.sig, self.L, self.dual, e)])

    def mask(self, e):
        out = []
        for a, s in zip(e, self.inner):
            z = torch.zeros_like(a)
            z[(Ellipsis,) + s] = a[(Ellipsis,) + s]
            out.append(z)
        return out

    def split(self, v):
        """All-edge vector -> components."""
        m = [math.prod(s) for s in self.shape]
        return [p.reshape(v.shape[:-1] + s) for p, s in zip(torch.split(v, m, -1), self.shape)]

    def interior(self, e):
        return torch.cat([a[(Ellipsis,) + s].flatten(-3) for a, s in zip(e, self.inner)], -1)

    def spread(self, v):
        """Interior-edge vector -> components, zero on the boundary."""
        z = [torch.zeros(v.shape[:-1] + s, dtype=v.dtype, device=v.device) for s in self.shape]
        a = 0
        for c, s in zip(z, self.inner):
            t = c[(Ellipsis,) + s]
            m = math.prod(t.shape[-3:])
            c[(Ellipsis,) + s] = v[..., a:a + m].reshape(t.shape)
            a += m
        return z

    def rhs(self, e):
        """-CCib e_b."""
        b = [a - m for a, m in zip(e, self.mask(e))]
        return -self.interior(self.curlcurl(b))

    def solve(self, omega, b, adjoint):
        """A x = b (A^T x = b) by block elimination over the k planes."""
        nx, ny, nz = self.n
        dims = [s[1:] for s in self.shape]
        off = np.cumsum([0] + [d[0] * d[1] for d in dims])
        m = int(off[-1])
        blk = torch.zeros((nz, 3, m, m), dtype=torch.complex128, device=DEV)
        K, J, I = (torch.arange(v, device=DEV) for v in (nz, ny + 1, nx + 1))
        for c in range(3):
            for col in range(27):
                ck, cj, ci = col // 9, col // 3 % 3, col % 3
                v = [torch.zeros(s, dtype=torch.complex128, device=DEV) for s in self.shape]
                v[c][ck::3, cj::3, ci::3] = 1.0
                y = self.apply(omega, v)
                for r in range(3):
                    rj, ri = dims[r]
                    near = lambda q, g: q + (g - q + 1) % 3 - 1    # noqa: E731
                    k2, j2, i2 = near(K, ck), near(J[:rj], cj), near(I[:ri], ci)
                    cols = int(off[c]) + j2[:, None] * dims[c][1] + i2[None, :]
                    ok = ((j2 >= 0) & (j2 < dims[c][0]))[:, None] & ((i2 >= 0) & (i2 < dims[c][1]))[None, :]
                    rows = int(off[r]) + (J[:rj, None] * ri + I[None, :ri])
                    for k in range(nz):
                        if 0 <= int(k2[k]) < nz:
                            blk[k, int(k2[k]) - k + 1, rows[ok], cols[ok]] = y[r][k][ok]
        eye = [(torch.ones(s, device=DEV), s) for s in self.shape]
        bound = [o - a for (o, _), a in zip(eye, self.mask([o for o, _ in eye]))]
        dg = torch.arange(m, device=DEV)
        for k in range(nz):
            blk[k, 1, dg, dg] += torch.cat([q[k].flatten() for q in bound])
        if adjoint:
            t = blk.transpose(2, 3).clone()
            blk[1:, 0], blk[:-1, 2], blk[:, 1] = t[:-1, 2], t[1:, 0], t[:, 1]
            del t
        f = self.spread(b)
        rhs = [torch.cat([q[:, k].flatten(1) for q in f], 1).T for k in range(nz)]
        up = []
        for k in range(nz):
            S = blk[k, 1]
            if k:
                S = S - blk[k, 0] @ up[-1]
                rhs[k] = rhs[k] - blk[k, 0] @ rhs[k - 1]
            w = torch.linalg.solve(S, torch.cat([blk[k, 2], rhs[k]], 1))
            up.append(w[:, :m])
            rhs[k] = w[:, m:]
        for k in range(nz - 2, -1, -1):
            rhs[k] = rhs[k] - up[k] @ rhs[k + 1]
        x = [torch.zeros(b.shape[:1] + s, dtype=b.dtype, device=DEV) for s in self.shape]
        for k in range(nz):
            for c in range(3):
                x[c][:, k] = rhs[k][int(off[c]):int(off[c + 1])].T.reshape((-1,) + tuple(dims[c]))
        return self.interior(x)


def _dual(d):
    return torch.cat([d[:1], d[:-1] + d[1:], d[-1:]]) / 2.0


def _te1d(omega, nza, dz, s):
    """1-D TE fields of columns s (columns, earth layers), 1 at the top, a
    skin depth below the last layer to 0."""
    ncol, nz = s.shape[0], len(dz)
    sg = torch.cat([s.new_full((ncol, nza), SIGMA_AIR), s, s[:, -1:]], 1)
    dd = torch.cat([dz[None, :].expand(ncol, nz), torch.sqrt(2.0 / (sg[:, -1:] * omega * MU0))], 1)
    up = 2.0 / dd
    a = -(up[:, :-1] + up[:, 1:]) + 1j * omega * MU0 * (sg[:, 1:] * dd[:, 1:] + sg[:, :-1] * dd[:, :-1])
    cp, r = [], []
    for i in range(nz):
        den = a[:, i] - (up[:, i] * cp[-1] if i else 0.0)
        cp.append(up[:, i + 1] / den)
        r.append(((-up[:, 0] + 0j) if i == 0 else -up[:, i] * r[-1]) / den)
    for i in range(nz - 2, -1, -1):
        r[i] = r[i] - cp[i] * r[i + 1]
    return torch.stack([torch.ones_like(r[0])] + r, 1)


def _te2d(omega, nza, dy, dz, cond):
    """2-D TE fields (slices, nh+1, nz+1) of slices cond (slices, nh, nz)."""
    ns, nh, nz = cond.shape
    c = cond.clone()
    c[:, :, :nza] = SIGMA_AIR
    w = dy[:, None] * dz[None, :]
    cw = c * w
    q = lambda a: a[..., 1:, 1:] + a[..., 1:, :-1] + a[..., :-1, 1:] + a[..., :-1, :-1]   # noqa: E731
    s2 = q(cw) / q(w)
    cy, cz = dy[:-1] + dy[1:], dz[:-1] + dz[1:]
    ar, al = 2.0 * cz[None, :] / dy[1:, None], 2.0 * cz[None, :] / dy[:-1, None]
    dn, up = 2.0 * cy[:, None] / dz[None, 1:], 2.0 * cy[:, None] / dz[None, :-1]
    diag = -(ar + al + dn + up) + 1j * omega * MU0 * cy[:, None] * cz[None, :] * s2
    e = torch.zeros((ns, nh + 1, nz + 1), dtype=torch.complex128, device=c.device)
    e[:, :, 0] = 1.0
    e[:, 0] = _te1d(omega, nza, dz, c[:, 0, nza:])
    e[:, -1] = _te1d(omega, nza, dz, c[:, -1, nza:])
    mid = (c[:, :-1] * dy[:-1, None] + c[:, 1:] * dy[1:, None]) / cy[:, None]
    e[:, 1:-1, -1] = _te1d(omega, nza, dz, mid[:, :, nza:].reshape(-1, nz - nza))[:, -1].reshape(ns, nh - 1)
    r = torch.zeros_like(diag)
    r[:, 0] -= al[0] * e[:, 0, 1:-1]
    r[:, -1] -= ar[-1] * e[:, -1, 1:-1]
    r[:, :, 0] -= up[:, 0] * e[:, 1:-1, 0]
    r[:, :, -1] -= dn[:, -1] * e[:, 1:-1, -1]
    ups, x = [], []
    for i in range(nh - 1):
        S = torch.diag_embed(diag[:, i]) + torch.diag_embed((dn[i, :-1] + 0j).expand(ns, -1), 1) + \
            torch.diag_embed((up[i, 1:] + 0j).expand(ns, -1), -1)
        f = r[:, i]
        if i:
            S = S - al[i][:, None] * ups[-1]
            f = f - al[i] * x[-1]
        sol = torch.linalg.solve(S, torch.cat([torch.diag(ar[i] + 0j).expand(ns, -1, -1), f[:, :, None]], 2))
        ups.append(sol[:, :, :-1])
        x.append(sol[:, :, -1])
    for i in range(nh - 3, -1, -1):
        x[i] = x[i] - (ups[i] @ x[i + 1][:, :, None])[:, :, 0]
    e[:, 1:-1, 1:-1] = torch.stack(x, 1)
    return e


def _fields(case, grid, lc):
    """All-edge start fields of every system of a case."""
    om, modes = _systems(case)
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=DEV)  # noqa: E731
    cond = torch.exp(t(lc))
    cond = torch.cat([cond.new_full((case["nx"], case["ny"], case["nair"]), SIGMA_AIR), cond], 2)
    dx, dy, dz = t(grid["dx"]), t(grid["dy"]), t(grid["dz"])
    nx, ny, nz = case["nx"], case["ny"], len(dz)
    nXe, nYe, nZe = P.edge_counts(nx, ny, nz)
    out = torch.zeros((len(om), nXe + nYe + nZe), dtype=torch.complex128, device=DEV)
    for s, (w, m) in enumerate(zip(om, modes)):
        if m == 2:
            e = _te2d(float(w), case["nair"], dy, dz, cond).permute(2, 1, 0).clone()
            e[-1] = 0
            out[s, :nXe] = e.flatten()
        else:
            e = _te2d(float(w), case["nair"], dx, dz, cond.transpose(0, 1)).permute(2, 0, 1).clone()
            e[-1] = 0
            out[s, nXe:nXe + nYe] = e.flatten()
    return out


def exact(case, seed):
    kind, size = case["kind"], case["nx"] * case["ny"]
    grid = _grid(case)
    lc = _model(case, grid, seed)
    nz = case["nz"] + case["nair"]
    if kind in ("solve", "dropin"):
        if size * nz > 22000 or case["nf"] > 1:   # elimination of larger planes takes minutes
            return None
        op = _Operator(grid, lc)
        om = 2 * PI * float(_freqs(case)[0])
        if kind == "dropin":
            e = torch.from_numpy(P.plane_wave(grid, om, seed % 2)).to(DEV)[None]
            return {"x": op.solve(om, op.rhs(op.split(e)), False)[0], "failed": None}
        if case["adjoint"]:
            b = torch.from_numpy(_adjoint_sources(case, grid, 2, seed)).to(DEV)
        else:
            b = op.rhs(op.split(_fields(case, grid, lc)))
        return {"x": op.solve(om, b, case["adjoint"]), "status": None}
    if kind == "fields":
        if size * nz * case["nf"] > 80000:               # as many slice eliminations
            return None
        e = _fields(case, grid, lc)
        op = _Operator(grid, lc)
        c = op.split(e)
        return {"e": e, "b": op.rhs(c), "x0": op.interior(c)}
    # gradient of Re(sum lam^T A(m) e) in the cells' log conductivity; the
    # fields e are the case's inputs (their own elimination takes minutes when
    # there are many, so then there is nothing to give)
    if size * nz * case["nf"] > 80000:
        return None
    op = _Operator(grid, lc)
    e = _fields(case, grid, lc)
    lam = torch.from_numpy(_adjoint_fields(case, grid, e.shape[0], seed)).to(DEV)
    m = op.lc.clone().requires_grad_(True)
    om, _ = _systems(case)
    dm = torch.zeros_like(op.lc)
    for s in range(e.shape[0]):
        op.set_model(m)
        y = op.interior(op.apply(float(om[s]), op.split(e[s])))
        dm += torch.autograd.grad((lam[s] * y).sum().real, m)[0]
    return {"resp": None, "s": None, "dm": dm.flatten()}
