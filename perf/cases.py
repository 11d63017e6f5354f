"""Performance cases of the BES solver core: what is timed, and on which sizes.

Every case is a piece of a flow computation as a program of this framework
runs it through ``bes_amd.core.Context``: hand the starting state over, advance
it (or assemble and solve its linear system, or train the learned
preconditioner on that system) and read the result back.  Meshes, schemes,
Courant numbers, Krylov settings and condition ranges are those of ``bench.py``
and the tests.

``exact`` evaluates the same second-order residual, local time step and
multistage scheme with plain torch operations in float64, from the mesh's
nodes and cells alone.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from bes_amd import core, meshgen as mg

GAMMA, R_GAS, HARTEN, VENKAT_K = 1.4, 287.0, 0.05, 5.0
RK4 = (0.0833, 0.2069, 0.4265, 1.0)
RK3 = (0.1481, 0.4, 1.0)   # Blazek's 3-stage coefficients for second-order upwind schemes
CFL_EXPLICIT = 0.8

_DEFAULT = dict(work="explicit", mesh="bump", ni=0, nj=0, nk=0, batch=1, steps=1, rk=4, graph=False, precision=64,
                precond="ilu0", rtol=5e-2, cfl=1.0, cfl_max=0.0, reorth=0.0, maxiter=300)


def _case(name, **kw):
    return {"name": name, **_DEFAULT, **kw}


def listed():
    return [
        # Explicit RK4 on a coarse 2D channel, each pseudo-time step one HIP
        # graph: start-up and debugging runs, the coarse grid of a mesh study.
        # All launch latency.
        _case("explicit-bump-3k", ni=60, nj=25, steps=200, graph=True),
        # The reference's own kind of run: a 40,000-triangle channel, RK4.
        _case("explicit-bump-40k", ni=200, nj=100, steps=200, graph=True),
        # A production-size explicit 3D run, one launch per pass (the default),
        # bound by memory and FP64 arithmetic.
        _case("explicit-box-750k", mesh="box", ni=50, nj=50, nk=50, steps=50),
        # A polar: 64 Mach numbers and angles of attack advance together on one
        # wing mesh (RK3), condition fastest in memory.
        _case("explicit-wing-31k-b64", mesh="wing", ni=24, nj=12, nk=18, batch=64, steps=60, rk=3, graph=True),
        # One residual evaluation of a given state: a caller with its own outer
        # iteration, or a check of a solution read from a file.
        _case("residual-wing-249k", work="residual", mesh="wing", ni=48, nj=24, nk=36),
        # A small evaluation of the same kind in 2D, odd sizes.
        _case("residual-bump-9k", work="residual", ni=93, nj=49),
        # Backward Euler on the 40,000-triangle channel with the library's
        # default Gram-Schmidt (DGKS) and ILU(0), FP64: whole pseudo-time steps.
        _case("implicit-bump-40k", work="run", ni=200, nj=100, steps=4, cfl=20.0, cfl_max=100.0, reorth=0.7),
        # One FP64 system of the wing at a large Courant number, solved tightly:
        # assembly, ILU(0) factorisation and several GMRES cycles.
        _case("solve-wing-83k-ilu", work="solve", mesh="wing", ni=36, nj=16, nk=24, cfl=100.0, rtol=1e-4),
        # The same on the two-million-cell wing, the size of the framework's
        # headline run, to its inexact-Newton tolerance.
        _case("solve-wing-2m-ilu", work="solve", mesh="wing", ni=96, nj=48, nk=72, cfl=200.0),
        # The mixed form with the aggregation AMG: hierarchy built on the system
        # and the FP32 solve.
        _case("solve-wing-486k-amg", work="solve", mesh="wing", ni=60, nj=30, nk=45, cfl=50.0, precision=32,
              precond="amg", rtol=1e-2),
        # Sixteen conditions of a polar advancing implicitly on one mesh, FP32
        # ILU(0), one launch per kernel for the batch.
        _case("implicit-wing-31k-b16", work="run", mesh="wing", ni=24, nj=12, nk=18, batch=16, steps=3, cfl=5.0,
              cfl_max=50.0, precision=32),
        # The learned preconditioner: Adam steps on the system just assembled
        # (forward and backward through the network), then a solve with it.
        _case("learned-wing-83k", work="train", mesh="wing", ni=36, nj=16, nk=24, cfl=50.0, precision=32,
              precond="learned", steps=2),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _sizes(rng, mesh, lo, hi):
    """Lattice numbers of a mesh with about lo..hi cells, odd ones among them."""
    n = _log_uniform(rng, lo, hi)
    if mesh == "bump":
        nj = max(8, int(round(math.sqrt(n / 4))) + rng.choice((0, 1)))
        return dict(mesh=mesh, ni=max(12, int(n / (2 * nj))), nj=nj, nk=0)
    if mesh == "box":
        a = max(5, int(round((n / 6) ** (1 / 3))))
        return dict(mesh=mesh, ni=a + rng.choice((0, 1)), nj=a, nk=max(4, int(n / (6 * a * a))))
    r = max(4, int(round((n / 144) ** (1 / 3))))
    return dict(mesh=mesh, ni=4 * r, nj=2 * r + rng.choice((0, 1)), nk=2 * max(4, int(n / (6 * 8 * r * r) / 2)))


def draw(rng):
    kind = rng.choice(("explicit2d", "explicit3d", "batch", "residual", "run", "solve", "solve", "amg", "runbatch",
                       "learned"))
    c = dict(_DEFAULT)
    if kind == "explicit2d":
        c.update(_sizes(rng, "bump", 2e3, 2e5), steps=rng.randrange(20, 100), graph=rng.random() < 0.6)
    elif kind == "explicit3d":
        c.update(_sizes(rng, rng.choice(("box", "wing")), 1e4, 7e5), steps=rng.randrange(5, 20), rk=rng.choice((3, 4)),
                 graph=rng.random() < 0.3)
    elif kind == "batch":
        B = rng.choice((2, 4, 8, 16, 32, 64))
        c.update(_sizes(rng, rng.choice(("bump", "wing")), 5e3, 1.5e6 / B), batch=B, steps=rng.randrange(5, 20),
                 rk=3, graph=rng.random() < 0.6)
    elif kind == "residual":
        c.update(_sizes(rng, rng.choice(("bump", "box", "wing")), 4e3, 2.4e5), work="residual")
    elif kind == "run":
        c.update(_sizes(rng, "bump", 4e3, 8e4), work="run", steps=rng.randrange(1, 3), cfl=rng.choice((10.0, 20.0)),
                 cfl_max=50.0, reorth=rng.choice((0.0, 0.7)), precond=rng.choice(("ilu0", "ilu0", "jacobi")),
                 precision=rng.choice((64, 64, 32)))
        if c["precond"] == "jacobi":
            c.update(cfl=5.0, cfl_max=0.0)
    elif kind == "solve":
        c.update(_sizes(rng, "wing", 1e4, 3e5), work="solve", cfl=rng.choice((20.0, 50.0, 100.0)),
                 rtol=rng.choice((5e-2, 1e-2, 1e-3)), precision=rng.choice((64, 64, 32)))
    elif kind == "amg":
        c.update(_sizes(rng, "wing", 1e4, 4e5), work="solve", cfl=rng.choice((20.0, 50.0)), precond="amg",
                 rtol=rng.choice((0.15, 1e-2)), precision=rng.choice((32, 32, 64)))
    elif kind == "runbatch":
        B = rng.choice((2, 4, 8, 16))
        c.update(_sizes(rng, "wing", 8e3, 3.5e5 / B), work="run", batch=B, steps=rng.randrange(1, 4), cfl=5.0,
                 cfl_max=20.0, precision=32)
    else:
        c.update(_sizes(rng, "wing", 1e4, 1e5), work="train", cfl=rng.choice((20.0, 50.0)), precision=32,
                 precond="learned", steps=rng.randrange(1, 3))
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

@functools.lru_cache(maxsize=4)
def _mesh(kind, ni, nj, nk):
    if kind == "bump":
        return mg.bump_channel(ni, nj)
    if kind == "box":
        return mg.box_tets(ni, nj, nk, seed=20261202, jitter=0.1, slip_faces=("zmin",))
    return mg.swept_wing(ni, nj, nk)


def _mesh_of(case):
    return _mesh(case["mesh"], case["ni"], case["nj"], case["nk"])


def _inputs(case, seed):
    """Mesh, freestream primitives [B][nv+1] and starting states [B][ncell][nv]."""
    md = _mesh_of(case)
    nd, B = md.ndim, case["batch"]
    rng = np.random.default_rng(seed)
    if B > 1:      # a polar's conditions
        mach, alpha = rng.uniform(0.3, 0.85, B), rng.uniform(-4.0, 8.0, B)
    elif nd == 3:  # a transonic cruise point
        mach, alpha = 0.84 + rng.uniform(-0.01, 0.01, 1), 3.06 + rng.uniform(-0.2, 0.2, 1)
    else:          # the subsonic channel
        mach, alpha = 0.5 + rng.uniform(-0.01, 0.01, 1), np.zeros(1)
    P = np.stack([core.freestream_primitive(core.wing_freestream(m, a) if nd == 3 else (m, 0.0), nd)
                  for m, a in zip(mach, alpha)])
    # the freestream with a smooth disturbance (a developing flow) and the cell
    # noise an unconverged solution carries
    cen = md.nodes[md.cells].mean(axis=1)
    span = cen.max(axis=0) - cen.min(axis=0)
    s = (cen - cen.min(axis=0)) / span
    U = np.empty((B, md.ncell, nd + 2))
    for b in range(B):
        base = core.conserved_from_primitive(P[b], nd)
        U[b] = base
        for v in range(nd + 2):
            k = rng.integers(1, 4, nd)
            ph = rng.uniform(0, 2 * np.pi, nd)
            wave = np.ones(md.ncell)
            for d in range(nd):
                wave *= np.sin(2 * np.pi * k[d] * s[:, d] + ph[d])
            U[b, :, v] *= 1.0 + 0.02 * wave + 0.002 * rng.uniform(-1, 1, md.ncell)
    return md, P, U


def prepare(case, seed):
    md, P, U = _inputs(case, seed)
    c = core.Context(md)
    if case["batch"] > 1:
        c.set_batch(case["batch"])
        c.set_freestream(P)
    else:
        c.set_freestream(P[0])
        U = U[0]
    st = {"case": dict(case), "ctx": c, "U": U}
    if case["work"] == "explicit":
        c.explicit_graph(case["graph"])
    elif case["work"] in ("run", "solve", "train"):
        c.implicit_setup(case["precision"], case["precond"], restart=30, maxiter=case["maxiter"], rtol=case["rtol"])
        c.implicit_set_reorth(case["reorth"])
        if case["precond"] in ("ilu0", "learned"):
            c.implicit_set_coloring("mesh")
        if case["precond"] == "amg":
            c.amg_set_params(relax="block_jacobi")
        if case["precond"] == "learned":
            c.lp_init(20261202)
            c.lp_neutral()
            st["params"] = c.lp_params()
    c.synchronize()
    return st


def run(state):
    case, c = state["case"], state["ctx"]
    c.set_state(state["U"])
    if case["work"] == "explicit":
        linf = c.explicit_run(case["steps"], CFL_EXPLICIT, alpha=RK4 if case["rk"] == 4 else RK3)
        return {"U": c.get_state(), "linf": linf}
    if case["work"] == "residual":
        R, mx = c.residual()
        return {"R": R, "max": mx}
    if case["work"] == "run":
        h = c.implicit_run(case["steps"], case["cfl"], case["cfl_max"], (0.5, 1.5), repeat_nv=False)
        return {"U": c.get_state(), "history": h}
    lb, lr = c.implicit_assemble(case["cfl"], repeat_nv=False)
    out = {"linf_b": lb, "linf_r": lr}
    if case["work"] == "train":
        c.lp_set_params(state["params"])
        out["loss"] = c.lp_train(case["steps"])
        out["params"] = c.lp_params()
    c.linear_solve(allow_unconverged=True)
    out["x"] = c.linear_solution()
    return out


def work(case):
    """Bytes every pass must move (each array of a sweep once, neighbour gathers
    from cache) and its FP64 operations, from the mesh's own counts."""
    n = {"bump": 2 * case["ni"] * case["nj"]}.get(case["mesh"], 6 * case["ni"] * case["nj"] * max(1, case["nk"]))
    nd = 2 if case["mesh"] == "bump" else 3
    nv, k, B = nd + 2, nd + 1, case["batch"]
    s = case["precision"] // 8
    geo = k * (16 * nd + 32) + 24                 # areas, vectors, weights, ids of a cell's faces
    state = 8 * nv
    stage = geo + B * (4 * state + 8 * nv * nd)   # U, U0, gradient and limiter products, U out
    flops = B * (k / 2 * 300 + nv * (nd * 6 + k * 30))
    copy = 2 * state * B                          # the state in and the result out
    if case["work"] == "explicit":
        it = case["steps"] * case["rk"]
        return {"bytes": n * (it * stage + copy), "flops": n * it * flops}
    if case["work"] == "residual":
        return {"bytes": n * (stage + copy), "flops": n * flops}
    block = nv * nv * s * B
    system = (k + 1) * block + B * 2 * state
    # per step: assembly, factorisation, and a GMRES cycle's products and
    # preconditioner applications (ten iterations, the least these solves take)
    it = 10
    steps = case["steps"] if case["work"] == "run" else 1
    solve = 3 * system + it * (2 * system + B * nv * s * (it + 6))
    extra = case["steps"] * (3 * 2 * 4 * 2 * system + 6 * 32 * 2 * (1 + k)) if case["work"] == "train" else 0
    return {"bytes": n * (steps * (stage + solve) + copy + extra),
            "flops": n * steps * (flops * 6 + (2 * it + 8) * (k + 1) * nv * nv * 2 * B)}


# ---------------------------------------------------------------------------
# 64-bit values by plain torch
# ---------------------------------------------------------------------------

_TET_FACES = ((0, 2, 1), (1, 2, 3), (0, 3, 2), (0, 1, 3))


class _Geo:
    """Faces and metrics of a mesh in the solver's conventions: boundary faces
    first, owner -> neighbour normals, a tetrahedron's volume without the factor
    1/3 and its centroid with the third vertex twice, and one reconstruction
    vector per cell (to its local face 0; to the last one for face 0)."""

    def __init__(self, md, dev):
        X, cells, bf = md.nodes, md.cells, md.bfaces
        nd, ne, nb = md.ndim, md.ncell, len(md.bfaces)
        k = nd + 1
        loc = [(0, 1), (1, 2), (2, 0)] if nd == 2 else _TET_FACES
        slots = cells[:, np.array(loc)].reshape(ne * k, nd)       # vertices of (cell, local face)
        key = np.sort(np.concatenate([bf, slots]), axis=1)
        _, inv = np.unique(key, axis=0, return_inverse=True)
        inv = inv.reshape(-1)
        binv, sinv = inv[:nb], inv[nb:]
        nf = int(inv.max()) + 1
        first = np.full(nf, ne * k, np.int64)
        np.minimum.at(first, sinv, np.arange(ne * k))
        last = np.full(nf, -1, np.int64)
        np.maximum.at(last, sinv, np.arange(ne * k))
        bt = np.full(nf, mg.INTERNAL)
        bt[binv] = md.btype
        verts = slots[first]                                      # oriented outward from the owner
        owner, nbr = first // k, np.where(last > first, last // k, -1)
        S, cen = self._metrics(X[verts], nd)
        area = np.sqrt((S ** 2).sum(-1))
        P = X[cells]
        c = P.mean(axis=1) if nd == 2 else (P[:, 0] + P[:, 1] + 2 * P[:, 2]) / 4
        sf = sinv.reshape(ne, k)
        own = owner[sf] == np.arange(ne)[:, None]
        sgn = np.where(own, 1.0, -1.0)
        Sc = S[sf] * sgn[..., None]
        if nd == 2:
            e1, e2 = P[:, 1] - P[:, 0], P[:, 2] - P[:, 0]
            vol = 0.5 * np.abs(e1[:, 0] * e2[:, 1] - e1[:, 1] * e2[:, 0])
        else:
            vol = 3.0 * np.abs(np.einsum("ij,ij->i", np.cross(P[:, 1] - P[:, 0], P[:, 2] - P[:, 0]),
                                         P[:, 3] - P[:, 0])) / 6.0
        adj = np.where(own, nbr[sf], owner[sf])
        r = cen[sf] - c[:, None, :]
        dO = np.sqrt((r ** 2).sum(-1))
        dN = np.sqrt(((cen[sf] - c[np.maximum(adj, 0)]) ** 2).sum(-1))
        rs = r[:, 0].copy()
        f0 = binv[0] if nb else -1                                # the mesh's face 0
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev)  # noqa: E731
        self.nd, self.k, self.ne = nd, k, ne
        self.n, self.area, self.bt = t(S / area[:, None]), t(area), t(bt)
        self.owner, self.nbr, self.sf, self.own, self.adj = t(owner), t(nbr), t(sf), t(own), t(adj)
        self.sgn, self.Sc, self.vol, self.w, self.r = t(sgn), t(Sc), t(vol), t(dN / (dO + dN)), t(r)
        ro = rs[owner]
        if f0 >= 0:
            ro[f0] = r[owner[f0], k - 1]
        self.ro, self.rn = t(ro), t(rs[np.maximum(nbr, 0)])
        self.sproj = t(np.abs(S[sf]).sum(1) / 2.0)
        self.eps2 = t((VENKAT_K * vol ** (1.0 / nd)) ** 3)
        self.wall = t(bt[sf] == mg.SLIP_WALL)
        self.nc = t((S / area[:, None])[sf])

    @staticmethod
    def _metrics(p, nd):
        if nd == 2:
            e = p[:, 1] - p[:, 0]
            return np.stack([e[:, 1], -e[:, 0]], 1), p.mean(axis=1)
        return np.cross(p[:, 2] - p[:, 1], p[:, 0] - p[:, 1]) / 2.0, p.mean(axis=1)


def _prim(U, nd):
    rho, u = U[:, 0], U[:, 1:1 + nd] / U[:, :1]
    q2 = (u ** 2).sum(1)
    p = (GAMMA - 1.0) * (U[:, -1] - rho * q2 / 2.0)
    return rho, u, p, q2


def _phys(rho, u, p, n):
    V = (u * n).sum(1)
    E = GAMMA / (GAMMA - 1.0) * p + rho * (u ** 2).sum(1) / 2.0   # rho * total enthalpy
    return torch.cat([(rho * V)[:, None], rho[:, None] * u * V[:, None] + p[:, None] * n, (E * V)[:, None]], 1)


def _roe(UL, UR, n, nd):
    rl, ul, pl, ql = _prim(UL, nd)
    rr, ur, pr, qr = _prim(UR, nd)
    F = _phys(rl, ul, pl, n) + _phys(rr, ur, pr, n)
    HL, HR = (UL[:, -1] + pl) / rl, (UR[:, -1] + pr) / rr
    sl, sr = rl.sqrt(), rr.sqrt()
    a = (rl * rr).sqrt()
    u = (ul * sl[:, None] + ur * sr[:, None]) / (sl + sr)[:, None]
    H = (HL * sl + HR * sr) / (sl + sr)
    q, V = (u ** 2).sum(1), (u * n).sum(1)
    c = ((GAMMA - 1.0) * (H - q / 2.0)).sqrt()
    dp, dr, du = pr - pl, rr - rl, ur - ul
    dV = (du * n).sum(1)
    d = c * HARTEN
    fix = lambda lam: torch.where(lam > d, lam, (lam ** 2 + d ** 2) / (2 * d))  # noqa: E731
    for s in (-1.0, 1.0):
        k = fix((V + s * c).abs()) * (dp + s * a * c * dV) / (2 * c * c)
        F = F - k[:, None] * torch.cat([torch.ones_like(k)[:, None], u + s * c[:, None] * n, (H + s * c * V)[:, None]],
                                       1)
    lam = fix(V.abs())
    c1, c2 = lam * (dr - dp / (c * c)), lam * a
    F = F - torch.cat([c1[:, None], c1[:, None] * u + c2[:, None] * (du - dV[:, None] * n),
                       (c1 * q / 2.0 + c2 * ((du * u).sum(1) - dV * V))[:, None]], 1)
    return F / 2.0


def _far(UL, fin, n, nd):
    r, u, p, _ = _prim(UL, nd)
    V = (u * n).sum(1)
    c = (GAMMA * p / r).sqrt()
    ri, ui, pi = fin[0], fin[1:1 + nd], fin[1 + nd]
    one = torch.ones_like(r)
    t = ((ui - u) * n).sum(1)
    pb = (pi + p - r * c * t) / 2.0
    Fin = _phys(ri + (pb - pi) / c ** 2, ui - ((pi - pb) / (r * c))[:, None] * n, pb, n)
    Fout = _phys(r + (pi - p) / c ** 2, u + ((p - pi) / (r * c))[:, None] * n, pi * one, n)
    Fi, Fo = _phys(ri * one, ui.expand_as(u), pi * one, n), _phys(r, u, p, n)
    sup, neg = ((V.abs() / c) >= 1)[:, None], (V <= 0)[:, None]
    return torch.where(neg, torch.where(sup, Fi, Fin), torch.where(sup, Fo, Fout))


def _residual(g, U, fin):
    nd = g.nd
    inner = g.adj >= 0
    Uj = U[g.adj.clamp(min=0)]                                    # [ne][k][nv]
    Ui = U[:, None, :].expand_as(Uj)
    fv = torch.where(inner[..., None], g.w[..., None] * Ui + (1 - g.w[..., None]) * Uj, Ui)
    m = Ui[..., 1:1 + nd]
    tang = m - (m * g.nc).sum(-1, keepdim=True) * g.nc
    fv = torch.cat([fv[..., :1], torch.where(g.wall[..., None], tang, fv[..., 1:1 + nd]), fv[..., 1 + nd:]], -1)
    G = (fv[..., :, None] * g.Sc[:, :, None, :]).sum(1) / g.vol[:, None, None]   # [ne][nv][nd]
    big = torch.where(inner[..., None], Uj, Ui)
    dmax = torch.maximum(big.amax(1), U) - U
    dmin = torch.minimum(big.amin(1), U) - U
    d2 = (G[:, None] * g.r[:, :, None, :]).sum(-1) / 2.0          # [ne][k][nv]
    b = torch.where(d2 > 0, dmax[:, None], dmin[:, None])
    e2 = g.eps2[:, None, None]
    f = (b * b + e2 + 2.0 * d2 * b) / (b * b + 2.0 * d2 * d2 + b * d2 + e2)
    f = torch.where((d2 != 0) & inner[..., None], f, torch.ones_like(f))
    G = G * f.amin(1).clamp(max=1.0)[..., None]
    UL = U[g.owner] + (G[g.owner] * g.ro[:, None, :]).sum(-1)
    F = torch.empty_like(UL)
    i, w, o = (torch.nonzero(g.bt == t).reshape(-1) for t in (mg.INTERNAL, mg.SLIP_WALL, mg.FREESTREAM))
    j = g.nbr[i]
    F[i] = _roe(UL[i], U[j] + (G[j] * g.rn[i][:, None, :]).sum(-1), g.n[i], nd)
    p = _prim(UL[w], nd)[2]
    F[w] = torch.cat([torch.zeros_like(p)[:, None], p[:, None] * g.n[w], torch.zeros_like(p)[:, None]], 1)
    F[o] = _far(UL[o], fin, g.n[o], nd)
    FA = F * g.area[:, None]
    return (FA[g.sf] * g.sgn[..., None]).sum(1)


def _dt_over_vol(g, U, cfl):
    r, u, p, _ = _prim(U, g.nd)
    c = GAMMA * (p / r).sqrt()   # the time step's sound speed: sqrt(gamma (gamma - 1) (H - q^2/2))
    return cfl / ((c[:, None] + u.abs()) * g.sproj).sum(1)


def exact(case, seed):
    """Explicit runs: state and monitors; residuals; the monitors of an assembled
    system.  A Krylov iterate stopped at a tolerance, and what training makes of
    the network, have no value of their own."""
    if case["work"] == "run":
        return None
    md, P, U = _inputs(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if case["work"] == "explicit":
        evals = md.ncell * case["batch"] * case["steps"] * case["rk"]
        if evals > (4e8 if dev == "cuda" else 4e6):
            return None
    g = _Geo(md, dev)
    outs, mons = [], []
    for b in range(case["batch"]):
        fin, Ub = torch.as_tensor(P[b], device=dev), torch.as_tensor(U[b], device=dev)
        if case["work"] == "explicit":
            mon = []
            for _ in range(case["steps"]):
                U0, dtv = Ub, _dt_over_vol(g, Ub, CFL_EXPLICIT)
                for al in RK4 if case["rk"] == 4 else RK3:
                    R = _residual(g, Ub, fin)
                    Ub = U0 - (al * dtv)[:, None] * R
                mon.append(R.abs().amax(0))
            outs.append(Ub.cpu().numpy())
            mons.append(torch.stack(mon).cpu().numpy())
        else:
            R = _residual(g, Ub, fin)
            if case["work"] == "residual":
                return {"R": R.cpu().numpy(), "max": R.abs().amax(0).cpu().numpy()}
            lb = (R * _dt_over_vol(g, Ub, case["cfl"])[:, None]).abs().amax(0)
            out = {"linf_b": lb.cpu().numpy(), "linf_r": R.abs().amax(0).cpu().numpy(), "x": None}
            if case["work"] == "train":
                out.update(loss=None, params=None)
            return out
    if case["batch"] == 1:
        return {"U": outs[0], "linf": mons[0]}
    return {"U": np.stack(outs), "linf": np.stack(mons, axis=1)}
