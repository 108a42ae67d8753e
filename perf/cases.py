"""The workloads whose speed matters to a user of nmesh_amd, their least work
and their results in plain torch.

Three things are done with the library: scalarwave1 is evolved on DG or FV
elements of box and cubed-sphere meshes (one right-hand side, or Runge-Kutta
steps, with the state handed over in device memory), the discrete adjoint of
those steps is taken, and special-relativistic Euler is evolved on a periodic
FV grid (whose state is handed over in host memory).
"""
import math

import numpy as np
import torch

import nmesh_amd as nm
from nmesh_amd import adjoint
from nmesh_amd.fv import FvGrid

DEV = "cuda"
ORDER_SEED = 2026          # per-element orders of the mixed meshes: part of the mesh, not of the data
WAVE = (0.8, -0.5, 0.33166247903554)   # the plane wave outside the outer boundary
STAGES = {"RK4": 4, "sspRK3": 3, "Euler": 1}
RIN, ROUT, DOUT = 2.0, 20.0, 8.0


def _mesh_case(name, what, mesh, luni, n_lo, n_hi, steps, **kw):
    c = {"name": name, "what": what, "mesh": mesh, "luni": luni, "n_lo": n_lo, "n_hi": n_hi, "steps": steps,
         "spheres": 0, "radius": 3, "flux": "upwind", "method": "RK4", "wave": False, "filter": False,
         "fv": "", "rec": "", "midpoint": "no", "path": "plain", "geometry": "analytic"}
    c.update(kw)
    if name is None:
        del c["name"]
    return c


def listed():
    return [
        # one right-hand side on a few elements, the least a host program
        # asks for (an own integrator, a test of a new flux)
        _mesh_case("rhs_box", "steps", "box", 2, 5, 5, 0),
        # a small box evolved for many steps: launches and latency
        _mesh_case("steps_box", "steps", "box", 2, 5, 5, 100),
        # a uniform cubed-sphere shell of 1.6M nodes, the usual conforming run
        _mesh_case("steps_shell", "steps", "shell", 3, 8, 8, 40),
        # an odd order, the other flux and integrator, a wave coming in through
        # the outer boundary and the exponential filter after each step
        _mesh_case("steps_shell_filter", "steps", "shell", 2, 7, 7, 25, flux="LLF", method="sspRK3", wave=True,
                   filter=True),
        # a small refined mesh of mixed orders
        _mesh_case("steps_amr_small", "steps", "shell", 1, 3, 7, 20, spheres=1, radius=8, path="batched"),
        # the large one: 19,200 elements of 4 to 10 points on three levels
        _mesh_case("steps_amr", "steps", "shell", 3, 4, 10, 16, spheres=2, radius=3, path="batched"),
        # the gradient of a boundary misfit through a small box's evolution
        _mesh_case("grad_box", "grad", "box", 2, 5, 5, 256),
        # adjoint steps on a refined mesh of mixed orders
        _mesh_case("adjoint_amr", "adjoint", "shell", 2, 4, 10, 8, spheres=2, radius=4, path="batched"),
        # FV elements throughout (WENO5 inside, WENO3 beside the faces)
        _mesh_case("steps_fv_box", "steps", "box", 4, 8, 8, 8, fv="0", rec="WENOm5_2"),
        # DG and FV patches side by side on a curved mesh
        _mesh_case("steps_fv_dg_shell", "steps", "shell", 2, 6, 6, 16, fv="0 2 4", rec="WENOmZ_2", midpoint="yes",
                   path="batched"),
        # a small relativistic-flow grid, from host data to host data
        {"name": "grid_small", "what": "grid", "n": 48, "method": "RK4", "steps": 20},
        # the large one: 16.8M cells
        {"name": "grid", "what": "grid", "n": 256, "method": "sspRK3", "steps": 50},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dg", "dg", "amr", "amr", "adjoint", "grad", "fv", "fv", "grid"])
    method = rng.choice(["RK4", "RK4", "sspRK3", "Euler"])
    if kind == "grid":
        n = 16 * _log(rng, 2, 14)
        return {"what": "grid", "n": n, "method": rng.choice(["RK4", "sspRK3"]), "steps": _log(rng, 1, 30)}
    opts = {"flux": rng.choice(["upwind", "LLF"]), "method": method}
    if kind == "grad":
        n = rng.randint(3, 8)
        return _mesh_case(None, "grad", rng.choice(["box", "shell"]), rng.randint(1, 2), n, n, _log(rng, 4, 128), **opts)
    if kind == "fv":
        mesh = rng.choice(["box", "shell"])
        n = rng.randint(4, 10)
        opts.update(rec=rng.choice(["WENOm3_2", "WENOm5_2", "WENOmZ_2"]), wave=rng.random() < 0.5)
        if mesh == "box":
            return _mesh_case(None, "steps", mesh, rng.randint(1, 4), n, n, _log(rng, 1, 16), fv="0", **opts)
        mixed = rng.random() < 0.5
        return _mesh_case(None, "steps", mesh, rng.randint(1, 3), n, n, _log(rng, 1, 16),
                          midpoint=rng.choice(["no", "yes"]), path="batched" if mixed else "plain",
                          fv=rng.choice(["0 2 4", "1 3 5", "5"]) if mixed else "0 1 2 3 4 5", **opts)
    opts.update(wave=rng.random() < 0.4 and kind != "adjoint", filter=rng.random() < 0.2 and kind != "adjoint",
                geometry="stored" if rng.random() < 0.15 else "analytic")
    if kind == "dg" or (kind == "adjoint" and rng.random() < 0.4):
        mesh = rng.choice(["box", "shell"])
        n = rng.randint(3, 10)
        luni = rng.randint(1, 4 if mesh == "box" else 3)
        steps = _log(rng, 1, 60) if rng.random() < 0.8 or kind == "adjoint" else 0
        return _mesh_case(None, "adjoint" if kind == "adjoint" else "steps", mesh, luni, n, n, steps, **opts)
    lo = rng.randint(3, 7)
    return _mesh_case(None, "adjoint" if kind == "adjoint" else "steps", "shell", rng.randint(1, 2), lo,
                      rng.randint(lo + 1, 10), _log(rng, 1, 24), spheres=rng.randint(0, 2), radius=rng.choice([3, 5, 8]),
                      path="batched", **opts)


# ---------------------------------------------------------------------------
# the mesh's elements, as nmesh orders them
# ---------------------------------------------------------------------------

class Forest:
    """Patches and leaf elements in depth-first octant order."""

    def __init__(self, c):
        box = c["mesh"] == "box"
        npat = 1 if box else 6
        self.box = box
        self.lo = np.array([-DOUT] * 3 if box else [0.0, -1.0, -1.0])
        self.len = np.array([2 * DOUT] * 3 if box else [1.0, 2.0, 2.0])
        self.p = np.arange(npat)
        self.l = np.zeros(npat, int)
        self.ic = np.zeros((npat, 3), int)
        for _ in range(c["luni"]):
            self._refine(np.ones(len(self.p), bool))
        if not box:
            r = c["radius"] * 2.0 ** (c["spheres"] - 1)
            for _ in range(c["spheres"]):   # the element's centre lies at radius rin + (rout - rin) lam
                lo, hi = self.bounds()
                self._refine(RIN + (ROUT - RIN) * 0.5 * (lo + hi)[:, 0] <= r)
                r *= 0.5
        if c["n_lo"] == c["n_hi"]:
            self.n = np.full(len(self.p), c["n_lo"])
        else:
            self.n = np.random.default_rng(ORDER_SEED).integers(c["n_lo"], c["n_hi"] + 1, len(self.p))
        self.off = np.concatenate([[0], np.cumsum(self.n ** 3)])
        self.nnodes = int(self.off[-1])
        self.fv = np.isin(self.p, [int(q) for q in c["fv"].split()])

    def _refine(self, flag):
        rep = np.where(flag, 8, 1)
        idx = np.repeat(np.arange(len(flag)), rep)
        child = np.arange(len(idx)) - np.repeat(np.cumsum(rep) - rep, rep)
        fl = flag[idx]
        bits = (child[:, None] >> np.arange(3)) & 1
        self.ic = np.where(fl[:, None], 2 * self.ic[idx] + bits, self.ic[idx])
        self.p, self.l = self.p[idx], self.l[idx] + fl

    def bounds(self):
        w = self.len / 2.0 ** self.l[:, None]
        return self.lo + self.ic * w, self.lo + (self.ic + 1) * w


def _dt(c, F):
    """a stable step: a fraction of the least distance of two nodes"""
    lo, hi = F.bounds()
    w = hi - lo
    if not F.box:   # radial and angular widths at the inner end of the element
        r0 = RIN + (ROUT - RIN) * lo[:, 0]
        w = np.stack([(ROUT - RIN) * w[:, 0], 0.5 * r0 * w[:, 1], 0.5 * r0 * w[:, 2]], 1)
    frac = np.array([_lgl(n)[0][1] + 1.0 for n in range(2, 11)])[F.n - 2] / 2
    return float(0.2 * (w.min(1) * frac).min())


def _params(c):
    n = c["n_lo"]
    k = WAVE if c["wave"] else (0, 0, 0)
    p = {"amr_mesh_type": "BoxMesh" if c["mesh"] == "box" else "Shell", "amr_luni": c["luni"], "amr_n0": n, "amr_n1": n,
         "amr_n2": n, "amr_BoxMesh_dout": DOUT, "amr_Shell_rin": RIN, "amr_Shell_rout": ROUT,
         "amr_hrefine_sphere_radius": c["radius"], "amr_hrefine_sphere_levels": c["spheres"],
         "scalarwave1_k": "%.17g %.17g %.17g" % tuple(k), "scalarwave1_numflux": c["flux"], "evolve_method": c["method"],
         "nmx_path": c["path"], "nmx_geometry": c["geometry"], "evolve_filter_all": "yes" if c["filter"] else "no"}
    if c["fv"]:
        p.update(amr_uniform_p=c["fv"], amr_fv_p=c["fv"], fv_rec=c["rec"], coordinates_midpoint_data=c["midpoint"],
                 basis_filter_fv="no")
    return p


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _wave_data(x, seed, box):
    """psi a pulse (box) or a Gaussian shell with an angular modulation, Phi_i
    its gradient, Pi a tenth of it; x[3][node]"""
    g = np.random.default_rng(seed)
    a = g.uniform(-0.1, 0.1, 4)
    if box:
        y = x - torch.tensor(g.uniform(-2, 2, 3), device=DEV)[:, None]
        psi = torch.exp(-(y ** 2).sum(0) / 4)
        dpsi = -0.5 * y * psi
    else:
        r = (x ** 2).sum(0).sqrt()
        d = torch.tensor(a[:3], device=DEV)
        ang = 1 + a[3] + (d[:, None] * x).sum(0) / r
        e = torch.exp(-(r - 8.0) ** 2 / 2)
        psi = e * ang
        dpsi = -(r - 8.0) * e * ang * x / r + e * (d[:, None] / r - x * (d[:, None] * x).sum(0) / r ** 3)
    return torch.cat([0.1 * psi[None], dpsi, psi[None]]).reshape(-1).contiguous()


def _flow_data(n, seed):
    """rho 1 plus 16 periodic Gaussian blobs, velocities U[-0.3, 0.3] per cell,
    p between 0.9 and 1.1; [5][z][y][x]"""
    g = np.random.default_rng(seed)
    t = torch.Generator(device=DEV).manual_seed(int(seed))
    x = torch.arange(n, device=DEV, dtype=torch.float64) + 0.5
    rho = torch.ones(n, n, n, dtype=torch.float64, device=DEV)
    for _ in range(16):
        amp, w = g.uniform(0.1, 1.0), g.uniform(2.0, 8.0)
        e = []
        for xc in g.uniform(0, n, 3):
            d = x - xc
            e.append(torch.exp(-(d - n * torch.round(d / n)) ** 2 / (2 * w * w)))
        rho += amp * e[0][:, None, None] * e[1][None, :, None] * e[2][None, None, :]
    v = 0.6 * torch.rand(3, n, n, n, dtype=torch.float64, device=DEV, generator=t) - 0.3
    p = 0.9 + 0.2 * torch.rand(1, n, n, n, dtype=torch.float64, device=DEV, generator=t)
    return torch.cat([rho[None], v, p])


def _mesh_input(c, F, seed, x):
    if c["what"] == "adjoint":
        t = torch.Generator(device=DEV).manual_seed(int(seed))
        return torch.randn(5 * F.nnodes, dtype=torch.float64, device=DEV, generator=t)
    return _wave_data(x, seed, F.box)


def prepare(c, seed):
    if c["what"] == "grid":
        g = FvGrid({"fv_n": c["n"], "evolve_method": c["method"]})
        g.setup()
        return {"case": c, "grid": g, "prim": _flow_data(c["n"], seed).cpu().numpy().reshape(-1)}
    F = Forest(c)
    m = nm.Mesh(_params(c))
    nm.amr_setup_mesh(m)
    if c["n_lo"] != c["n_hi"]:
        m.set_elm_n(F.n)
    m.dt = _dt(c, F)
    x = torch.from_numpy(m.coords()).to(DEV)
    u = _mesh_input(c, F, seed, x)
    s = {"case": c, "mesh": m, "in": u, "out": torch.empty_like(u)}
    if c["what"] == "grad":
        s["nodes"] = adjoint.outer_boundary_nodes(m)
        s["target"] = s["in"].reshape(5, -1)[4][s["nodes"]] * 0.5 + 0.01
    nm.autotune(m)
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(s):
    c = s["case"]
    if c["what"] == "grid":
        g = s["grid"]
        g.upload_prim(s["prim"])
        g.evolve(c["steps"])
        return g.download()
    m = s["mesh"]
    if c["what"] == "adjoint":
        return adjoint.adjoint_evolve(m, s["in"], c["steps"])
    if c["what"] == "grad":
        m.time = 0.0
        u = s["in"].clone().requires_grad_(True)
        traj = adjoint.evolve(m, u, c["steps"], 16)
        psi = traj[-1].reshape(5, -1)[4][s["nodes"]]
        loss = ((psi - s["target"]) ** 2).sum()
        (grad,) = torch.autograd.grad(loss, u)
        return traj.detach(), grad
    torch.cuda.current_stream().synchronize()
    m.copy_in(s["in"].data_ptr())
    if c["steps"] == 0:
        nm.evolve.check(nm.lib().nmx_setrhs(m.ctx, nm.REG_R, nm.REG_U, 0.0))
        m.copy_out(s["out"].data_ptr(), nm.REG_R)
    else:
        m.time = 0.0
        nm.evolve_myln(m, c["steps"])
        m.copy_out(s["out"].data_ptr())
    m.synchronize()
    return s["out"]


# ---------------------------------------------------------------------------
# least work
# ---------------------------------------------------------------------------

# doubles per node that a step's fused stages read and write: the first reads
# u and writes two registers, the inner ones read three and write two (the
# second of sspRK3 the same), the last reads two and writes one
STEP_DOUBLES = {"RK4": 80, "sspRK3": 55, "Euler": 10}


def work(c):
    if c["what"] == "grid":
        cells, s = c["n"] ** 3, STAGES[c["method"]] * c["steps"]
        # per stage the primitives' solve (reads u and a guess, writes 5) and
        # one read of them, beside the step's registers; per cell 3 faces of
        # 10 reconstructions and two fluxes, about 2700 operations
        return {"bytes": 8.0 * cells * (s * 16 + c["steps"] * STEP_DOUBLES[c["method"]] + 10), "flops": 2700.0 * cells * s}
    F = Forest(c)
    n = F.n.astype(float)
    nodes = n ** 3
    stages = STAGES[c["method"]] * c["steps"]
    # 12 derivatives of 2n operations (4 on a box) and 36 for their sums on DG
    # elements; about 12 reconstructions of 60 and the fluxes on FV ones
    per = np.where(F.fv, 1300.0, (8.0 if F.box else 24.0) * n + 36.0)
    per_filter = 30.0 * n if c["filter"] else 0.0
    if c["steps"] == 0:
        return {"bytes": 8.0 * 10 * F.nnodes, "flops": float((nodes * per).sum())}
    both = 2 if c["what"] == "grad" else 1
    doubles = both * c["steps"] * (STEP_DOUBLES[c["method"]] + (10 if c["filter"] else 0)) + 10
    if c["what"] == "grad":
        doubles += 5 * -(-c["steps"] // 16)
    return {"bytes": 8.0 * doubles * F.nnodes,
            "flops": float((nodes * (both * stages * per + c["steps"] * per_filter)).sum())}


def tolerance(c):
    # everything is held and summed in 64 bits.  Against the same steps in
    # plain torch the outputs are off by 3e-16 to 4e-15, and by 1.2e-14 with
    # the filter's Jacobian weighting after each step.
    return {"rel": 5e-14 if c.get("filter") else 2e-14, "max": 1e-11}


# ---------------------------------------------------------------------------
# the same in plain torch
# ---------------------------------------------------------------------------

def _lgl(n):
    """Legendre-Gauss-Lobatto nodes and weights: the ends and the roots of P'_{n-1}"""
    P = np.polynomial.legendre.Legendre.basis(n - 1)
    x = np.concatenate([[-1.0], np.sort(np.real(P.deriv().roots())), [1.0]])
    for _ in range(3):
        x[1:-1] -= P.deriv()(x[1:-1]) / P.deriv(2)(x[1:-1])
    x = 0.5 * (x - x[::-1])
    return x, 2.0 / (n * (n - 1) * P(x) ** 2)


def _bary(x):
    return np.array([1.0 / np.prod([x[q] - x[m] for m in range(len(x)) if m != q]) for q in range(len(x))])


def _deriv(n):
    x, _ = _lgl(n)
    w = _bary(x)
    D = np.array([[0.0 if i == l else w[l] / w[i] / (x[i] - x[l]) for l in range(n)] for i in range(n)])
    return D - np.diag(D.sum(1))


def _filter_matrix(n):
    """synthesis x exp(-36 (i/N)^32) x analysis in normalised Legendre polynomials"""
    x, w = _lgl(n)
    V = np.stack([np.polynomial.legendre.Legendre.basis(i)(x) for i in range(n)], 1)
    c = np.array([(2 * i + 1) / 2 for i in range(n)])
    c[-1] = (n - 1) / 2
    f = np.exp(-36.0 * (np.arange(n) / (n - 1)) ** 32)
    return (V * (c * f)) @ (V.T * w)


def _t(a, dtype=torch.float64):
    return torch.as_tensor(np.asarray(a), dtype=dtype, device=DEV)


def _axes(p):
    """axis that patch p's radial coordinate runs along, those A and B scale, its sign"""
    d = p // 2
    ia = torch.where(d == 1, 0, 1)
    return d, ia, 3 - d - ia, 2.0 * (p % 2) - 1


def _xyz(p, X):
    """Cartesian point of patch point X = (lam, A, B): x[3 .. last]"""
    d, ia, ib, sg = _axes(p)
    r = sg * (RIN + (ROUT - RIN) * X[..., 0]) / torch.sqrt(1 + X[..., 1] ** 2 + X[..., 2] ** 2)
    x = torch.zeros_like(X)
    x.scatter_(-1, d[..., None], r[..., None])
    x.scatter_(-1, ia[..., None], (X[..., 1] * r)[..., None])
    x.scatter_(-1, ib[..., None], (X[..., 2] * r)[..., None])
    return x


def _patch_point(p, x):
    """patch coordinates of Cartesian x in patch p"""
    d, ia, ib, _ = _axes(p)
    r = x.gather(-1, d[..., None])[..., 0]
    A = x.gather(-1, ia[..., None])[..., 0] / r
    B = x.gather(-1, ib[..., None])[..., 0] / r
    return torch.stack([((x ** 2).sum(-1).sqrt() - RIN) / (ROUT - RIN), A, B], -1)


def _metric(F, p, X):
    """dX^m/dx^q at patch point X: M[..][m][q]"""
    M = torch.zeros(*X.shape, 3, dtype=torch.float64, device=DEV)
    if F.box:
        return M + torch.eye(3, dtype=torch.float64, device=DEV)
    d, ia, ib, sg = _axes(p)
    A, B = X[..., 1], X[..., 2]
    s = torch.sqrt(1 + A * A + B * B)
    c0, c1 = sg / ((ROUT - RIN) * s), sg * s / (RIN + (ROUT - RIN) * X[..., 0])
    for m, k, v in ((0, d, c0), (0, ia, A * c0), (0, ib, B * c0), (1, d, -A * c1), (1, ia, c1), (2, d, -B * c1), (2, ib, c1)):
        M[..., m, :].scatter_(-1, k[..., None], v[..., None])
    return M


class Wave:
    """scalarwave1 on the case's mesh: u[5][node] -> RHS and steps."""

    def __init__(self, c):
        self.c, self.F = c, Forest(c)
        F = self.F
        self.lo, self.hi = (_t(a) for a in F.bounds())
        self.g = 2.0 / (self.hi - self.lo)
        self.p = _t(F.p, torch.long)
        self.groups = []
        base = 0
        for fv in (False, True):
            for n in range(2, 11):
                el = np.nonzero((F.n == n) & (F.fv == fv))[0]
                if len(el):
                    self.groups.append(self._group(n, fv, el, base))
                    base += 6 * n * n * len(el)
        self.npts = base
        # face points: adjacent values are sums of weights times nodes
        self._gather()

    def _coords(self, el, ref):
        """patch points of element el[i] at reference coordinates ref[..][3]"""
        sh = (-1,) + (1,) * (ref.dim() - 2) + (3,)
        lo, hi = self.lo[el].reshape(sh), self.hi[el].reshape(sh)
        return 0.5 * ((hi - lo) * ref + (hi + lo))

    def _group(self, n, fv, el, base):
        x = np.linspace(-1, 1, n) if fv else _lgl(n)[0]
        el = _t(el, torch.long)
        E = len(el)
        G = {"n": n, "fv": fv, "el": el, "x": _t(x), "base": base,
             "idx": _t(self.F.off, torch.long)[el][:, None] + torch.arange(n ** 3, device=DEV)}
        xt = _t(x)
        ref = torch.stack([xt[None, None, :].expand(n, n, n), xt[None, :, None].expand(n, n, n),
                           xt[:, None, None].expand(n, n, n)], -1)
        G["X"] = self._coords(el, ref.unsqueeze(0))
        G["p"] = self.p[el].reshape(E, 1, 1, 1).expand(E, n, n, n)
        G["M"] = _metric(self.F, G["p"], G["X"])
        G["ooJ"] = self.g[el].prod(1).reshape(E, 1, 1, 1) * torch.linalg.det(G["M"])
        G["xyz"] = G["X"] if self.F.box else _xyz(G["p"], G["X"])
        G["D"] = _t(_deriv(n)) if not fv else None
        G["wend"] = _lgl(n)[1][0]
        G["filt"] = _t(_filter_matrix(n)) if not fv else None
        return G

    @staticmethod
    def _face(T, d, side):
        """face plane [.., b, a] of T[.., k, j, i]"""
        return T.select(-1 - d, 0 if side == 0 else T.shape[-1] - 1)

    def _gather(self):
        F = self.F
        L = int(F.l.max())
        N = 2 ** L
        leaf = np.full((len(set(F.p.tolist())), N, N, N), -1)
        for lev in np.unique(F.l):
            e = np.nonzero(F.l == lev)[0]
            s = 2 ** (L - lev)
            o = np.arange(s)
            i = (F.ic[e, 0, None] * s + o)[:, :, None, None]
            j = (F.ic[e, 1, None] * s + o)[:, None, :, None]
            k = (F.ic[e, 2, None] * s + o)[:, None, None, :]
            leaf[F.p[e][:, None, None, None], i, j, k] = e[:, None, None, None]
        leaf, lo, ln = _t(leaf, torch.long), _t(F.lo), _t(F.len)
        n_of, fv_of, off_of = _t(F.n, torch.long), _t(F.fv, torch.bool), _t(F.off, torch.long)

        def across(p, X):
            """patch and patch point of X of patch p, which may lie just outside it; whether it lies in the mesh"""
            if F.box:
                return p, X, ((X - lo).abs() <= ln).logical_and(X >= lo).all(-1)
            x = _xyz(p, X)
            d = x.abs().argmax(-1)
            q = 2 * d + (x.gather(-1, d[..., None])[..., 0] > 0)
            return q, _patch_point(q, x), (X[..., 0] > 0) & (X[..., 0] < 1)

        def find(q, X):
            ijk = ((X - lo) / ln * N).floor().long().clamp(0, N - 1)
            return leaf[q, ijk[..., 0], ijk[..., 1], ijk[..., 2]]

        found = {}   # (order, kind) of the neighbour: (points, element, weight, patch point, normal direction, side)
        for G in self.groups:
            n, el, xt = G["n"], G["el"], G["x"]
            E = len(el)
            for f in range(6):
                d, side = f // 2, f % 2
                t1, t2 = [q for q in range(3) if q != d]
                ref = torch.zeros(1, n, n, 3, dtype=torch.float64, device=DEV)   # [b][a]
                ref[..., d] = 2.0 * side - 1
                ref[..., t1] = xt[None, None, :]
                ref[..., t2] = xt[None, :, None]
                p = self.p[el].reshape(E, 1, 1).expand(E, n, n)
                mid = torch.zeros(1, 1, 1, 3, dtype=torch.float64, device=DEV)
                mid[..., d] = (2.0 * side - 1) * (1 + 1e-5)
                q0, Xm, inside = across(p[:, :1, :1], self._coords(el, mid))
                q0, inside = q0.expand(E, n, n), inside.expand(E, n, n)
                Xf = self._coords(el, ref)
                # the neighbours' face: the same direction, or the patch boundary
                if F.box:
                    Xq, d2, s2 = Xf, torch.full_like(q0, d), torch.full_like(q0, 1 - side)
                else:
                    same = q0 == p
                    Xq = torch.where(same[..., None], Xf, _patch_point(q0, _xyz(p, Xf)))
                    eB = (Xm[..., 2].abs() > Xm[..., 1].abs()).expand(E, n, n)
                    d2 = torch.where(same, d, torch.where(eB, 2, 1))
                    s2 = torch.where(same, 1 - side, (Xm.expand(E, n, n, 3).gather(-1, d2[..., None])[..., 0] > 0).long())
                cand = []
                for sa in (-1, 1):
                    for sb in (-1, 1):
                        nd = ref.clone()
                        nd[..., d] *= 1 + 1e-5
                        ea = torch.where(xt == 1, -1.0, torch.where(xt == -1, 1.0, float(sa)))
                        eb = torch.where(xt == 1, -1.0, torch.where(xt == -1, 1.0, float(sb)))
                        nd[..., t1] += 1e-5 * ea[None, None, :]
                        nd[..., t2] += 1e-5 * eb[None, :, None]
                        q, X, _ = across(p, self._coords(el, nd))
                        cand.append(find(q, X))
                cand = torch.stack(cand, -1).sort(-1)[0]
                new = torch.ones_like(cand, dtype=torch.bool)
                new[..., 1:] = cand[..., 1:] != cand[..., :-1]
                new &= inside[..., None]
                w = new / new.sum(-1, keepdim=True).clamp(min=1)
                pts = G["base"] + ((torch.arange(E, device=DEV)[:, None, None] * 6 + f) * n * n +
                                   torch.arange(n, device=DEV)[:, None] * n + torch.arange(n, device=DEV))
                for k in range(4):
                    keep = new[..., k]
                    e2, pt = cand[..., k][keep], pts[keep]
                    ww, XX, dd, ss = w[..., k][keep], Xq[keep], d2[keep], s2[keep]
                    for m in torch.unique(n_of[e2]).tolist():
                        for fv in (False, True):
                            h = (n_of[e2] == m) & (fv_of[e2] == fv)
                            if h.any():
                                found.setdefault((m, fv), []).append((pt[h], e2[h], ww[h], XX[h], dd[h], ss[h]))
        self.sources = []
        for (m, fv), parts in found.items():
            pt, e2, ww, XX, dd, ss = (torch.cat(z) for z in zip(*parts))
            ref = (2 * XX - self.lo[e2] - self.hi[e2]) / (self.hi[e2] - self.lo[e2])
            u1, u2 = (dd == 0).long(), torch.where(dd == 2, 1, 2)     # the face's own two directions
            r1 = self._rows(m, fv, ref.gather(-1, u1[:, None])[:, 0])
            r2 = self._rows(m, fv, ref.gather(-1, u2[:, None])[:, 0])
            stride = torch.tensor([1, m, m * m], device=DEV)
            a = torch.arange(m, device=DEV)
            node = (off_of[e2] + ss * (m - 1) * stride[dd])[:, None, None] + \
                a[None, :, None] * stride[u2][:, None, None] + a[None, None, :] * stride[u1][:, None, None]
            W = ww[:, None, None] * r2[:, :, None] * r1[:, None, :]
            W, node = W.reshape(len(pt), -1), node.reshape(len(pt), -1)
            one = (W.abs() > 0.9999999).any(1) & ((W.abs() > 1e-12).sum(1) == 1)   # points that meet a node
            if one.any():
                j = W[one].abs().argmax(1)
                self.sources.append((pt[one], node[one].gather(1, j[:, None]), torch.ones(int(one.sum()), 1, dtype=torch.float64, device=DEV)))
            if (~one).any():
                self.sources.append((pt[~one], node[~one], W[~one]))

    @staticmethod
    def _rows(m, fv, x):
        if fv:   # piecewise linear on uniform points
            s = ((x + 1) * (m - 1) / 2).clamp(0, m - 1)
            return (1 - (s[:, None] - torch.arange(m, device=DEV)).abs()).clamp(min=0)
        xn, wb = _lgl(m)[0], _bary(_lgl(m)[0])
        df = x[:, None] - _t(xn)
        return torch.stack([df[:, [k for k in range(m) if k != q]].prod(1) * wb[q] for q in range(m)], 1)

    def _adjacent(self, u, t):
        aj = torch.zeros(4, self.npts, dtype=torch.float64, device=DEV)
        if self.c["wave"]:
            k = _t(WAVE)
            om = k.norm()
            for G in self.groups:
                v = torch.cos((G["xyz"] * k).sum(-1) - om * t)
                v = torch.stack([-om * v, k[0] * v, k[1] * v, k[2] * v])
                n = G["n"]
                z = torch.stack([self._face(v, f // 2, f % 2) for f in range(6)], 2)   # [4][E][6][b][a]
                aj[:, G["base"]:G["base"] + z[0].numel()] = z.reshape(4, -1)
        seen = torch.zeros(self.npts, dtype=torch.bool, device=DEV)
        for pt, _, _ in self.sources:
            seen[pt] = True
        aj = torch.where(seen, torch.zeros_like(aj), aj)
        for pt, node, W in self.sources:
            for i in range(0, len(pt), 1 << 18):
                q = slice(i, i + (1 << 18))
                aj = aj.index_add(1, pt[q], (u[:4][:, node[q]] * W[q]).sum(-1))
        return aj

    def _jump(self, nrm, d):
        """F = fnum - f of the jumps d[4], normals nrm[..][3]"""
        nv = nrm.movedim(-1, 0)
        Fp = 0.5 * (d[0] + (nv * d[1:]).sum(0))
        if self.c["flux"] == "upwind":
            return torch.cat([Fp[None], nv * Fp])
        return torch.cat([Fp[None], 0.5 * (d[1:] + nv * d[0])])

    def rhs(self, u, t):
        aj = self._adjacent(u, t)
        r = torch.zeros_like(u)
        for G in self.groups:
            n, E = G["n"], len(G["el"])
            U = u[:, G["idx"]].reshape(5, E, n, n, n)
            A = aj[:, G["base"]:G["base"] + 6 * n * n * E].reshape(4, E, 6, n, n)
            R = self._fv(G, U, A) if G["fv"] else self._dg(G, U, A)
            r = r.index_copy(1, G["idx"].reshape(-1), torch.cat([R, U[:1]]).reshape(5, -1))
        return r

    def _dg(self, G, U, A):
        n, E = G["n"], len(G["el"])
        D, M = G["D"], G["M"]
        g = self.g[G["el"]].reshape(E, 1, 1, 1, 3)
        rows = [torch.zeros_like(U[0]) for _ in range(4)]
        for m in range(3):
            T = torch.matmul(U[:4].movedim(-1 - m, -1).contiguous(), D.T.contiguous()).movedim(-1, -1 - m) * g[..., m]
            rows[0] = rows[0] + (M[..., m, :].movedim(-1, 0) * T[1:]).sum(0)
            for q in range(3):
                rows[1 + q] = rows[1 + q] + M[..., m, q] * T[0]
        R = torch.stack(rows)
        for f in range(6):
            d, side = f // 2, f % 2
            nr = self._face(M[..., d, :].movedim(-1, 0), d, side).movedim(0, -1)
            s = nr.norm(dim=-1)
            F = self._jump((2 * side - 1) * nr / s[..., None], self._face(U[:4], d, side) - A[:, :, f])
            lift = F * s * (self.g[G["el"]][:, d] / G["wend"])[:, None, None]
            pad = torch.zeros(n, dtype=torch.float64, device=DEV)
            pad[0 if side == 0 else n - 1] = 1.0
            shape = [1, 1, 1]
            shape[2 - d] = n
            R = R - lift.unsqueeze(-1 - d) * pad.reshape(shape)
        return R

    def _fv(self, G, U, A):
        n, el = G["n"], G["el"]
        x = G["x"]
        h = 2.0 / (n - 1)
        wc = _t([h / 2] + [h] * (n - 2) + [h / 2])
        total = 0
        for m in range(3):
            q = U[:4].movedim(-1 - m, -1)                        # [4][E][b][a][line]
            Mn = G["M"].movedim(3 - m, 3)
            oj = G["ooJ"].movedim(-1 - m, -1)
            g = self.g[el][:, m].reshape(-1, 1, 1, 1)
            nrow = Mn[..., m, :]
            soj = g * nrow.norm(dim=-1) / oj
            if self.c["midpoint"] == "yes":
                Xm = G["X"].movedim(3 - m, 3)
                Xm = 0.5 * (Xm[..., :-1, :] + Xm[..., 1:, :])
                pm = G["p"].movedim(-1 - m, -1)[..., :-1]
                Mm = _metric(self.F, pm, Xm)
                mrow = Mm[..., m, :]
                som = g * mrow.norm(dim=-1) / (self.g[el].prod(1).reshape(-1, 1, 1, 1) * torch.linalg.det(Mm))
            else:
                mrow, som = nrow[..., :-1, :], soj[..., :-1]
            up, um = self._reconstruct(q)
            fm = self._fnum(mrow / mrow.norm(dim=-1, keepdim=True), up, um)
            un = nrow / nrow.norm(dim=-1, keepdim=True)
            fl = self._fnum(-un[..., 0, :], q[..., 0], A[:, :, 2 * m])
            fr = self._fnum(un[..., -1, :], q[..., -1], A[:, :, 2 * m + 1])
            right = torch.cat([som * fm, (soj[..., -1] * fr)[..., None]], -1)
            left = torch.cat([(soj[..., 0] * fl)[..., None], -som * fm], -1)
            df = (right + left) / wc
            a = df[..., 0] / 0.75 + (1 - 1 / 0.75) * df[..., 1]
            b = df[..., -1] / 0.75 + (1 - 1 / 0.75) * df[..., -2]
            df = torch.cat([a[..., None], df[..., 1:-1], b[..., None]], -1)
            total = total + (df * oj).movedim(-1, -1 - m)
        return -total

    def _fnum(self, nrm, ui, ua):
        nv = nrm.movedim(-1, 0)
        f = torch.cat([-(nv * ui[1:]).sum(0)[None], -nv * ui[0]])
        return f + self._jump(nrm, ui - ua)

    def _reconstruct(self, q):
        n = q.shape[-1]
        up, um = [], []
        wide = {"WENOm5_2": 5, "WENOmZ_2": 7}.get(self.c["rec"], 0)
        for i in range(n - 1):
            at = lambda *o: [q[..., i + k] for k in o]  # noqa: E731
            if wide and 2 <= i <= n - 3:
                up.append(_weno5(wide, *at(-2, -1, 0, 1, 2)))
            elif i >= 1:
                up.append(_weno3(*at(-1, 0, 1)))
            else:
                up.append(0.5 * (q[..., 0] + q[..., 1]))
            if wide and 1 <= i <= n - 4:
                um.append(_weno5(wide, *at(3, 2, 1, 0, -1)))
            elif i <= n - 3:
                um.append(_weno3(*at(2, 1, 0)))
            else:
                um.append(0.5 * (q[..., n - 2] + q[..., n - 1]))
        return torch.stack(up, -1), torch.stack(um, -1)

    def _filtered(self, u):
        out = u.clone()
        for G in self.groups:
            if G["fv"]:
                continue
            n, E = G["n"], len(G["el"])
            U = u[:, G["idx"]].reshape(5, E, n, n, n) / G["ooJ"]
            for m in range(3):
                U = torch.matmul(U.movedim(-1 - m, -1).contiguous(), G["filt"].T.contiguous()).movedim(-1, -1 - m)
            out = out.index_copy(1, G["idx"].reshape(-1), (U * G["ooJ"]).reshape(5, -1))
        return out

    def step(self, u, t, dt):
        u = _rk(self.c["method"], lambda w, s: self.rhs(w, s), u, t, dt)
        return self._filtered(u) if self.c["filter"] else u


def _rk(method, f, u, t, dt):
    if method == "RK4":
        k1 = f(u, t)
        k2 = f(u + dt / 2 * k1, t + dt / 2)
        k3 = f(u + dt / 2 * k2, t + dt / 2)
        return u + dt / 6 * (k1 + 2 * k2 + 2 * k3 + f(u + dt * k3, t + dt))
    if method == "sspRK3":
        k1 = f(u, t)
        w = u + dt * k1
        k2 = f(w, t + dt)
        return u + dt / 6 * (k1 + k2 + 4 * f(0.75 * u + 0.25 * (w + dt * k2), t + dt / 2))
    return u + dt * f(u, t)


def _weno3(a, b, c):
    """the value right of b from b - a and c - b, ideal weights 1 : 2"""
    w1, w2 = 1 / ((b - a) ** 2 + 1e-6) ** 2, 2 / ((c - b) ** 2 + 1e-6) ** 2
    return (w1 * (1.5 * b - 0.5 * a) + w2 * 0.5 * (b + c)) / (w1 + w2)


def _weno5(kind, a, b, c, d, e):
    """the value right of c: WENO5 (kind 5) or WENO-Z (7), ideal weights 1 : 6 : 3"""
    b0 = 13 / 12 * (a - 2 * b + c) ** 2 + (a - 4 * b + 3 * c) ** 2 / 4 + 1e-40
    b1 = 13 / 12 * (b - 2 * c + d) ** 2 + (b - d) ** 2 / 4 + 1e-40
    b2 = 13 / 12 * (c - 2 * d + e) ** 2 + (3 * c - 4 * d + e) ** 2 / 4 + 1e-40
    if kind == 7:
        tau = (b0 - b2).abs()
        w = (1 + tau / b0, 6 * (1 + tau / b1), 3 * (1 + tau / b2))
    else:
        s = torch.minimum(torch.minimum(b0, b1), b2)   # the weights' ratios, without overflow
        w = ((s / b0) ** 2, 6 * (s / b1) ** 2, 3 * (s / b2) ** 2)
    q = ((2 * a - 7 * b + 11 * c) / 6, (-b + 5 * c + 2 * d) / 6, (2 * c + 5 * d - e) / 6)
    return (w[0] * q[0] + w[1] * q[1] + w[2] * q[2]) / (w[0] + w[1] + w[2])


class Flow:
    """special-relativistic Euler (Gamma = 2) on the periodic grid, [5][z][y][x]"""

    def __init__(self):
        self.p = None

    @staticmethod
    def conserved(P):
        rho, v, p = P[0], P[1:4], P[4]
        W2 = 1 / (1 - (v ** 2).sum(0))
        q = (rho + 2 * p) * W2
        D = rho * W2.sqrt()
        return torch.cat([D[None], q * v, (q - p - D)[None]])

    def primitives(self, U):
        D, S, E = U[0], U[1:4], U[4] + U[0]
        S2 = (S ** 2).sum(0)
        p = self.p if self.p is not None else 0.5 * E
        for _ in range(30):
            v2 = S2 / (E + p) ** 2
            W = 1 / torch.sqrt(1 - v2)
            f = E - S2 / (E + p) - D / W - p
            df = v2 * (1 - D * W / (E + p)) - 1
            new = p - f / df
            new = torch.where(new > 0, new, 0.5 * p)
            done = bool(((new - p).abs() <= 1e-15 * new).all())
            p = new
            if done:
                break
        self.p = p
        v = S / (E + p)
        return torch.cat([(D * torch.sqrt(1 - (v ** 2).sum(0)))[None], v, p[None]])

    @staticmethod
    def _flux(P, d):
        rho, v, p = P[0], P[1:4], P[4]
        U = Flow.conserved(P)
        F = U * v[d]
        F[1 + d] += p
        F[4] += p * v[d]
        v2 = (v ** 2).sum(0)
        cs2 = 2 * p / (rho + 2 * p)
        root = torch.sqrt(cs2 * (1 - v2) * (1 - v2 * cs2 - v[d] ** 2 * (1 - cs2)))
        den = 1 - v2 * cs2
        a = v[d] * (1 - cs2)
        return F, U, torch.maximum(((a - root) / den).abs(), ((a + root) / den).abs())

    def rhs(self, U, t):
        P = self.primitives(U)
        r = torch.zeros_like(U)
        for d in range(3):
            ax = -1 - d
            at = [torch.roll(P, -k, ax) for k in range(-2, 4)]
            L, R = _weno5(5, *at[:5]), _weno5(5, *at[:0:-1])
            for s, cell in ((L, at[2]), (R, at[3])):
                bad = ~((s[0] > 0) & (s[4] > 0) & ((s[1:4] ** 2).sum(0) < 1))
                s.copy_(torch.where(bad, cell, s))
            FL, UL, aL = self._flux(L, d)
            FR, UR, aR = self._flux(R, d)
            F = 0.5 * (FL + FR - torch.maximum(aL, aR) * (UR - UL))
            r -= F - torch.roll(F, 1, ax)
        return r


def exact(c, seed):
    if c["what"] == "grid":
        if c["n"] ** 3 * c["steps"] * STAGES[c["method"]] > 8e8:
            return None      # over 20 seconds
        P = _flow_data(c["n"], seed)
        fl = Flow()
        u = fl.conserved(P)
        for _ in range(c["steps"]):
            u = _rk(c["method"], fl.rhs, u, 0.0, 0.25)
        return u.reshape(-1).cpu().numpy()
    W = Wave(c)
    x = torch.empty(3, W.F.nnodes, dtype=torch.float64, device=DEV)
    for G in W.groups:
        x[:, G["idx"]] = G["xyz"].reshape(*G["idx"].shape, 3).movedim(-1, 0)
    u = _mesh_input(c, W.F, seed, x).reshape(5, -1)
    dt = _dt(c, W.F)
    if c["steps"] == 0:
        return W.rhs(u, 0.0).reshape(-1)
    if c["what"] != "adjoint":
        rows = []
        psi0 = u[4]
        for k in range(c["steps"]):
            u = W.step(u, k * dt, dt)
            if c["what"] == "grad" and ((k + 1) % 16 == 0 or k + 1 == c["steps"]):
                rows.append(u.reshape(-1))
        if c["what"] == "steps":
            return u.reshape(-1)
        on = torch.zeros(W.F.nnodes, dtype=torch.bool, device=DEV)
        seen = torch.zeros(W.npts, dtype=torch.bool, device=DEV)
        for pt, _, _ in W.sources:
            seen[pt] = True
        for G in W.groups:
            n, E = G["n"], len(G["el"])
            out = ~seen[G["base"]:G["base"] + 6 * n * n * E].reshape(E, 6, n, n)
            node = G["idx"].reshape(E, n, n, n)
            for f in range(6):
                on[W._face(node, f // 2, f % 2)[out[:, f]]] = True
        lam = torch.zeros_like(u)
        lam[4] = torch.where(on, 2 * (u[4] - (0.5 * psi0 + 0.01)), torch.zeros_like(psi0))
    else:
        lam = u
    zero = torch.zeros_like(lam).requires_grad_(True)
    for _ in range(c["steps"]):   # the step is linear: its transpose does not depend on the state
        lam = torch.autograd.grad(W.step(zero, 0.0, dt), zero, lam)[0]
    return (torch.stack(rows), lam.reshape(-1)) if c["what"] == "grad" else lam.reshape(-1)
