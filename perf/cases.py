"""The work a user of this framework has it do, as measured cases.

Every case goes through the public entry points (semtex_amd.solver): the
per-Fourier-mode Helmholtz solve in its precisions and boundary conditions,
the set-up of new systems, the gradient through a solve, an uneven batch of
independent problems, and the DNS time step.  Sizes are those of this
repository's configurations and tests, or generic ones beside them.

  listed()            the measured cases
  draw(rng)           one more case of the same ranges
  prepare(case, seed) inputs from the seed, and the systems a program keeps
  run(state)          one pass, its outputs whole
  work(case)          bytes and operations no implementation can avoid
  exact(case, seed)   the outputs in 64 bits by plain torch (separable
                      tensor-product solve), without the framework
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from semtex_amd.mesh import edgemaps, rect_mesh
from semtex_amd.solver import (DNS, SX_ALTSKEW, SX_FP64, SX_JACPCG, SX_MIXED, SX_SKEW, Batch,
                               Field, GpuMesh, ModalMatrixSys, helmholtz_solve, mass_weight)

PRECISION = {"fp64": SX_FP64, "mixed": SX_MIXED, "pcg": SX_JACPCG}
LX, Y0, Y1 = 2 * math.pi, -1.0, 1.0


def listed():
    return [
        # one small 2D elliptic solve (the plain 4x4 N_P=8 configuration):
        # the smallest call, all launch and dependency latency
        dict(name="helmholtz_2d_4x4", kind="helmholtz", nx=4, ny=4, np=8, nz=1, lam2=1.0,
             periodic=False, bc="DDDD", lines=False, precision="fp64"),
        # the batched 2.5D solve over all Fourier modes (the main benchmark)
        dict(name="helmholtz_16x16_nz64", kind="helmholtz", nx=16, ny=16, np=10, nz=64, lam2=1.0,
             periodic=True, bc="DNDN", lines=False, precision="fp64"),
        # an ordinary odd-sized problem: no periodicity, walls with given
        # values, natural sides with given fluxes, an odd number of modes
        dict(name="helmholtz_9x7_nz18", kind="helmholtz", nx=9, ny=7, np=7, nz=18, lam2=2.5,
             periodic=False, bc="DNND", lines=True, precision="fp64"),
        # one large plane: a 2D problem on a fine mesh (wide band)
        dict(name="helmholtz_2d_48x40", kind="helmholtz", nx=48, ny=40, np=9, nz=1, lam2=0.5,
             periodic=False, bc="DDDN", lines=True, precision="fp64"),
        # the mixed-precision option: FP32 element work, FP64 refinement
        dict(name="helmholtz_mixed_12x9_nz32", kind="helmholtz", nx=12, ny=9, np=9, nz=32,
             lam2=1.0, periodic=True, bc="DNDN", lines=False, precision="mixed"),
        # the iterative option (ITERATIVE sessions, start-up steps): Jacobi-PCG
        dict(name="helmholtz_pcg_6x8_nz16", kind="helmholtz", nx=6, ny=8, np=8, nz=16, lam2=500.0,
             periodic=True, bc="DNDN", lines=True, precision="pcg"),
        # new constants: systems built, factorised and used once (a changed
        # time step or lambda2, a parameter sweep)
        dict(name="new_system_12x10_nz32", kind="new_system", nx=12, ny=10, np=8, nz=32, lam2=3.0,
             periodic=True, bc="DNDN", lines=False, precision="fp64"),
        # the gradient of a misfit through the batched solve, with respect to
        # the forcing and lambda2 (forward and adjoint solve)
        dict(name="gradient_16x16_nz32", kind="gradient", nx=16, ny=16, np=10, nz=32, lam2=1.0,
             periodic=True, bc="DNDN", lines=False, precision="fp64"),
        # many independent uneven 2D problems in one graph launch, half of
        # them cylindrical
        dict(name="batch_64", kind="batch", count=64, sizes=20261202, small=4, large=20),
        # the DNS channel of the benchmark: restart from a state, a few steps
        dict(name="dns_channel_12x24_nz128", kind="dns", nx=12, ny=24, np=8, nz=128, steps=5,
             advection="skew", dealias=False, nord=2),
        # a small 2D DNS (two components, one plane): launches count
        dict(name="dns_2d_8x6", kind="dns", nx=8, ny=6, np=9, nz=1, steps=20,
             advection="altskew", dealias=False, nord=2),
        # dealiased products, a number of planes that is no power of two,
        # third-order time stepping
        dict(name="dns_dealias_8x10_nz48", kind="dns", nx=8, ny=10, np=7, nz=48, steps=5,
             advection="skew", dealias=True, nord=3),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _planes(rng, hi):
    n = _log_int(rng, 1, hi)
    return 1 if n == 1 else 2 * max(1, n // 2)


def draw(rng):
    """Kinds by how often a program meets them; sizes log-uniform over the
    listed ranges (odd ones among them), the points of a case no more than
    the largest listed one of its kind holds."""
    u = rng.random()
    if u < 0.07:
        return dict(kind="batch", count=rng.randint(9, 64), sizes=rng.randint(1, 10 ** 6),
                    small=4, large=rng.randint(8, 20))
    while True:
        nx, ny, np_ = _log_int(rng, 2, 28), _log_int(rng, 2, 28), rng.randint(4, 12)
        if u < 0.33:
            nz = _planes(rng, 96)
            if nx * ny * np_ * np_ * max(nz, 4) > 6e5:
                continue
            dealias = nz >= 4 and nz % 4 == 0 and rng.random() < 0.3
            return dict(kind="dns", nx=nx, ny=ny, np=np_, nz=nz, steps=rng.randint(2, 6),
                        advection="altskew" if not dealias and rng.random() < 0.4 else "skew",
                        dealias=dealias, nord=rng.choice([1, 2, 2, 3]))
        nz = _planes(rng, 80)
        points = nx * ny * np_ * np_ * nz
        if points > 1.2e6 or (u > 0.72 and points > 3e5):
            continue
        if u < 0.72:
            kind, precision = "helmholtz", "fp64"
        else:
            kind, precision = rng.choice([("helmholtz", "mixed"), ("helmholtz", "pcg"),
                                          ("new_system", "fp64"), ("new_system", "fp64"),
                                          ("gradient", "fp64")])
        periodic = kind == "gradient" or rng.random() < 0.5
        bc = rng.choice(["DNDN", "DNNN", "NNDN"] if periodic
                        else ["DDDD", "DNND", "NDNN", "DNDN", "NNND"])
        lam2 = round(10 ** (rng.uniform(2, 3) if precision == "pcg" else rng.uniform(-2, 2)), 6)
        return dict(kind=kind, nx=nx, ny=ny, np=np_, nz=nz, lam2=lam2, periodic=periodic, bc=bc,
                    lines=kind == "helmholtz" and rng.random() < 0.6, precision=precision)


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _mesh(nx, ny, np_, x1, y0, y1, bc, periodic, cyl=0, x0=0.0):
    """The mesh and numbering a session holds (a program reads it once)."""
    return rect_mesh(nx, ny, np_, x0, x1, y0, y1, bc=tuple(bc), periodic_x=periodic, cyl=cyl)


def _case_mesh(c):
    return _mesh(c["nx"], c["ny"], c["np"], LX, Y0, Y1, c["bc"], c["periodic"])


def _points(c):
    return c["nx"] * c["ny"] * c["np"] ** 2


def _forcing(c, seed):
    """[nz][nel*np*np], N(0,1) falling with the mode as (1+k)^-2, the
    Nyquist plane (never solved) zero."""
    n, nz = _points(c), c["nz"]
    f = np.random.default_rng([seed, 1]).standard_normal((nz, n))
    f *= (1.0 + (np.arange(nz) >> 1))[:, None] ** -2.0
    if nz > 1:
        f[1] = 0.0
    return f


def _side_value(k, x, y, seed):
    """Smooth boundary data of plane k at (x, y), periodic in x over LX."""
    a, b, p, q = np.random.default_rng([seed, 2, k]).uniform(-1, 1, 4)
    s = 1.0 / (1.0 + (k >> 1)) ** 2
    return s * (a * np.cos((1 + k % 3) * x + 3 * p) + b * np.sin(y + q))


def _boundary_lines(mesh, nz, seed):
    out = np.zeros((nz, mesh.nbound * mesh.np))
    xy = [mesh.side_xy(b) for b in range(mesh.nbound)]
    x, y = np.concatenate([v[0] for v in xy]), np.concatenate([v[1] for v in xy])
    for k in range(nz):
        if k != 1:
            out[k] = _side_value(k, x, y, seed)
    return out


def _padded(a, stride):
    t = torch.zeros(a.shape[:-1] + (stride,), dtype=torch.float64)
    t[..., :a.shape[-1]] = torch.from_numpy(np.ascontiguousarray(a))
    return t.cuda()


def _batch_problems(c):
    """N_P 4..12, `small`..`large` elements a side, aspect 1..4, lambda2
    1e-2..1e2; the second half cylindrical with the axis on y = 0."""
    rng = np.random.default_rng(c["sizes"])
    out = []
    for i in range(c["count"]):
        np_ = int(rng.integers(4, 13))
        nx, ny = (int(v) for v in rng.integers(c["small"], c["large"] + 1, 2))
        a, lam2 = float(rng.uniform(1.0, 4.0)), float(10.0 ** rng.uniform(-2.0, 2.0))
        cyl = int(i >= c["count"] // 2)
        out.append(dict(nx=nx, ny=ny, np=np_, x1=a, lam2=lam2, cyl=cyl,
                        bc="ANDN" if cyl else "DDDD"))
    return out


def _batch_forcing(mesh_y, seed, i, cyl):
    f = np.random.default_rng([seed, 3, i]).standard_normal(mesh_y.shape)
    return f * mesh_y if cyl else f        # r-weighted, as cylindrical callers supply it


def _dns_state(mesh, ncom, nz, seed):
    """Poiseuille flow with a U(-1e-2, 1e-2) perturbation, single-valued on
    shared element-boundary nodes."""
    n = mesh.nel * mesh.npnp
    u = np.random.default_rng([seed, 4]).uniform(-1e-2, 1e-2, (ncom, nz, n))
    u[0] += 1.0 - mesh.y.ravel() ** 2
    em, _ = edgemaps(mesh.np)
    slot = np.arange(mesh.nel)[:, None] * mesh.npnp + em[:mesh.next][None, :]
    owner = np.zeros(mesh.nglobal, dtype=np.int64)
    owner[mesh.btog.ravel()] = slot.ravel()
    u[:, :, slot.ravel()] = u[:, :, owner[mesh.btog.ravel()]]
    return u


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "dns":
        mu = _mesh(c["nx"], c["ny"], c["np"], 2 * LX, Y0, Y1, "DNDN", True)
        mp = _mesh(c["nx"], c["ny"], c["np"], 2 * LX, Y0, Y1, "NNNN", True)
        gu, gp = GpuMesh(mu), GpuMesh(mp)
        d = DNS(gu, gp, c["nz"], 1.0, 1.0 / 2000.0, 1e-3, const_force=(1e-3, 0.0, 0.0),
                advection=SX_SKEW if c["advection"] == "skew" else SX_ALTSKEW, nord=c["nord"])
        if c["dealias"]:
            d.set_dealias(True)
        u0 = _padded(_dns_state(mu, d.ncom, c["nz"], seed), d.stride)
        return dict(kind=kind, dns=d, u0=u0, steps=c["steps"], keep=(gu, gp))
    if kind == "batch":
        items = []
        for i, p in enumerate(_batch_problems(c)):
            m = _mesh(p["nx"], p["ny"], p["np"], p["x1"], 0.0, 1.0, p["bc"], False, p["cyl"])
            gm = GpuMesh(m)
            items.append((ModalMatrixSys(p["lam2"], 0.0, 0, 1, gm), Field(gm, 1),
                          _padded(_batch_forcing(m.y, seed, i, p["cyl"]).reshape(1, -1),
                                  m.plane_size)))
        return dict(kind=kind, batch=Batch(items), fields=[u for _, u, _ in items])
    m = _case_mesh(c)
    gm = GpuMesh(m)
    modes = max(1, c["nz"] // 2)
    f = _padded(_forcing(c, seed), m.plane_size)
    st = dict(kind=kind, mesh=gm, f=f, lam2=c["lam2"], modes=modes)
    if kind == "gradient":
        target = np.random.default_rng([seed, 5]).standard_normal((c["nz"], _points(c))) * 1e-2
        st["target"] = _padded(target, m.plane_size)
        st["weight"] = mass_weight(gm, torch.ones_like(f), 1.0)
        return st
    st["u"] = Field(gm, c["nz"])
    if c["lines"]:
        st["u"].lines.copy_(torch.from_numpy(_boundary_lines(m, c["nz"], seed)))
    if kind == "helmholtz":
        st["work"] = torch.empty_like(f)
        st["pcg"] = c["precision"] == "pcg"
        st["sys"] = ModalMatrixSys(c["lam2"], 1.0, 0, modes, gm, PRECISION[c["precision"]])
    return st


def run(state):
    s, kind = state, state["kind"]
    if kind == "dns":
        d = s["dns"]
        d.set_state(s["u0"])
        d.step(s["steps"])
        return [d.field(i) for i in range(d.ncom + 1)]
    if kind == "batch":
        s["batch"].run()
        return [u.data for u in s["fields"]]
    if kind == "gradient":
        f = s["f"].detach().requires_grad_(True)
        lam2 = torch.tensor(s["lam2"], dtype=torch.float64, requires_grad=True)
        u = helmholtz_solve(f, lam2, s["mesh"], 1.0, s["modes"])
        d = u - s["target"]
        (0.5 * (d * d * s["weight"]).sum()).backward()
        return u.detach(), f.grad, lam2.grad
    if kind == "new_system":
        system = ModalMatrixSys(s["lam2"], 1.0, 0, s["modes"], s["mesh"])
        return s["u"].solve(s["f"].clone(), system).data
    s["work"].copy_(s["f"])                # the solve consumes its forcing
    if s["pcg"]:
        s["u"].data.zero_()                # the iteration's first guess
    return s["u"].solve(s["work"], s["sys"]).data


# --------------------------------------------------------------------------
# what no implementation can avoid
# --------------------------------------------------------------------------
def work(case):
    """Bytes: inputs read once, outputs written once (doubles).  Operations:
    the tensor-product contractions of the elements (2 np^3 each) that a
    solve or a step applies at least."""
    c, kind = case, case["kind"]
    if kind == "batch":
        ps = _batch_problems(c)
        return {"bytes": sum(16.0 * _points(p) for p in ps),
                "flops": sum(8.0 * _points(p) * p["np"] for p in ps)}
    pts, nz = _points(c), c["nz"]
    if kind == "dns":
        ncom = 2 if nz == 1 else 3
        # per step: u^n and the older levels of u and N in, u, N and p out
        fields = ncom * (2 + 2 * c["nord"] - 1) + 1
        step = 8.0 * fields * pts * nz
        ops = pts * nz * (2.0 * c["np"] * (8 * ncom + 4 + 4 * (ncom + 1)) +
                          (5.0 * 5 * ncom * math.log2(nz) if nz > 1 else 0.0))
        return {"bytes": c["steps"] * step, "flops": c["steps"] * ops}
    planes = nz - 1 if nz > 1 else 1
    one = dict(bytes=16.0 * pts * planes, flops=8.0 * pts * planes * c["np"])
    if kind == "gradient":      # forward solve (u out), adjoint solve (df out), the target in
        return {"bytes": 2 * one["bytes"] + 8.0 * pts * planes, "flops": 2 * one["flops"]}
    if kind == "new_system":    # and one element's condensation per mode
        nint, nb = (c["np"] - 2) ** 2, 4 * (c["np"] - 1)
        one["flops"] += max(1, nz // 2) * (nint ** 3 / 3.0 + 2.0 * nint * nint * nb)
    return one


# --------------------------------------------------------------------------
# exact values: the meshes are tensor products of two 1D grids, so the
# assembled operator is My x Kx + Ky x Mx + h My x Mx; diagonalised in x and
# y (cylindrical: My is 0 on the axis, so y is solved densely per x eigenvalue)
# --------------------------------------------------------------------------
def _gll(n):
    leg = np.polynomial.legendre
    c = np.zeros(n)
    c[-1] = 1.0
    z = np.concatenate([[-1.0], np.sort(leg.legroots(leg.legder(c)).real), [1.0]])
    for _ in range(3):          # Newton on P'_{n-1}
        d1, d2 = leg.legval(z, leg.legder(c)), leg.legval(z, leg.legder(c, 2))
        z[1:-1] -= d1[1:-1] / d2[1:-1]
    pn = leg.legval(z, c)
    w = 2.0 / (n * (n - 1) * pn ** 2)
    dz = z[:, None] - z[None, :] + np.eye(n)
    D = pn[:, None] / pn[None, :] / dz
    np.fill_diagonal(D, 0.0)
    np.fill_diagonal(D, -D.sum(axis=1))
    return z, w, D


class _Line:
    """A 1D grid of n equal elements on [a, b]: node indices and positions
    per element, assembled stiffness and mass, weighted by `radius`."""

    def __init__(self, n, np_, a, b, periodic=False, radius=False):
        z, w, D = _gll(np_)
        h = (b - a) / n
        self.idx = np.arange(n)[:, None] * (np_ - 1) + np.arange(np_)[None, :]
        self.size = n * (np_ - 1) + (0 if periodic else 1)
        self.idx %= self.size
        self.pos = a + h * (np.arange(n)[:, None] + 0.5 * (1.0 + z)[None, :])
        self.w = np.broadcast_to(w * h / 2, self.pos.shape)
        self.K = np.zeros((self.size, self.size))
        self.M = np.zeros(self.size)
        for e in range(n):
            r = self.pos[e] if radius else np.ones(np_)
            i = self.idx[e]
            self.K[np.ix_(i, i)] += D.T @ ((w * r)[:, None] * D) * (2.0 / h)
            np.add.at(self.M, i, w * r * h / 2)


class _Grid:
    def __init__(self, nx, ny, np_, x1, y0, y1, bc, periodic, cyl=0):
        self.X = _Line(nx, np_, 0.0, x1, periodic)
        self.Y = _Line(ny, np_, y0, y1, False, bool(cyl))
        fx, fy = np.ones(self.X.size, bool), np.ones(self.Y.size, bool)
        fy[0], fy[-1] = bc[0] != "D", bc[2] != "D"
        if not periodic:
            fx[-1], fx[0] = bc[1] != "D", bc[3] != "D"
        self.fx, self.fy, self.bc, self.periodic = fx, fy, bc, periodic
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev)
        # element (ey, ex), node (i, j) -> global row and column
        shape = (ny, nx, np_, np_)
        row = np.broadcast_to(self.Y.idx[:, None, :, None], shape).ravel()
        col = np.broadcast_to(self.X.idx[None, :, None, :], shape).ravel()
        self.at = self.t(row * self.X.size + col)
        self.q = self.t((self.Y.w[:, None, :, None] * self.X.w[None, :, None, :]).ravel())
        self.lx, self.Vx = self._modes(self.X, fx)
        self.cyl = cyl
        if cyl:
            self.Ky, self.My = self.t(self.Y.K[np.ix_(fy, fy)]), self.t(self.Y.M[fy])
        else:
            self.ly, self.Vy = self._modes(self.Y, fy)

    def _modes(self, line, free):
        r = np.sqrt(line.M[free])
        lam, V = np.linalg.eigh(line.K[np.ix_(free, free)] / (r[:, None] * r[None, :]))
        return self.t(lam), self.t(V / r[:, None])

    def gather(self, g):                   # [planes][Ny][Nx] -> element nodes
        return g.reshape(g.shape[0], -1)[:, self.at]

    def assemble(self, w):                 # element nodes -> [planes][Ny][Nx]
        g = torch.zeros(w.shape[0], self.Y.size * self.X.size, dtype=torch.float64,
                        device=self.at.device)
        g.index_add_(1, self.at, w)
        return g.reshape(-1, self.Y.size, self.X.size)

    def solve(self, rhs, h, value=None):
        """A u = rhs per plane with constants h [planes]; u = value on the
        Dirichlet sides."""
        u = torch.zeros_like(rhs) if value is None else value.clone()
        fx, fy = self.t(np.flatnonzero(self.fx)), self.t(np.flatnonzero(self.fy))
        mx, my = self.t(self.X.M), self.t(self.Y.M)
        u[:, fy[:, None], fx[None, :]] = 0.0
        if value is not None:
            Kx, Ky = self.t(self.X.K), self.t(self.Y.K)
            rhs = rhs - ((u @ Kx) * my[:, None] + (Ky @ u) * mx +
                         h[:, None, None] * u * my[:, None] * mx)
        b = rhs[:, fy[:, None], fx[None, :]]
        if self.cyl:
            b = (b @ self.Vx).cpu()
            s = (self.lx[None, :] + h[:, None])[..., None]
            A = (self.Ky + torch.diag_embed(s * self.My)).cpu()
            x = torch.linalg.solve(A, b.transpose(1, 2).unsqueeze(-1)).squeeze(-1)
            x = x.transpose(1, 2).to(rhs.device)
        else:
            x = self.Vy.T @ b @ self.Vx
            x = self.Vy @ (x / (self.ly[:, None] + self.lx + h[:, None, None]))
        u[:, fy[:, None], fx[None, :]] = x @ self.Vx.T
        return u

    def boundary(self, planes, seed):
        """Dirichlet values on the grid, natural fluxes as a right-hand side."""
        X, Y = self.X, self.Y
        px, py = np.zeros(X.size), np.zeros(Y.size)
        px[X.idx], py[Y.idx] = X.pos, Y.pos
        if self.periodic:
            px[0] = 0.0
        val = np.zeros((len(planes), Y.size, X.size))
        flux = np.zeros_like(val)
        for p, k in enumerate(planes):
            for s, r in ((0, 0), (2, Y.size - 1)):
                g = _side_value(k, px, np.full(X.size, py[r]), seed)
                if self.bc[s] == "D":
                    val[p, r] = g
                elif self.bc[s] == "N":
                    flux[p, r] += g * X.M
            for s, q in ((1, X.size - 1), (3, 0)) if not self.periodic else ():
                g = _side_value(k, np.full(Y.size, px[q]), py, seed)
                if self.bc[s] == "D":
                    val[p, :, q] = g
                elif self.bc[s] == "N":
                    flux[p, :, q] += g * Y.M
        return self.t(val), self.t(flux)


def exact(case, seed):
    """None for the DNS: many coupled solves, no short independent form."""
    c, kind = case, case["kind"]
    if kind == "dns":
        return None

    def padded(planes, nz, vals):
        n = vals.shape[1]
        out = torch.zeros(nz, n + (n & 1), dtype=torch.float64)
        out[planes, :n] = vals.cpu()
        return out

    if kind == "batch":
        res = []
        for i, p in enumerate(_batch_problems(c)):
            g = _Grid(p["nx"], p["ny"], p["np"], p["x1"], 0.0, 1.0, p["bc"], False, p["cyl"])
            y = np.broadcast_to(g.Y.pos[:, None, :, None],
                                (p["ny"], p["nx"], p["np"], p["np"])).reshape(p["nx"] * p["ny"], -1)
            f = g.t(_batch_forcing(y, seed, i, p["cyl"]).reshape(1, -1))
            u = g.solve(g.assemble(-g.q * f), g.t(np.array([p["lam2"]])))
            res.append(padded([0], 1, g.gather(u)))
        return res
    nz = c["nz"]
    planes = [k for k in range(nz) if nz == 1 or k != 1]
    g = _Grid(c["nx"], c["ny"], c["np"], LX, Y0, Y1, c["bc"], c["periodic"])
    h = g.t(c["lam2"] + np.array([(k >> 1) ** 2 for k in planes], dtype=float))
    f = g.t(_forcing(c, seed)[planes])
    rhs, value = g.assemble(-g.q * f), None
    if c["lines"]:
        value, flux = g.boundary(planes, seed)
        rhs = rhs + flux
    u = g.gather(g.solve(rhs, h, value))
    if kind != "gradient":
        return padded(planes, nz, u)
    target = g.t(np.random.default_rng([seed, 5]).standard_normal((nz, _points(c)))[planes] * 1e-2)
    adj = g.gather(g.solve(g.assemble(g.q * (u - target)), h))
    dlam2 = -(g.q * adj * u).sum().cpu()
    return padded(planes, nz, u), padded(planes, nz, -g.q * adj), dlam2
