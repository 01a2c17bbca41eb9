"""The dissection solve (layout kernel 4) against the oracle at the FP64 bar
(1e-12) and against the band solve of the same system, over the forms its
plan meets: one element and one row of elements (a single front), several
levels with and without shared classes (graded meshes), the smallest and
largest orders, periodic directions, every boundary kind, one mode and many,
a base mode, and a singular mode (pure Neumann, its last unknown dropped).
A mesh whose elements hold a node twice keeps the band solve.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _graded(n, a, b):
    t = np.linspace(0.0, 1.0, n + 1)
    return a + (b - a) * (0.6 * t + 0.4 * t ** 2)


CASES = {  # nx, ny, np, nz, bc, periodic_x, periodic_y, graded, lambda2, base mode
    "one_element": (1, 1, 6, 1, "NNDN", False, False, False, 1.0, 0),
    "one_row": (7, 1, 5, 2, "DNNN", False, False, False, 0.3, 0),
    "one_column": (1, 9, 4, 4, "DDNN", False, False, False, 0.3, 0),
    "lowest_order": (5, 6, 3, 4, "DNND", False, False, False, 1.0, 0),
    "two_periodic": (2, 3, 4, 4, "DNNN", True, False, False, 1.0, 0),
    "doubly_periodic": (5, 4, 5, 4, "NNNN", True, True, False, 2.0, 0),
    "graded_uneven": (11, 7, 6, 6, "DNNN", True, False, True, 0.5, 0),
    "graded_many_modes": (9, 10, 7, 40, "DNDN", True, False, True, 1.0, 0),
    "order_twelve": (6, 5, 12, 4, "DDDD", False, False, False, 5.0, 0),
    "order_fourteen": (4, 3, 14, 4, "DNDN", True, False, False, 5.0, 0),
    "many_levels": (24, 20, 7, 2, "DDDN", False, False, False, 0.5, 0),
    "base_mode": (8, 6, 6, 4, "DNNN", True, False, False, 0.5, 3),
    "natural": (10, 9, 6, 4, "NNNN", False, False, False, 0.1, 0),
}


def _problem(name):
    from semtex_amd.mesh import rect_mesh
    nx, ny, np_, nz, bc, px, py, graded, lam2, base = CASES[name]
    kw = dict(bc=tuple(bc), periodic_x=px, periodic_y=py)
    if graded:
        kw.update(xs=_graded(nx, 0.0, 2 * np.pi), ys=_graded(ny, -1.0, 1.0))
    m = rect_mesh(nx, ny, np_, 0.0, 2 * np.pi, -1.0, 1.0, **kw)
    rng = np.random.default_rng(nx * 100 + ny)
    planes = [k for k in range(nz) if nz == 1 or base or k != 1]
    F = np.zeros((nz, m.plane_size))
    lines = np.zeros((nz, m.nbound * np_))
    for k in planes:
        F[k, :m.nel * m.npnp] = rng.standard_normal(m.nel * m.npnp)
        for b in range(m.nbound):
            xs, ys = m.side_xy(b)
            lines[k, b * np_:(b + 1) * np_] = (np.cos((k + 1) * xs) + ys if m.bnd_kind[b] == 0
                                               else rng.standard_normal(np_))
    return m, nz, lam2, base, planes, F, lines


def _solve(torch, m, nz, lam2, base, F, lines):
    from semtex_amd.solver import Field, GpuMesh, ModalMatrixSys
    gm = GpuMesh(m)
    M = ModalMatrixSys(lam2, 1.0, base, max(1, nz // 2), gm)
    u = Field(gm, nz)
    if m.nbound:
        u.lines.copy_(torch.from_numpy(lines))
    u.solve(torch.from_numpy(F).cuda(), M)
    torch.cuda.synchronize()
    return u.data.cpu().numpy()[:, :m.nel * m.npnp], M.layout()["kernel"]


@pytest.mark.parametrize("name", list(CASES))
def test_tree_matches_oracle_and_band(torch_cuda, oracle, monkeypatch, name):
    from oracle.oracle import OracleMesh, OracleMsys
    print("case:", name, flush=True)
    m, nz, lam2, base, planes, F, lines = _problem(name)
    ug, kernel = _solve(torch_cuda, m, nz, lam2, base, F, lines)
    assert kernel == 4
    monkeypatch.setenv("SX_BAND_TWIST", "0")
    ub, kernel = _solve(torch_cuda, m, nz, lam2, base, F, lines)
    assert kernel != 4
    om = OracleMesh(m)
    for k in planes:
        S = OracleMsys(om, lam2, float(base + (k >> 1)) ** 2)
        uo = S.solve_plane(F[k, :ug.shape[1]], lines[k] if m.nbound else None)
        scale = np.linalg.norm(uo)
        assert np.linalg.norm(ug[k] - uo) / scale < TOL, (k, "oracle")
        assert np.linalg.norm(ug[k] - ub[k]) / scale < TOL, (k, "band")


@pytest.mark.parametrize("nx,ny,np_,nz", [(3, 2, 4, 1), (8, 10, 8, 8)])
def test_singular_mode_is_the_same_by_tree_and_band(torch_cuda, monkeypatch, nx, ny, np_, nz):
    """Pure Neumann, lambda2 = 0: both solves end on the exact solution of
    the assembled system (the refinement), so they agree to rounding."""
    from semtex_amd.mesh import rect_mesh
    print("case: singular", nx, ny, np_, nz, flush=True)
    m = rect_mesh(nx, ny, np_, 0.0, 2 * np.pi, -1.0, 1.0, bc=("N", "N", "N", "N"),
                  periodic_x=True)
    rng = np.random.default_rng(7)
    F = np.zeros((nz, m.plane_size))
    n = m.nel * m.npnp
    for k in range(nz):
        if k != 1:
            F[k, :n] = np.sin(m.x.ravel() * (1 + k)) * m.y.ravel() + (
                0.01 * rng.standard_normal(n) if k else 0.0)
    lines = np.zeros((nz, m.nbound * np_))
    ug, kernel = _solve(torch_cuda, m, nz, 0.0, 0, F, lines)
    assert kernel == 4
    monkeypatch.setenv("SX_BAND_TWIST", "0")
    ub, kernel = _solve(torch_cuda, m, nz, 0.0, 0, F, lines)
    assert kernel != 4
    for k in range(nz):
        if k != 1 or nz == 1:
            assert np.linalg.norm(ug[k] - ub[k]) < TOL * np.linalg.norm(ub[k]), k


def test_element_holding_a_node_twice_keeps_the_band(torch_cuda, oracle):
    from semtex_amd.mesh import rect_mesh
    print("case: one periodic column of elements", flush=True)
    m = rect_mesh(1, 3, 5, 0.0, 2.0, -1.0, 1.0, bc=("D", "N", "N", "N"), periodic_x=True)
    F = np.zeros((1, m.plane_size))
    F[0, :m.nel * m.npnp] = np.random.default_rng(3).standard_normal(m.nel * m.npnp)
    lines = np.zeros((1, m.nbound * m.np))
    ug, kernel = _solve(torch_cuda, m, 1, 1.0, 0, F, lines)
    assert kernel != 4
    uo = oracle.solve_modes(m, 1.0, 1.0, F[:, :m.nel * m.npnp], lines)[0]
    assert np.linalg.norm(ug[0] - uo) < TOL * np.linalg.norm(uo)


def test_captured_singular_solve_outlives_a_batch(torch_cuda):
    """A graph captured of a pure Neumann solve replays to the same solution
    after a batch has taken its system."""
    from semtex_amd.mesh import rect_mesh
    from semtex_amd.solver import Batch, Field, GpuMesh, ModalMatrixSys
    torch = torch_cuda
    print("case: captured singular solve, then a batch", flush=True)
    m = rect_mesh(4, 3, 6, 0.0, 2 * np.pi, -1.0, 1.0, bc=("N", "N", "N", "N"), periodic_x=True)
    F = np.zeros((1, m.plane_size))
    F[0, :m.nel * m.npnp] = np.sin(m.x.ravel()) * m.y.ravel()
    gm = GpuMesh(m)
    M = ModalMatrixSys(0.0, 1.0, 0, 1, gm)
    u, v = Field(gm, 1), Field(gm, 1)
    src = torch.tensor(F, device="cuda")
    f = src.clone()
    u.solve(f, M)
    torch.cuda.synchronize()
    expect = u.data.clone()
    f.copy_(src)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        u.solve(f, M)
    B = Batch([(M, v, src)])
    for _ in range(3):
        f.copy_(src)
        u.data.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.linalg.norm(u.data - expect) <= TOL * torch.linalg.norm(expect)
        B.run()
        torch.cuda.synchronize()
