"""The dissection solve and the PCG on meshes that are no rectangle
(tests/odd_meshes.py) against the oracle: fronts that take contributions from
more than four parts, elements that share their centre, islands, a node that eight elements hold."""
import numpy as np
import pytest

from odd_meshes import apart, fan, twice_round, winding_ring

pytestmark = pytest.mark.gpu

MESHES = {  # mesh, modes, dissection
    "fan_of_ten": (lambda: fan(10, 2, 8), 32, True),
    "fan_of_24": (lambda: fan(24, 2, 4), 32, True),
    "uneven_fan": (lambda: fan(7, 6, 5, even=False), 8, True),
    "ring_twice_round": (lambda: winding_ring(16, 4, 6), 8, True),
    "twice_round_a_node": (lambda: twice_round(4, 6), 8, True),
    "two_islands": (lambda: apart(2, 8, 6), 16, True),
    "four_islands": (lambda: apart(4, 3, 9), 32, False),
}


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _problem(m, nz):
    rng = np.random.default_rng(m.nel)
    F = np.zeros((nz, m.plane_size))
    lines = np.zeros((nz, m.nbound * m.np))
    for k in range(nz):
        if k == 1:
            continue
        F[k, :m.nel * m.npnp] = rng.standard_normal(m.nel * m.npnp)
        for b in range(m.nbound):
            xs, ys = m.side_xy(b)
            lines[k, b * m.np:(b + 1) * m.np] = np.cos(xs + 0.1 * k) + ys
    return F, lines


@pytest.mark.parametrize("name", list(MESHES))
def test_direct_solve_matches_oracle(torch_cuda, oracle, name):
    import torch
    from oracle.oracle import OracleMesh, OracleMsys
    from semtex_amd.solver import Field, GpuMesh, ModalMatrixSys
    print("case:", name, flush=True)
    make, modes, dissection = MESHES[name]
    m, nz = make(), 2 * modes
    F, lines = _problem(m, nz)
    gm = GpuMesh(m)
    M = ModalMatrixSys(0.7, 1.0, 0, modes, gm)
    u = Field(gm, nz)
    u.lines.copy_(torch.from_numpy(lines))
    u.solve(torch.from_numpy(F).cuda(), M)
    torch.cuda.synchronize()
    assert (M.layout()["kernel"] == 4) == dissection, M.layout()
    om, n = OracleMesh(m), m.nel * m.npnp
    for k in (0, 2, 3, nz - 1):
        uo = OracleMsys(om, 0.7, float(k >> 1) ** 2).solve_plane(F[k, :n], lines[k])
        assert np.linalg.norm(u.data[k, :n].cpu().numpy() - uo) < 1e-12 * np.linalg.norm(uo), k


# A thread of the PCG's plane kernel keeps 2, 4 or 8 values in registers, or
# the plane stays in memory: planes just past 1, 2, 4 and 8 times its 1,024
# threads
@pytest.mark.parametrize("points,shape", [(1026, (9, 3, 7)), (2050, (10, 8, 6)),
                                          (4104, (9, 7, 9)), (8208, (18, 7, 9))])
def test_pcg_matches_oracle(torch_cuda, oracle, points, shape):
    """Solution and largest iteration count against the oracle's JACPCG at
    the bars of test_gpu_pcg.py for a tolerance of 1e-12."""
    import torch
    from oracle.oracle import OracleMesh, OracleMsys
    from semtex_amd.mesh import rect_mesh
    from semtex_amd.solver import SX_JACPCG, Field, GpuMesh, ModalMatrixSys
    print("case: pcg", points, flush=True)
    m = rect_mesh(*shape, 0.0, 2 * np.pi, -1.0, 1.0, bc=("D", "N", "N", "N"), periodic_x=True)
    assert m.nglobal + m.nel * m.nint == points
    nz, lam2 = 4, 500.0
    F, lines = _problem(m, nz)
    gm = GpuMesh(m)
    M = ModalMatrixSys(lam2, 1.0, 0, nz // 2, gm, precision=SX_JACPCG)
    u = Field(gm, nz)
    u.lines.copy_(torch.from_numpy(lines))
    u.solve(torch.from_numpy(F).cuda(), M, tol_rel=1e-12, step_max=800)
    torch.cuda.synchronize()
    om, n, its = OracleMesh(m), m.nel * m.npnp, []
    for k in (0, 2, 3):
        S = OracleMsys(om, lam2, float(k >> 1) ** 2)
        uo, it = S.solve_plane_pcg(F[k, :n], lines[k], np.zeros(n), 1e-12, 800)
        its.append(it)
        got = u.data[k, :n].cpu().numpy()
        assert np.linalg.norm(got - uo) < 1e-10 * np.linalg.norm(uo), k
    assert 0 < max(its) < 799 and abs(u.last_iters - max(its)) <= 2, (u.last_iters, its)


@pytest.mark.parametrize("n,np_", [(2, 5), (4, 6), (5, 7), (6, 7)])
def test_pcg_first_iterations_with_eight_elements_at_a_node(torch_cuda, oracle, n, np_):
    """The gather past its four loads with two, four and eight values a thread
    and through memory: five iterations, which neither run ends before
    (tolerance 0, step_max 6), so the iterates differ by rounding only -- five
    times sums of up to 10,657 terms, some 1e-14 each, held to 1e-11.  (On
    rectangles: the preconditioner keeps the reference's diagonal, which is
    not positive on skewed elements and carries its rounding far there.)"""
    import torch
    from oracle.oracle import OracleMesh, OracleMsys
    from semtex_amd.solver import SX_JACPCG, Field, GpuMesh, ModalMatrixSys
    print("case: pcg twice round", n, np_, flush=True)
    m, nz, lam2 = twice_round(n, np_), 4, 500.0
    F, lines = _problem(m, nz)
    gm = GpuMesh(m)
    M = ModalMatrixSys(lam2, 1.0, 0, nz // 2, gm, precision=SX_JACPCG)
    u = Field(gm, nz)
    u.lines.copy_(torch.from_numpy(lines))
    u.solve(torch.from_numpy(F).cuda(), M, tol_rel=0.0, step_max=6)
    torch.cuda.synchronize()
    om, npt = OracleMesh(m), m.nel * m.npnp
    for k in (0, 2, 3):
        S = OracleMsys(om, lam2, float(k >> 1) ** 2)
        uo, it = S.solve_plane_pcg(F[k, :npt], lines[k], np.zeros(npt), 0.0, 6)
        assert u.last_iters == 5 and it == 6           # the oracle counts the step it did not take
        got = u.data[k, :npt].cpu().numpy()
        assert np.linalg.norm(got - uo) < 1e-11 * np.linalg.norm(uo), k
