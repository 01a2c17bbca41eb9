"""Systems of more than 32 modes, whose dissection is cut by another cost and
which solve by band sweeps where those are estimated faster: each route the
rule takes (the layout query names it) against the oracle at the FP64 bar
(1e-12), on the first and last modes, with more modes than workgroups a chip
holds and mode counts that end inside a group of eight."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# nx, ny, np, nz, graded, dissection
CASES = [(16, 12, 5, 90, False, True), (14, 16, 6, 134, True, True), (24, 20, 6, 260, False, True),
         (5, 5, 6, 256, False, False), (12, 10, 5, 530, True, False)]


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.mark.parametrize("nx,ny,np_,nz,graded,dissection", CASES)
def test_many_modes_match_oracle(torch_cuda, oracle, nx, ny, np_, nz, graded, dissection):
    import torch
    from oracle.oracle import OracleMesh, OracleMsys
    from semtex_amd.mesh import rect_mesh
    from semtex_amd.solver import Field, GpuMesh, ModalMatrixSys
    print("case: many modes", nx, ny, np_, nz, flush=True)
    t = lambda n: 0.6 * np.linspace(0, 1, n + 1) + 0.4 * np.linspace(0, 1, n + 1) ** 2
    kw = dict(xs=2 * np.pi * t(nx), ys=2 * t(ny) - 1) if graded else {}
    m = rect_mesh(nx, ny, np_, 0.0, 2 * np.pi, -1.0, 1.0, bc=("D", "N", "D", "N"),
                  periodic_x=True, **kw)
    n = m.nel * m.npnp
    rng = np.random.default_rng(nx + nz)
    F = np.zeros((nz, m.plane_size))
    F[:, :n] = rng.standard_normal((nz, n))
    lines = np.zeros((nz, max(m.nbound * np_, 1)))
    planes = [0, 2, 3, nz // 2, nz - 2, nz - 1]
    for k in planes:
        for b in range(m.nbound):
            xs, ys = m.side_xy(b)
            lines[k, b * np_:(b + 1) * np_] = np.cos((k + 1) * xs) + ys
    gm = GpuMesh(m)
    M = ModalMatrixSys(0.7, 1.0, 0, nz // 2, gm)
    u = Field(gm, nz)
    u.lines.copy_(torch.from_numpy(lines))
    u.solve(torch.from_numpy(F).cuda(), M)
    torch.cuda.synchronize()
    assert (M.layout()["kernel"] == 4) == dissection, M.layout()
    om = OracleMesh(m)
    for k in planes:
        uo = OracleMsys(om, 0.7, float(k >> 1) ** 2).solve_plane(F[k, :n], lines[k])
        got = u.data[k, :n].cpu().numpy()
        assert np.linalg.norm(got - uo) < 1e-12 * np.linalg.norm(uo), k
