"""The own solves of systems a batch holds, and the batch itself, with a
singular mode (pure Neumann): the batch records the same dissection and
refinement as the system's own solves without split sweeps (equal bit for
bit), and every route ends on the exact solution of the assembled system, so
all agree with the solve before the batch was made to 1e-12.  A system whose
band layout has no split sweeps keeps the dissection for its own solves."""
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


@pytest.mark.parametrize("nx,ny,np_,band,fused", [(5, 4, 6, False, True), (16, 12, 8, False, True),
                                                  (16, 12, 8, False, False), (16, 12, 8, True, True)])
def test_singular_system_in_a_batch(torch_cuda, monkeypatch, nx, ny, np_, band, fused):
    import torch
    from semtex_amd.mesh import rect_mesh
    from semtex_amd.solver import Batch, Field, GpuMesh, ModalMatrixSys
    print("case: singular in a batch", nx, ny, np_, "band" if band else "dissection", fused, flush=True)
    m = rect_mesh(nx, ny, np_, 0.0, 2 * np.pi, -1.0, 1.0, bc=("N", "N", "N", "N"), periodic_x=True)
    F = np.zeros((1, m.plane_size))
    F[0, :m.nel * m.npnp] = np.sin(m.x.ravel()) * m.y.ravel()
    src = torch.tensor(F, device="cuda")
    gm = GpuMesh(m)
    if band:
        monkeypatch.setenv("SX_BAND_TWIST", "1")
    M = ModalMatrixSys(0.0, 1.0, 0, 1, gm)
    monkeypatch.delenv("SX_BAND_TWIST", raising=False)
    u, v = Field(gm, 1), Field(gm, 1)

    def own():
        u.data.zero_()
        u.solve(src.clone(), M)
        torch.cuda.synchronize()
        return u.data.clone(), M.layout()["kernel"]

    before, kernel = own()
    assert (kernel == 4) == (not band)
    if not fused:
        monkeypatch.setenv("SX_BATCH_FUSED", "0")
    B = Batch([(M, v, src)])
    assert B.info().startswith("fused=1" if fused else "fused=0")
    monkeypatch.setenv("SX_BAND_SPLIT", "0")
    same, _ = own()
    monkeypatch.delenv("SX_BAND_SPLIT")
    after, kernel = own()
    assert (kernel == 3) == (np_ == 8)             # the smaller mesh has no split sweeps
    near = lambda a, b: float(torch.linalg.norm(a - b) / torch.linalg.norm(b))
    assert near(same, before) < TOL and near(after, before) < TOL
    for rep in range(3):
        v.data.zero_()
        B.run()
        torch.cuda.synchronize()
        assert torch.equal(v.data, same), rep
