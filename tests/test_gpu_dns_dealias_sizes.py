"""Dealiased products on k_zmat's edges -- planes whose 3/2 grid ends inside a
16-row block or past a staging chunk of 96 k rows, and the library products
kept past 128 planes -- against the oracle's dealiased step, velocity to the
FP64 DNS bar of test_gpu_dns.py (1e-11 after two steps)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.mark.parametrize("nz", [4, 12, 20, 44, 72, 128, 260])
def test_dealiased_step_at_plane_counts(torch_cuda, oracle, nz):
    import torch
    from oracle.dns_oracle import DnsOracle
    from semtex_amd.problems import dns_channel
    from semtex_amd.solver import DNS, SX_SKEW, GpuMesh
    print("case: dealiased channel 2x3 np=5 nz", nz, flush=True)
    P = dns_channel(nx=2, ny=3, np_=5, nz=nz, Re=100.0)
    mu = P["mesh_u"]
    n = mu.nel * mu.npnp
    D = DNS(GpuMesh(mu), GpuMesh(P["mesh_p"]), nz, P["beta"], P["kinvis"], P["dt"],
            const_force=P["const_force"], advection=SX_SKEW)
    D.set_dealias(True)
    O = DnsOracle(mu, P["mesh_p"], nz, P["beta"], P["kinvis"], P["dt"],
                  const_force=P["const_force"], advection="skew")
    O.dealias = True
    u0 = torch.zeros((3, nz, D.stride), dtype=torch.float64)
    u0[:, :, :n] = torch.from_numpy(P["u0"])
    D.set_state(u0.cuda())
    O.set_initial(P["u0"])
    planes = [k for k in range(nz) if k != 1]
    for _ in range(2):
        D.step(1)
        O.step()
    scale = max(np.linalg.norm(O.u[i][planes]) for i in range(3))
    for i in range(3):
        g = D.field(i).cpu().numpy()[planes, :n]
        assert np.linalg.norm(g - O.u[i][planes]) < 1e-11 * scale, i
