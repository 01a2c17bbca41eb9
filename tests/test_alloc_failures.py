"""Device allocations that fail, on the CPU: the library's host code runs on
tests/hip_stub.cpp (host memory for device memory, launches counted and not
run), which makes any chosen allocation fail.  A call that fails for memory
must leave the system it was given as it was -- the same plan, operators,
refinement and reserved right-hand sides -- hold no memory it did not hold
before, and succeed when it is called again with memory there."""
import os
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "hip_stub.cpp")
STUB = os.path.join(ROOT, "tests", "_bin", "libhip_stub.so")

PRELUDE = textwrap.dedent("""
    import ctypes as C, os, sys
    import numpy as np
    from semtex_amd import _lib
    from semtex_amd.mesh import rect_mesh
    from semtex_amd import solver
    solver._stream = lambda: None
    from semtex_amd.solver import GpuMesh, ModalMatrixSys
    L = _lib.load()
    S = C.CDLL(os.environ["LD_PRELOAD"])
    S.stub_bytes.restype = C.c_size_t
    S.stub_limit.argtypes = [C.c_size_t]
    for f in ("stub_allocs", "stub_live", "stub_launches", "stub_bad_pointers", "stub_freed"): getattr(S, f).restype = C.c_long
    S.stub_fail.argtypes = [C.c_long, C.c_long]
    S.stub_device.argtypes = [C.c_long]
    launches = lambda name: S.stub_launches(name.encode())

    class Buf:                       # a device array
        def __init__(self, n):
            self.p = C.c_void_p()
            assert S.hipMalloc(C.byref(self.p), C.c_size_t(8 * n)) == 0
            C.memset(self.p, 0, 8 * n)
        def free(self): S.hipFree(self.p)

    def reserve(M, nr): return L._ZN2sx16msys_reserve_rhsEP7sx_msysi(M.handle, nr)
    def solve_nr(M, nr): return L._ZN2sx10tree_solveEPK7sx_msysiP12ihipStream_t(M.handle, nr, None)

    def drain():                     # the blocks kept of earlier systems, given back
        S.stub_fail(0, 2)
        try: GpuMesh(rect_mesh(2, 2, 4))
        except _lib.SxError: pass
        S.stub_fail(-1, 0)

    class RawBatch:
        def __init__(self, Ms, nz=1):
            n = len(Ms)
            nz = [nz] * n if isinstance(nz, int) else nz
            self.bufs = [[Buf(z * M.gmesh.plane_size) for _ in range(3)] for M, z in zip(Ms, nz)]
            pp = lambda j: (C.c_void_p * n)(*[b[j].p for b in self.bufs])
            self.args = (n, (C.c_void_p * n)(*[M.handle for M in Ms]), (C.c_int * n)(*nz),
                         (C.c_int * n)(*[M.gmesh.plane_size for M in Ms]), pp(0), pp(1), pp(2), None, 1)
            self.h = None
        def create(self):
            h = C.c_void_p()
            rc = L.sx_batch_create(*self.args, C.byref(h))
            self.h = h if rc == 0 else None
            return rc
        def destroy(self):
            if self.h: L.sx_batch_destroy(self.h)
            self.h = None
        def free(self):
            for b in self.bufs:
                for x in b: x.free()

    def own_solve(M, nz=1):
        b = [Buf(nz * M.gmesh.plane_size) for _ in range(2)]
        rc = L.sx_field_solve(M.handle, nz, M.gmesh.plane_size, b[0].p, b[1].p, None, None)
        for x in b: x.free()
        return rc
""")


def run(body, **env):
    if not os.path.exists(STUB) or os.path.getmtime(STUB) < os.path.getmtime(SRC):
        os.makedirs(os.path.dirname(STUB), exist_ok=True)
        subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__",
                        "-I/opt/rocm/include", SRC, "-o", f"{STUB}.{os.getpid()}"], check=True)
        os.replace(f"{STUB}.{os.getpid()}", STUB)
    e = {k: v for k, v in os.environ.items() if not k.startswith("SX_")}
    e.update(LD_PRELOAD=STUB, PYTHONPATH=ROOT, **env)
    r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(body)], env=e, cwd=ROOT,
                       capture_output=True, text=True, timeout=240)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout[-2000:] + r.stderr[-4000:]


def test_failed_reservation_keeps_the_reserved_count():
    """msys_reserve_rhs: whichever allocation fails, a solve of more
    right-hand sides than the arrays hold is refused afterwards."""
    run("""
    m = rect_mesh(12, 10, 6, 0.0, 6.0, -1.0, 1.0, bc=("D", "N", "D", "N"), periodic_x=True)
    for bc in (("D", "N", "D", "N"), ("N", "N", "N", "N")):       # the second with a singular mode
        m = rect_mesh(12, 10, 6, 0.0, 6.0, -1.0, 1.0, bc=bc, periodic_x=True)
        M = ModalMatrixSys(0.0, 1.0, 0, 4, GpuMesh(m))
        assert M.layout()["operators"] > 0
        drain()
        k = 0
        while True:
            held = S.stub_bytes()
            S.stub_fail(k, 1)
            rc = reserve(M, 6)
            failed = S.stub_allocs() > k
            S.stub_fail(-1, 0)
            if not failed: break
            assert rc == _lib.SX_ERR_HIP, rc
            assert solve_nr(M, 6) == _lib.SX_ERR_ARG, k
            assert solve_nr(M, 2) == 0
            assert S.stub_bytes() == held, (k, S.stub_bytes(), held)
            k += 1
        assert rc == 0 and k >= 5, (rc, k)
        assert solve_nr(M, 6) == 0
    assert S.stub_bad_pointers() == 0
    print("ok")
    """)


@pytest.mark.parametrize("bc", ["DNDN", "NNNN"])
def test_failed_batch_leaves_its_systems_as_they_were(bc):
    """sx_batch_create over two systems: whichever allocation fails, both keep
    their own plan, operators and refinement and solve as before."""
    run(f"""
    ms = [rect_mesh(nx, ny, 6, 0.0, 6.0, -1.0, 1.0, bc=tuple("{bc}"), periodic_x=True)
          for nx, ny in ((16, 12), (9, 7))]
    Ms = [ModalMatrixSys(0.0, 1.0, 0, 1, GpuMesh(m)) for m in ms]
    B = RawBatch(Ms)
    keys = ("panels", "D", "twisted", "unit", "operators")
    def state():
        out = []
        for M in Ms:
            a, r = launches("k_tree_level"), launches("k_tree_residual")
            assert own_solve(M) == 0
            out.append((launches("k_tree_level") - a, launches("k_tree_residual") - r,
                        [M.layout()[k] for k in keys], M.layout()["kernel"]))
        return out
    was = state()
    # (plans and row lists stay with their meshes: made by a batch that works)
    Ms2 = [ModalMatrixSys(0.0, 1.0, 0, 1, M.gmesh) for M in Ms]
    B2 = RawBatch(Ms2)
    S.stub_fail(0, 0); assert B2.create() == 0
    total = S.stub_allocs()
    B2.destroy(); B2.free()
    del Ms2
    drain()
    assert [w[2][4] > 0 for w in was] == [True, True] and total > 4
    assert all(w[1] == ("{bc}" == "NNNN") for w in was)
    k = 0
    while True:
        held = S.stub_bytes()
        S.stub_fail(k, 1)
        rc = B.create()
        failed = S.stub_allocs() > k
        S.stub_fail(-1, 0)
        if not failed: break
        assert rc == _lib.SX_ERR_HIP, (k, rc, L.sx_last_error())
        assert S.stub_bytes() == held, (k, S.stub_bytes(), held)
        assert state() == was, (k, state(), was)
        k += 1
    assert rc == 0 and k > 4, (rc, k)
    B.destroy(); B.free()
    del Ms
    assert S.stub_live() == 0, S.stub_live()
    assert S.stub_bad_pointers() == 0
    print("ok")
    """)


def test_held_system_keeps_its_refinement_and_builds_a_band_only_when_asked():
    """A batch factorises no band for its systems and records the singular
    mode's refinement; a held system's own solves keep the refinement, run
    split band sweeps only where its layout has them, and the dissection where
    the band factor does not fit."""
    run("""
    def held(nx, ny, np_, bc, **kw):
        m = rect_mesh(nx, ny, np_, 0.0, 6.0, -1.0, 1.0, bc=tuple(bc), **kw)
        M = ModalMatrixSys(0.0, 1.0, 0, 1, GpuMesh(m))
        B = RawBatch([M])
        bands, res = launches("k_band_factor"), launches("FnTreeResidual")
        assert B.create() == 0
        assert launches("k_band_factor") == bands
        assert (launches("FnTreeResidual") > res) == (bc == "NNNN")
        return M, B
    # a layout with split sweeps, its mode singular
    M, B = held(16, 12, 8, "NNNN", periodic_x=True)
    r = launches("k_tree_residual")
    assert own_solve(M) == 0 and M.layout()["kernel"] == 3
    bands = launches("k_band_factor")
    assert bands > 0 and launches("k_tree_residual") == r + 1
    assert own_solve(M) == 0 and launches("k_band_factor") == bands
    B.destroy(); B.free(); del M, B
    # the band factor does not fit: the dissection, and nothing kept
    M, B = held(16, 12, 8, "NNNN", periodic_x=True)
    drain()
    bytes_, r = S.stub_bytes(), launches("k_tree_residual")
    b = [Buf(M.gmesh.plane_size) for _ in range(2)]
    S.stub_fail(0, 1 << 30)
    assert L.sx_field_solve(M.handle, 1, M.gmesh.plane_size, b[0].p, b[1].p, None, None) == 0
    S.stub_fail(-1, 0)
    for x in b: x.free()
    assert M.layout()["kernel"] == 4 and S.stub_bytes() == bytes_
    assert launches("k_tree_residual") == r + 1
    B.destroy(); B.free(); del M, B
    # a band past the panel sweeps
    M, B = held(48, 40, 9, "DDDN")
    assert M.layout()["nband"] > 513
    bands = launches("k_band_factor")
    assert own_solve(M) == 0 and M.layout()["kernel"] == 4
    assert launches("k_band_factor") == bands
    B.destroy(); B.free(); del M, B
    assert S.stub_live() == 0 and S.stub_bad_pointers() == 0
    print("ok")
    """)


def test_pcg_keeps_one_set_of_pinned_flags_a_device():
    """Solves that alternate between devices allocate no pinned memory after
    the first on each, and a solve whose events or buffer could not be made
    leaves nothing half made for the next."""
    run("""
    m = rect_mesh(6, 4, 6, 0.0, 6.0, -1.0, 1.0, bc=("D", "N", "D", "N"), periodic_x=True)
    M = []
    for d in (0, 1):
        S.stub_device(d)
        M.append(ModalMatrixSys(500.0, 1.0, 0, 2, GpuMesh(m), precision=_lib.SX_JACPCG))
    b = [Buf(4 * m.plane_size) for _ in range(2)]
    def pcg(i):
        S.stub_device(i)
        return L.sx_field_solve_pcg(M[i].handle, 4, m.plane_size, b[0].p, b[1].p, None, 1e-8, 20, None, None)
    S.stub_fail(0, 0); assert pcg(0) == 0
    n = S.stub_allocs()                                   # workspace, flags
    for k in range(n):
        S.stub_fail(k, 1); rc = pcg(1); S.stub_fail(-1, 0)
        assert rc == _lib.SX_ERR_HIP and L.sx_last_error()
    assert pcg(1) == 0
    S.stub_fail(-1, 0)
    for i in (0, 1, 0, 1, 1, 0): assert pcg(i) == 0
    assert S.stub_allocs() == 0
    print("ok")
    """)


def test_system_whose_dissection_does_not_fit_solves_by_band():
    """With memory for the band but not for the operators and fronts of a mesh
    graded both ways, the system is made and solves by band sweeps."""
    run("""
    t = lambda n: 0.6 * np.linspace(0, 1, n + 1) + 0.4 * np.linspace(0, 1, n + 1) ** 2
    m = rect_mesh(16, 16, 6, 0.0, 6.0, -1.0, 1.0, bc=("D", "N", "D", "N"), periodic_x=True,
                  xs=6 * t(16), ys=t(16))
    g = GpuMesh(m)
    M = ModalMatrixSys(1.0, 1.0, 0, 16, g)
    ops = M.layout()["operators"] * 16 * 8
    assert ops > 0
    del M
    drain()
    own = S.stub_bytes()
    hi, lo = own + 4 * ops, own
    while hi - lo > 1 << 20:                  # the least memory a system is made in
        mid = (lo + hi) // 2
        S.stub_limit(mid)
        try:
            M = ModalMatrixSys(1.0, 1.0, 0, 16, g)
            hi, kernel = mid, M.layout()["operators"]
            del M
        except _lib.SxError:
            lo = mid
        S.stub_limit(0)
        drain()
    assert kernel == 0
    S.stub_limit(hi)
    M = ModalMatrixSys(1.0, 1.0, 0, 16, g)
    S.stub_limit(0)
    assert own_solve(M, 32) == 0 and M.layout()["kernel"] in (1, 2, 3)
    del M, g
    assert S.stub_live() == 0 and S.stub_bad_pointers() == 0
    print("ok")
    """)


def test_kept_blocks_make_room_for_any_allocation():
    """Blocks kept of systems that went are given back when an allocation that
    is not a system's block (a mesh, FP32 operators, a solve's workspace)
    does not fit beside them."""
    run("""
    big = rect_mesh(16, 12, 8, 0.0, 6.0, -1.0, 1.0, bc=("D", "N", "D", "N"), periodic_x=True)
    g = GpuMesh(big)
    empty = S.stub_bytes()
    M = ModalMatrixSys(1.0, 1.0, 0, 8, g); del M
    kept = S.stub_bytes() - empty
    assert kept > 1 << 20
    S.stub_limit(S.stub_bytes() + 1000)
    g2 = GpuMesh(rect_mesh(8, 6, 6, bc=("D", "N", "D", "N")))
    S.stub_limit(0)
    assert S.stub_bytes() < empty + kept
    del g, g2
    assert S.stub_live() == 0
    print("ok")
    """)


def test_block_that_may_be_in_use_is_not_kept():
    """A system destroyed while the device cannot be waited for (during a
    capture) gives its block back instead of handing it to the next system."""
    run("""
    g = GpuMesh(rect_mesh(8, 6, 6, bc=("D", "N", "D", "N")))
    M = ModalMatrixSys(1.0, 1.0, 0, 4, g)
    drain()
    held = S.stub_bytes()
    S.stub_sync_fails(1); del M; S.stub_sync_fails(0)
    after = S.stub_bytes()
    drain()
    assert after < held and S.stub_bytes() == after       # nothing of it was kept
    M = ModalMatrixSys(1.0, 1.0, 0, 4, g)
    assert own_solve(M, 8) == 0                           # and no error was left behind
    del M, g
    assert S.stub_live() == 0
    print("ok")
    """)


def test_noalloc_solve_of_a_held_system_allocates_nothing():
    """sx_field_solve_mixed_noalloc on a system a batch holds, before any
    other solve of it: no allocation, the dissection."""
    run("""
    g = GpuMesh(rect_mesh(16, 12, 8, 0.0, 6.0, -1.0, 1.0, bc=("D", "N", "D", "N"), periodic_x=True))
    M = ModalMatrixSys(1.0, 1.0, 0, 1, g, precision=_lib.SX_MIXED)
    B = RawBatch([M])
    assert B.create() == 0
    b = [Buf(M.gmesh.plane_size) for _ in range(2)]
    S.stub_fail(0, 0)
    it = C.c_int()
    assert L.sx_field_solve_mixed_noalloc(M.handle, 1, M.gmesh.plane_size, b[0].p, b[1].p, None, 1e-6, 2,
                                          C.byref(it), None) == 0
    assert S.stub_allocs() == 0 and M.layout()["kernel"] == 4
    assert L.sx_field_solve_mixed(M.handle, 1, M.gmesh.plane_size, b[0].p, b[1].p, None, 1e-6, 2,
                                  C.byref(it), None) == 0
    assert M.layout()["kernel"] == 3
    print("ok")
    """)


@pytest.mark.parametrize("fused", ["1", "0"])
def test_mixed_batch_keeps_the_workspace_its_graph_records(fused):
    """Problems of one mixed system with different plane counts, and a later
    solve of more planes on it: no workspace that the graph holds is freed."""
    run(f"""
    os.environ["SX_BATCH_FUSED"] = "{fused}"
    g = GpuMesh(rect_mesh(6, 4, 6, 0.0, 6.0, -1.0, 1.0, bc=("D", "N", "D", "N"), periodic_x=True))
    freed = []
    for nz in ([2, 8], [8, 2]):
        M = ModalMatrixSys(1.0, 1.0, 0, 4, g, precision=_lib.SX_MIXED)
        B = RawBatch([M, M], nz)
        n = S.stub_freed()
        assert B.create() == 0
        freed.append(S.stub_freed() - n)
        b = [Buf(8 * M.gmesh.plane_size) for _ in range(2)]
        n = S.stub_freed()
        assert L.sx_field_solve_mixed(M.handle, 8, M.gmesh.plane_size, b[0].p, b[1].p, None, 1e-6, 2,
                                      None, None) == 0
        assert S.stub_freed() == n
        for x in b: x.free()
        B.destroy(); B.free(); del M, B
    assert freed[0] == freed[1], freed
    del g
    assert S.stub_live() == 0, S.stub_live()
    print("ok")
    """)


def test_batch_keeps_the_systems_cut_when_its_own_does_not_factor():
    """A pivot that the batch's cut finds not positive leaves the system on the
    cut it was made with; a new system still fails for it."""
    run("""
    g = GpuMesh(rect_mesh(16, 12, 6, 0.0, 6.0, -1.0, 1.0, bc=("D", "N", "D", "N"), periodic_x=True))
    M, M2 = [ModalMatrixSys(1.0, 1.0, 0, 1, g) for _ in range(2)]
    ops = M.layout()["operators"]
    B, B2 = RawBatch([M]), RawBatch([M2])
    S.stub_bad_pivots(1)
    assert B.create() == 0 and M.layout()["operators"] == ops
    try: ModalMatrixSys(1.0, 1.0, 0, 1, g)
    except _lib.SxError as e: assert e.code == _lib.SX_ERR_FACTOR
    else: assert 0
    S.stub_bad_pivots(0)
    assert B2.create() == 0 and M2.layout()["operators"] != ops
    for x in (B, B2): x.destroy(); x.free()
    del M, M2, g
    assert S.stub_live() == 0
    print("ok")
    """)
