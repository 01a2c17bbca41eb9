"""Which solve a mesh gets, on the CPU (tests/hip_stub.cpp counts launches and
runs none): the level kernels' 8-slot instances where more than four fronts
meet at a node, the split of elements that share their centre, islands, and mode counts on both sides of the rule."""
import pytest

from test_alloc_failures import run

ROUTES = [  # mesh, modes, slots of the level kernels (0: band)
    ("fan(10, 2, 8)", 32, 8), ("fan(24, 2, 4)", 32, 8), ("fan(7, 6, 5, even=False)", 8, 4),
    ("winding_ring(16, 4, 6)", 8, 4), ("apart(2, 8, 6)", 16, 4), ("apart(4, 3, 9)", 32, 0),
    ("rect_mesh(5, 5, 6)", 32, 4), ("rect_mesh(5, 5, 6)", 128, 0), ("rect_mesh(24, 20, 6)", 128, 4),
]


@pytest.mark.parametrize("mesh,modes,slots", ROUTES)
def test_route(mesh, modes, slots):
    run(f"""
    sys.path.insert(0, "tests")
    from odd_meshes import apart, fan, winding_ring
    m = {mesh}
    M = ModalMatrixSys(0.7, 1.0, 0, {modes}, GpuMesh(m))
    assert own_solve(M, 2 * {modes}) == 0
    n = {{w: launches("k_tree_levelILi2ELi%dE" % w) for w in (4, 8)}}
    assert n == {{4: {int(slots == 4)}, 8: {int(slots == 8)}}}, n
    assert (M.layout()["operators"] > 0) == ({slots} > 0) and (M.layout()["kernel"] == 4) == ({slots} > 0)
    print("ok")
    """)
