"""Meshes that are no rectangle, for the tests: fans (more than four elements
at a node), a ring that winds round twice (elements that share their centre),
and islands (nothing connects them)."""
import numpy as np

from semtex_amd.mesh import ESSENTIAL, NATURAL, Mesh2D, _bandwidth, edgemaps, gll, number_nodes


def from_quads(np_, corners, keys_of, kinds):
    """corners: [nel][4][2], CCW; keys_of (e, i): a hashable name of element-
    boundary node i of element e (equal names are one node); kinds: {(e, side):
    "D" or "N"}."""
    z, _, _ = gll(np_)
    s = 0.5 * (1.0 + z)
    C = np.asarray(corners, float)
    nel = len(C)
    a, b = np.meshgrid(s, s)                       # a along the first side
    w = [(1 - a) * (1 - b), a * (1 - b), a * b, (1 - a) * b]
    X = np.array([sum(w[q] * C[e, q, 0] for q in range(4)).ravel() for e in range(nel)])
    Y = np.array([sum(w[q] * C[e, q, 1] for q in range(4)).ravel() for e in range(nel)])
    emap, _ = edgemaps(np_)
    nx = 4 * (np_ - 1)
    bx, by = X[:, emap[:nx]], Y[:, emap[:nx]]
    names, keys = {}, np.zeros((nel, nx), np.int64)
    for e in range(nel):
        for i in range(nx):
            keys[e, i] = names.setdefault(keys_of(e, i, bx[e, i], by[e, i]), len(names))
    coords = np.zeros((len(names), 2))
    coords[keys.ravel(), 0], coords[keys.ravel(), 1] = bx.ravel(), by.ravel()
    ess = np.zeros(len(names), bool)
    nm = np_ - 1
    for (e, side), k in kinds.items():
        if k == "D":
            ess[keys[e, [side * nm + i for i in range(nm)] + [0 if side == 3 else side * nm + nm]]] = True
    btog, nsolve, how = number_nodes(keys, ess, coords, (None, None))
    bmask = ess[keys].astype(np.int32)
    order = sorted(kinds)
    return Mesh2D(np=np_, nel=nel, x=np.ascontiguousarray(X), y=np.ascontiguousarray(Y),
                  btog=np.ascontiguousarray(btog), bmask=np.ascontiguousarray(bmask),
                  emask=bmask.any(axis=1).astype(np.int32), nglobal=len(names), nsolve=nsolve,
                  nband=_bandwidth(btog, bmask, nsolve),
                  bnd_elmt=np.array([e for e, _ in order], np.int32),
                  bnd_side=np.array([s_ for _, s_ in order], np.int32),
                  bnd_kind=np.array([{"D": ESSENTIAL, "N": NATURAL}[kinds[o]] for o in order], np.int32),
                  cyl=0, info={"ordering": how})


def _by_place(e, i, x, y):
    return round(x * 1e7), round(y * 1e7)


def fan(sectors, n, np_, bc="D", at=(0.0, 0.0), even=True):
    """`sectors` kites round one node, each n x n elements; even: all alike
    (turned), otherwise each of its own size."""
    th = 2 * np.pi / sectors
    corners, kinds = [], {}
    for s in range(sectors):
        r = 1.0 if even else 1.0 + 0.07 * s
        p = [np.zeros(2)] + [r_ * np.array([np.cos(t), np.sin(t)]) for r_, t in
                             ((1.0, s * th), (r / np.cos(th / 2), (s + 0.5) * th), (1.0, (s + 1) * th))]
        f = lambda u, v: ((1 - u) * (1 - v) * p[0] + u * (1 - v) * p[1] + u * v * p[2] + (1 - u) * v * p[3]
                          + np.asarray(at))
        for j in range(n):
            for i in range(n):
                e = len(corners)
                corners.append([f(i / n, j / n), f((i + 1) / n, j / n), f((i + 1) / n, (j + 1) / n),
                                f(i / n, (j + 1) / n)])
                if i == n - 1: kinds[e, 1] = bc
                if j == n - 1: kinds[e, 2] = bc if bc == "N" else ("D" if s % 2 == 0 else "N")
    return from_quads(np_, corners, _by_place, kinds)


def winding_ring(nt, nr, np_):
    """A ring of nr layers that closes after two turns of nt elements each."""
    corners, kinds = [], {}
    th = 2 * np.pi / nt
    for j in range(nr):
        for t in range(2 * nt):
            e = len(corners)
            c = lambda r, a: [(1.0 + 0.5 * r) * np.cos(a * th), (1.0 + 0.5 * r) * np.sin(a * th)]
            corners.append([c(j, t), c(j + 1, t), c(j + 1, t + 1), c(j, t + 1)])
            if j == 0: kinds[e, 3] = "D"
            if j == nr - 1: kinds[e, 1] = "N"
    nm = np_ - 1

    def key(e, i, x, y):
        j, t = divmod(e, 2 * nt)
        side, q = divmod(i, nm)
        u, v = ((q, 0), (nm, q), (nm - q, nm), (0, nm - q))[side]
        return j * nm + u, (t * nm + v) % (2 * nt * nm)
    return from_quads(np_, corners, key, kinds)


def twice_round(n, np_):
    """Eight squares of n x n elements round one node (each quarter of the
    plane twice): rectangles all, with eight elements at the node."""
    corners, kinds, nm = [], {}, np_ - 1
    turn = lambda q, u, v: [(u, v), (-v, u), (-u, -v), (v, -u)][q % 4]
    for s in range(8):
        for j in range(n):
            for i in range(n):
                e = len(corners)
                corners.append([turn(s, i + a, j + b) for a, b in ((0, 0), (1, 0), (1, 1), (0, 1))])
                if i == n - 1: kinds[e, 1] = "D" if s % 2 else "N"
                if j == n - 1: kinds[e, 2] = "N"

    def key(e, i, x, y):
        s, q = divmod(e, n * n)
        side, t = divmod(i, nm)
        a, b = ((t, 0), (nm, t), (nm - t, nm), (0, nm - t))[side]
        u, v = (q % n) * nm + a, (q // n) * nm + b
        if u == 0 and v == 0: return "node"
        if u == 0: return "ray", (s + 1) % 8, v     # the next square's first axis
        if v == 0: return "ray", s, u
        return s, u, v
    return from_quads(np_, corners, key, kinds)


def apart(islands, n, np_):
    corners, kinds = [], {}
    for x0 in (n + 2.0) * np.arange(islands):
        for j in range(n):
            for i in range(n):
                e = len(corners)
                corners.append([(x0 + i, j), (x0 + i + 1, j), (x0 + i + 1, j + 1), (x0 + i, j + 1)])
                if j == 0: kinds[e, 0] = "D"
                if i == n - 1: kinds[e, 1] = "N"
                if j == n - 1: kinds[e, 2] = "N"
                if i == 0: kinds[e, 3] = "D"
    return from_quads(np_, corners, _by_place, kinds)
