"""The grid path of mesh level sets (kMeshPrep to kMeshSolid in meshsdf.hip)
against the oracle, bit for bit, on both sides of the rule that takes it
(nodes times triangles) and where its parts can go wrong: triangles in no
spatial order, chunk remainders, meshes with faces, edges and vertices on grid
nodes and on the columns' rays, open meshes and soups (solid angles at every
node), inverted and nested surfaces, and duplicated triangles (ties)."""
import numpy as np
import pytest

import pyoracle as po
from fundem_amd import generators as G

pytestmark = pytest.mark.gpu


def fine_box(n):
    """A cube of n x n quads per face, its faces on multiples of 1 / n."""
    v, f = [], []
    for axis in range(3):
        for side in (0, 1):
            base = len(v)
            for i in range(n + 1):
                for j in range(n + 1):
                    p = np.zeros(3)
                    p[axis], p[(axis + 1) % 3], p[(axis + 2) % 3] = side, i / n, j / n
                    v.append(p)
            for i in range(n):
                for j in range(n):
                    a, b = base + i * (n + 1) + j, base + (i + 1) * (n + 1) + j
                    quad = [(a, b, b + 1), (a, b + 1, a + 1)]
                    f += quad if side else [t[::-1] for t in quad]
    return np.array(v), np.array(f)


def torus(shuffle=False):
    v, f = G.torus_mesh(1.0, 0.4, 61, 31)
    return v, np.random.default_rng(1).permutation(f) if shuffle else f


def nested():
    v, f = G.icosphere(1.0, 3)
    return np.concatenate([v, 0.5 * v]), np.concatenate([f, f + len(v)])


def hollow():
    v, f = G.icosphere(1.0, 3)
    return np.concatenate([v, 0.5 * v]), np.concatenate([f, f[:, ::-1] + len(v)])


MESHES = {
    "torus": torus,
    "shuffled": lambda: torus(True),
    "inverted": lambda: (torus()[0], torus()[1][:, ::-1]),
    "open": lambda: (torus()[0], torus()[1][200:]),
    "one short": lambda: (torus()[0], torus()[1][1:]),
    "box on nodes": lambda: fine_box(12),
    "nested": nested,
    "hollow": hollow,
    "doubled": lambda: (torus()[0], np.concatenate([torus()[1], torus()[1]])),
}


@pytest.mark.parametrize("res", [12, 24])
@pytest.mark.parametrize("name", list(MESHES))
def test_grid_path_equals_oracle(name, res):
    v, f = MESHES[name]()
    m = G.MeshParticle(v, f, positive_inside=res == 12)
    origin, h, size, vals = m.build_grid(1.0 / 12 if name == "box on nodes" else (v.max(0) - v.min(0)).max() / res)
    o2, s2, v2 = po.mesh_grid(v, f, h, 2, res == 12)
    assert np.array_equal(origin, o2) and size == s2
    bad = np.flatnonzero(vals != v2)
    print(f"{name}: {len(f)} triangles, {vals.size} nodes, {int((vals < 0).sum())} negative", flush=True)
    assert bad.size == 0, (bad[:10], vals[bad[:10]], v2[bad[:10]])


@pytest.mark.parametrize("subdivisions,h", [(1, 0.0185), (1, 0.0165), (4, 0.12), (3, 0.06)])
def test_either_side_of_the_rule(subdivisions, h):
    """About 2^22 nodes times triangles, and a few chunks or hundreds."""
    v, f = G.icosphere(1.0, subdivisions)
    v = v + np.array([0.013, -0.021, 0.007])
    if subdivisions == 1:
        v = v * 0.3
    m = G.MeshParticle(v, f)
    origin, hh, size, vals = m.build_grid(h)
    o2, s2, v2 = po.mesh_grid(v, f, h, 2)
    print(f"{len(f)} triangles x {vals.size} nodes = {len(f) * vals.size / 2**22:.2f} x 2^22", flush=True)
    assert np.array_equal(origin, o2) and size == s2 and np.array_equal(vals, v2)


@pytest.mark.parametrize("what", ["no number", "huge", "tiny", "plain"])
def test_unusual_coordinates_equal_the_point_kernel(what):
    """Coordinates that are no numbers or whose products leave the range of a
    double: the grid equals the point queries, which take every triangle's
    solid angle, at the same nodes."""
    v, f = torus()
    v = v.copy()
    if what == "no number":
        v[7] = np.nan
    v = v * {"huge": 1e110, "tiny": 1e-32}.get(what, 1.0)
    h = float(np.nanmax(np.abs(torus()[0]))) * {"huge": 1e110, "tiny": 1e-32}.get(what, 1.0) / 8
    m = G.MeshParticle(v, f)
    origin, h, size, vals = m.build_grid(h)
    assert len(f) * vals.size >= 1 << 22
    k, j, i = np.meshgrid(*(np.arange(n) for n in size[::-1]), indexing="ij")
    val, grad = m.evaluate(origin + h * np.stack([i, j, k], -1).reshape(-1, 3))
    with np.errstate(all="ignore"):
        gn = np.sqrt(grad[:, 0] ** 2 + grad[:, 1] ** 2 + grad[:, 2] ** 2)
        want = np.where(gn > 1e-12, val / gn, np.where(val <= 0.0, -0.5 * h, 0.5 * h))
    assert np.array_equal(vals, want, equal_nan=True)
