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


@pytest.mark.parametrize("name,h", [("solo", 0.08), ("bricks", 0.05), ("many bricks", 0.035)])
def test_open_mesh_on_either_side_of_the_brick_rule(name, h):
    """Every node of an open mesh takes the solid angles: with the nearest
    triangle in one loop on grids of less than 768 bricks, after kMeshNearest
    (sixteen waves a brick below 4096, four above) on larger ones; numbers of
    nodes and triangles that are no multiple of eight."""
    v, f = G.icosphere(1.0, 1 if name == "many bricks" else 3)
    f = f[:-1]
    m = G.MeshParticle(v * (1.0, 1.1, 1.2), f)
    origin, hh, size, vals = m.build_grid(h)
    bricks = int(np.prod([(n + 3) // 4 for n in size]))
    print(f"{len(f)} triangles, {vals.size} nodes, {bricks} bricks", flush=True)
    assert len(f) * vals.size >= 1 << 22 and len(f) % 8 and vals.size % 8
    assert name == ("solo" if bricks < 768 else "bricks" if bricks < 4096 else "many bricks")
    o2, s2, v2 = po.mesh_grid(v * (1.0, 1.1, 1.2), f, h, 2)
    assert np.array_equal(origin, o2) and size == s2 and np.array_equal(vals, v2)


@pytest.mark.parametrize("nu,nv,res", [(40, 20, 30), (80, 32, 50), (160, 64, 30)])
def test_open_mesh_is_not_slower_than_every_triangle_at_every_node(nu, nv, res):
    """The grid path of an open mesh against the kernel that takes solid angle
    and distance of every triangle at every node (the shortest of ten launches
    each; a fifth is left for the spread between runs, less than half of what
    the path was slower when each node had a workgroup of its own)."""
    import ctypes as C
    import torch
    from fundem_amd import build
    lib = C.CDLL(build.CORE_LIB)
    lib.fdm_meshGridWorkspaceBytes.restype = C.c_size_t
    v, f = G.torus_mesh(1.0, 0.35, nu, nv)
    f = f[:-1]
    origin, h, size, vals = G.MeshParticle(v, f).build_grid_by_resolution(res)
    tri = torch.tensor(v[f].reshape(-1), dtype=torch.float64, device="cuda")
    out = torch.zeros(vals.size, dtype=torch.float64, device="cuda")
    n3, o3 = (C.c_int * 3)(*size), (C.c_double * 3)(*origin)
    need = lib.fdm_meshGridWorkspaceBytes(C.c_int(len(f)), n3)
    work = torch.zeros(int(need), dtype=torch.uint8, device="cuda")
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    common = (C.c_void_p(tri.data_ptr()), C.c_int(len(f)), o3, C.c_double(h), n3, C.c_int(0), C.c_void_p(out.data_ptr()))

    def shortest(call):
        best, got = 1e9, None
        for _ in range(10):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            assert call() == 0
            b.record()
            b.synchronize()
            best, got = min(best, a.elapsed_time(b)), out.cpu().numpy()
        return best, got

    old, u = shortest(lambda: lib.fdm_launchMeshSignedDistanceGrid(*common, stream))
    new, w = shortest(lambda: lib.fdm_launchMeshSignedDistanceGridWith(*common, C.c_void_p(work.data_ptr()),
                                                                       C.c_size_t(need), stream))
    print(f"{len(f)} triangles, {vals.size} nodes: {1e3 * old:.0f} us, grid path {1e3 * new:.0f} us", flush=True)
    assert need > 0 and np.array_equal(u, w) and new <= 1.2 * old


@pytest.mark.parametrize("n", [17, 19, 20, 24])
def test_undecided_nodes_of_a_closed_mesh_around_the_eighth(n):
    """A closed mesh far larger than the range whose signs are taken from
    crossings: every node takes the solid angles, a workgroup each below 7168
    nodes and eight a workgroup from there on; the grid equals the kernel that
    takes every triangle at every node."""
    import ctypes as C
    import torch
    from fundem_amd import build
    lib = C.CDLL(build.CORE_LIB)
    lib.fdm_meshGridWorkspaceBytes.restype = C.c_size_t
    v, f = torus()
    tri = torch.tensor((1e110 * v[f]).reshape(-1), dtype=torch.float64, device="cuda")
    n3, o3, h = (C.c_int * 3)(n, n, n), (C.c_double * 3)(*[-1.6e110] * 3), 3.2e110 / (n - 1)
    need = lib.fdm_meshGridWorkspaceBytes(C.c_int(len(f)), n3)
    work = torch.zeros(int(need), dtype=torch.uint8, device="cuda")
    stream, got = C.c_void_p(torch.cuda.current_stream().cuda_stream), []
    for grid in (False, True):
        out = torch.zeros(n ** 3, dtype=torch.float64, device="cuda")
        args = (C.c_void_p(tri.data_ptr()), C.c_int(len(f)), o3, C.c_double(h), n3, C.c_int(0), C.c_void_p(out.data_ptr()))
        if grid:
            r = lib.fdm_launchMeshSignedDistanceGridWith(*args, C.c_void_p(work.data_ptr()), C.c_size_t(need), stream)
        else:
            r = lib.fdm_launchMeshSignedDistanceGrid(*args, stream)
        assert r == 0 and need > 0
        got.append(out.cpu().numpy())
    assert np.array_equal(got[0], got[1], equal_nan=True)
