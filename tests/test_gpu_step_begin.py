"""The first phase of a step through the C interface: fdm_launchStepBegin and
fdm_launchStepDecide, which leave the workgroups' findings in a workspace, and
fdm_launchStepBeginDecide, whose last workgroup decides (one workgroup, a few,
more than the 64 slots). Bodies, cell ids, visibility, control words,
displacement bound and counters are the same bits, on steps that keep the lists
and on one that does not; the gate skips both."""
import ctypes as C

import numpy as np
import pytest

from fundem_amd import build
from test_gpu_cell_codes import Template

pytestmark = pytest.mark.gpu
P, I, D, L = C.c_void_p, C.c_int, C.c_double, C.c_longlong


def struct(name, fields):
    return type(name, (C.Structure,), {"_fields_": fields})


Bodies = struct("Bodies", [("n", I)] + [(k, P) for k in ("x", "v", "w", "q", "F", "T", "mat", "geo")])
Geometry = struct("Geometry", [("num", I)] + [(k, P) for k in ("info", "sdf", "nodes", "chunks", "groups",
                                                              "groupNodes", "cells")])
Grid = struct("Grid", [("min", D * 3), ("max", D * 3), ("inv", D * 3), ("size", I * 3), ("num", L)])
Table = struct("Table", [(k, P) for k in ("hash", "sortKey", "sortIndex", "cellStart", "cellEnd", "prevKey",
                                          "prevCount", "validAtBuild")])
Periodic = struct("Periodic", [("x", I), ("y", I), ("sector", I), ("pad", I)] +
                  [(k, D * 3) for k in ("angle", "A", "B", "halfCos", "halfSin")])
Instances = struct("Instances", [("count", I)] + [(k, P) for k in "abcdefgh"])
Args = struct("Args", [("particles", Bodies), ("pgeo", Geometry), ("pgrid", Grid), ("ptable", Table),
                       ("walls", Bodies), ("wgeo", Geometry), ("wgrid", Grid), ("wtable", Table),
                       ("gravity", D * 3), ("dt", D), ("kick", I), ("drift", I), ("periodic", Periodic),
                       ("ghostFlag", P * 3), ("ghostAtBuild", P), ("inst", Instances), ("clear", P * 8),
                       ("gate", P)])
Skin = struct("Skin", [("skin", D), ("rhoMax", D), ("dt", D)] + [(k, P) for k in ("ctl", "disp", "ring", "fold")])
COUNTERS = 64 * 32  # FDM_REC_COUNTERS


class Side:
    """One set of device buffers, made from the seed, and its launch arguments."""

    def __init__(self, n, walls, seed, gate):
        import torch
        rng = np.random.default_rng(seed)
        self.buf = {}

        def dev(name, a, kind):
            self.buf[name] = torch.from_numpy(np.ascontiguousarray(a, kind)).cuda()
            return self.buf[name].data_ptr()

        t = Template(radius=0.1, invMass=2.0, invSpacing=10.0, boxReach=0.2)
        t.inertia[:], t.invInertia[:] = (1, 2, 3, 0, 0, 0), (1, 0.5, 1 / 3, 0, 0, 0)
        info = dev("info", np.frombuffer(bytes(t), np.uint8).copy(), np.uint8)

        def bodies(tag, m):
            q = rng.normal(size=(4, m))
            vec = lambda k, s: dev(tag + k, s * rng.normal(size=3 * m), np.float32)
            return Bodies(m, dev(tag + "x", rng.uniform(0.0, 4.0, 3 * m), np.float64), vec("v", 0.5), vec("w", 2.0),
                          dev(tag + "q", q / np.linalg.norm(q, axis=0), np.float32), vec("F", 1.0), vec("T", 1.0),
                          dev(tag + "mat", np.zeros(m), np.int32), dev(tag + "geo", np.zeros(m), np.int32))

        def table(tag, m):
            h = dev(tag + "hash", np.full(m, -7), np.int32)
            return Table(h, None, None, None, None, None, None, dev(tag + "valid", np.ones(m), np.int32))

        a = self.args = Args()
        a.particles, a.walls = bodies("p", n), bodies("w", walls)
        a.pgeo = a.wgeo = Geometry(1, info)
        a.pgrid = a.wgrid = Grid((0, 0, 0), (4, 4, 4), (2, 2, 2), (8, 8, 8), 512)
        a.ptable, a.wtable = table("p", n), table("w", walls)
        a.gravity[:] = (0, 0, -9.81)
        a.dt, a.kick, a.drift, a.periodic.x, a.periodic.y = 1e-4, 1, 1, 1, 1
        for k in range(3):
            a.ghostFlag[k] = dev(f"flag{k}", np.full(n, 9), np.int32)
        a.ghostAtBuild = dev("at", np.zeros(n), np.int32)
        a.clear[2] = dev("count", np.arange(COUNTERS), np.int32)
        a.gate = dev("gate", [gate], np.int32)
        self.skin = Skin(0.05, 0.2, 1e-4, dev("ctl", np.zeros(16), np.int32), dev("disp", [0.0], np.float64), None,
                         dev("fold", np.zeros(16 * 64 + 16), np.int32))
        self.work = torch.zeros(1 << 20, dtype=torch.uint8, device="cuda")

    def host(self):
        return {k: v.cpu().numpy() for k, v in self.buf.items()}


@pytest.mark.parametrize("n,walls,gate", [(1, 0, 1), (200, 56, 1), (200, 57, 1), (3000, 2, 1), (20000, 3, 1),
                                          (700, 2, 0)])
def test_two_launches_equal_one(n, walls, gate):
    import torch
    lib = C.CDLL(build.CORE_LIB)
    lib.fdm_stepBeginWorkspaceBytes.restype = C.c_size_t
    stream = P(torch.cuda.current_stream().cuda_stream)
    a, b = Side(n, walls, 3, gate), Side(n, walls, 3, gate)
    need = lib.fdm_stepBeginWorkspaceBytes(C.c_size_t(n + walls))
    before = a.host()
    for step in range(3):
        two = (C.byref(a.args), C.byref(a.skin), P(a.work.data_ptr()), C.c_size_t(need), stream)
        assert lib.fdm_launchStepBegin(*two) == 0 and lib.fdm_launchStepDecide(*two) == 0
        assert lib.fdm_launchStepBeginDecide(C.byref(b.args), C.byref(b.skin), stream) == 0
        u, v = a.host(), b.host()
        for key in u:
            assert np.array_equal(u[key], v[key], equal_nan=True), (step, key)
    if gate:
        assert not u["count"].any() and not u["fold"].any() and u["ctl"][10] == 3  # three decisions
        assert u["disp"][0] > 0 or u["ctl"][8] > 0
        assert not np.array_equal(u["px"], before["px"]) and (u["phash"] != -7).all()
    else:
        assert all(np.array_equal(u[k], before[k]) for k in u)
    short = (C.byref(a.args), C.byref(a.skin), P(a.work.data_ptr()), C.c_size_t(need - 1), stream)
    assert lib.fdm_launchStepBegin(*short) == -1
    a.skin.fold = None
    assert lib.fdm_launchStepBeginDecide(C.byref(a.args), C.byref(a.skin), stream) == -1
