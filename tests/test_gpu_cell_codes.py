"""Cell codes of templates (fdm_launchCellCodes): 0 where the interpolant can be
at or below zero, elsewhere the distance to the nearest such cell, against every
cell and marked cell in numpy: a closed surface, one corner, no cell and every
cell marked, one cell, rows longer than the sixteen cells told apart, values
around the threshold, and a grid past the largest that is told."""
import ctypes as C

import numpy as np
import pytest

from fundem_amd import build

pytestmark = pytest.mark.gpu


class Template(C.Structure):
    _fields_ = [("radius", C.c_double), ("invMass", C.c_double), ("inertia", C.c_double * 6),
                ("invInertia", C.c_double * 6), ("origin", C.c_double * 3), ("invSpacing", C.c_double),
                ("lipschitz", C.c_double), ("boxReach", C.c_double), ("sdfStart", C.c_longlong),
                ("size", C.c_int * 3), ("nodeStart", C.c_int), ("nodeCount", C.c_int), ("chunkStart", C.c_int),
                ("chunkCount", C.c_int), ("affine", C.c_int), ("plane", C.c_double * 4),
                ("planeSlack", C.c_double), ("cellStart", C.c_longlong), ("groupStart", C.c_int),
                ("groupCount", C.c_int)]


def device_codes(sdfs, spacing):
    import torch
    lib = C.CDLL(build.CORE_LIB)
    ts, s0, c0, most = (Template * len(sdfs))(), 0, 0, 0
    for t, s in zip(ts, sdfs):
        nz, ny, nx = s.shape
        t.size[:] = (nx, ny, nz)
        t.invSpacing = 1.0 / spacing
        t.sdfStart, t.cellStart = s0, c0
        s0 += s.size
        n = (nx - 1) * (ny - 1) * (nz - 1)
        c0 += n
        most = max(most, n)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    table = dev(np.frombuffer(bytes(ts), np.uint8).copy())
    sdf = dev(np.concatenate([s.reshape(-1) for s in sdfs]).astype(np.float32))
    cells = torch.full((c0,), 77, dtype=torch.uint8, device="cuda")
    work = torch.full((2 * c0,), 99, dtype=torch.uint8, device="cuda")
    p = lambda a: C.c_void_p(a.data_ptr())
    args = (p(table), C.c_int(len(sdfs)), C.c_longlong(most), p(sdf), p(cells), C.c_longlong(c0), p(work))
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.fdm_launchCellCodes(*args, C.c_size_t(2 * c0 - 1), stream) == -1  # workspace too small
    assert lib.fdm_launchCellCodes(*args, C.c_size_t(2 * c0), stream) == 0
    got, at, out = cells.cpu().numpy(), 0, []
    for s in sdfs:
        shape = tuple(n - 1 for n in s.shape)
        out.append(got[at:at + int(np.prod(shape))].reshape(shape))
        at += int(np.prod(shape))
    return out


def codes(s, low):
    """By definition: gaps of one cell's box to another's, per axis."""
    low = np.float32(low)
    s = s.astype(np.float32)
    solid = np.zeros(tuple(n - 1 for n in s.shape), bool)
    for q in range(8):
        solid |= s[tuple(slice(q >> a & 1, s.shape[a] - 1 + (q >> a & 1)) for a in range(3))] <= low
    marked = np.argwhere(solid)
    out = np.zeros(solid.shape, np.uint8)
    for c in np.argwhere(~solid):
        d2 = 256
        if len(marked):
            d2 = min(d2, int((np.maximum(np.abs(marked - c) - 1, 0) ** 2).sum(1).min()))
        out[tuple(c)] = min(255, 1 + int(np.floor(15 * np.sqrt(float(d2)) * (1.0 - 1e-9))))
    return out


def grids():
    rng = np.random.default_rng(5)
    ball = np.stack(np.meshgrid(*[np.linspace(-1.6, 1.6, n) for n in (14, 12, 17)], indexing="ij"))
    corner = np.ones((9, 8, 7))
    corner[-1, 0, -1] = -1.0
    long = np.ones((4, 3, 60))
    long[1, 1, 30] = 0.0
    column = np.ones((55, 5, 2))
    column[0, 0, 0] = column[54, 4, 1] = -1.0
    few = np.where(rng.random((15, 21, 24)) < 0.002, -1.0, 1.0)
    edge = 1e-9 * rng.choice([0.5, 0.999, 1.001, 30.0], size=(8, 9, 10))  # about a millionth of the spacing
    return [np.sqrt((ball ** 2).sum(0)) - 0.8, corner, np.ones((5, 6, 7)), -np.ones((5, 6, 7)), np.ones((2, 2, 2)),
            -np.ones((2, 2, 2)), long, column, few, edge, np.full((3, 3, 3), np.nan)]


def test_codes_equal_their_definition():
    sdfs = grids()
    for k, (got, s) in enumerate(zip(device_codes(sdfs, 1e-3), sdfs)):
        want = codes(s, 1e-9)
        print(k, s.shape, "codes", int(want.min()), "to", int(want.max()), flush=True)
        assert np.array_equal(got, want), (k, np.argwhere(got != want)[:5])


def test_a_grid_past_the_largest_keeps_zeros_and_others_their_codes():
    s = grids()[0]
    big, small = device_codes([np.ones((163, 163, 163), np.float32), s], 1e-3)
    assert not big.any() and np.array_equal(small, codes(s, 1e-9))
