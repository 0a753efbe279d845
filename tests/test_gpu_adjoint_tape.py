"""The contact tape by tiles of 256 pairs and the reverse gather by sixteen
bodies per workgroup: copies of one small system, solved together, have the
system's own gradient in every bit, for numbers of bodies and contacts around
those units (three bodies and three to four contacts per copy), with contacts
that come and go between the steps."""
import numpy as np
import pytest

import pyoracle as po
from fundem_amd import workloads as W
from test_gpu_adjoint import PARAMS, _scenario, resting_pile

pytestmark = pytest.mark.gpu


def gradient(copies, steps, every, periodic):
    from fundem_amd import Adjoint, Solver
    tm, x, q = resting_pile(periodic)
    rng = np.random.default_rng(5)
    v, w = rng.normal(0.0, 1e-2, size=(3, 3)), rng.normal(0.0, 2.0, size=(3, 3))
    v[2] = [0.05, 0.01, 0.0]
    scn = _scenario(tm, x, q, v, w, PARAMS, periodic)
    g = Solver()
    if copies == 1:
        W.apply(scn, g)
    else:
        W.apply_batch([scn] * copies, g)
    adj = Adjoint(g)
    adj.forward(steps, every)
    assert g.status() == 0
    seen = sum(g.contacts(s)["A"].size for s in (po.SET_PP, po.SET_PW, po.SET_GX))
    st = g.state()
    out = adj.backward(v_bar=st["v"], w_bar=1e-6 * st["w"])
    return out, seen


@pytest.mark.parametrize("copies,periodic", [(5, False), (6, True), (11, False), (85, False), (86, True), (257, False)])
def test_copies_have_the_systems_gradient(copies, periodic):
    one, c1 = gradient(1, 120, 120, periodic)
    many, c = gradient(copies, 120, 40, periodic)
    print(f"{3 * copies} bodies, {c} contacts at the end", flush=True)
    assert c == copies * c1 and np.abs(one["v"]).max() > 0
    for key in ("x", "q", "v", "w"):
        got = many[key].reshape(copies, 3, -1)
        for k in range(copies):
            assert np.array_equal(got[k], one[key]), (key, k)
