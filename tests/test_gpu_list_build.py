"""Candidate lists by the few-launch build (build.hip) at the sizes where its
parts change hands: sixteen lanes per particle, four particles per wave, the
one-workgroup sort of up to 2048 keys, the one-workgroup scan of up to 8192
counts, the walls' table of up to 1024 walls, and particles with more
candidates than are sorted in LDS (32) or than the wave's scratch holds. States
and contacts against the oracle, bit for bit, with lists kept over steps."""
import dataclasses

import numpy as np
import pytest

import pyoracle as po
from fundem_amd import workloads as W
from test_gpu_parity import assert_contacts_equal, assert_states_equal
from test_gpu_sweep import squeezed

pytestmark = pytest.mark.gpu


def small_family():
    return W.superellipsoid_family(2, 11, n_grid=12, n_nodes=40, axes=(0.8e-3, 1.2e-3))


def against_oracle(scn, steps, every, precision="fp32", skin=None, builds=0):
    from fundem_amd import Solver
    g = Solver(precision=precision)
    if skin is not None:
        g.set_capacity(200, 64)
        g.set_skin(skin)
    W.apply(scn, g)
    o = po.OracleSim(precision == "fp32", True)
    W.apply(scn, o)
    seen = 0
    for i in range(every, steps + 1, every):
        g.step(every)
        o.step(every)
        assert_states_equal(g.state(), o.state(), f"step {i}")
        assert_contacts_equal(g, o, f"step {i}")
        seen += sum(o.contacts(s)["A"].size for s in range(5))
    assert g.status() == 0
    print(f"n {scn.n} pairs {g.pair_totals()} contacts seen {seen}", flush=True)
    g.close()
    return seen


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 15, 16, 17, 511, 513])
def test_particles_per_group_and_block_bitexact(n, precision):
    against_oracle(squeezed(n=n, templates=small_family()), 150, 50, precision)


@pytest.mark.parametrize("n", [2047, 2048, 2049, 8191, 8192])
def test_sort_and_scan_edges_bitexact(n):
    scn = W.cluster(n=n, seed=2, speed=6.0, spin=200.0, spacing=2.5, periodic=(True, n % 2 == 0),
                    templates=small_family())
    assert against_oracle(scn, 80, 40) > 0


@pytest.mark.parametrize("skin,periodic", [(0.0, True), (2e-3, True), (6e-3, False)])
def test_many_candidates_bitexact(skin, periodic):
    scn = squeezed(n=125, templates=small_family())
    if not periodic:  # (4 N pairs per image set would not hold these)
        scn = dataclasses.replace(scn, periodic=(False, False))
    assert against_oracle(scn, 240, 60, skin=skin) > 0


@pytest.mark.parametrize("walls", [33, 1024, 1025])
def test_many_walls_bitexact(walls):
    scn = squeezed(n=8, templates=small_family())
    p, *rest = scn.walls[0]
    more = [(np.asarray(p) + [0., 0., 1e-7 * i], *rest) for i in range(1, walls)]
    scn = dataclasses.replace(scn, walls=[scn.walls[0]] + more, v=scn.v - [0., 0., 3.0])
    assert against_oracle(scn, 120, 40) > 0
