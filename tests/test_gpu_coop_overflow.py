"""Several work-items per particle where the neighbour lists end: lists longer
than a row (48 to 128 entries by size and key) or than the LDS holds (96), one
batch of cells alone past that, rows of 17-bit slots in 16 bits (thin scenes,
whose neighbours lie far apart in slots, and a grid that wraps, which breaks the
order that they count on), rows short enough for two loads, and the last size
that takes these forms; single scenes, batches and sph_update_noalloc, bit-exact
against the oracle."""
import numpy as np
import pytest

import pyoracle as O
import sph_amd as S
import test_zz_no_alloc as N
from helpers import announce, assert_bitexact, orc_params
from sph_amd import workloads as W

pytestmark = pytest.mark.gpu
DT = float(np.float32(np.float32(W.DT) / np.float32(W.SUBSTEPS)))
H = 0.2


def _scene(n, per_cell, seed=1, box=None, outside=False, tall=None):
    """n particles, per_cell a cell on average, in the lower half of a box (or all of the one given)."""
    lower = 0.5 if box is None else 1.0
    if box is None:
        a = H * (n / (2.0 * per_cell)) ** (1.0 / 3.0)
        box = (2 * a, a, 2 * a)
    r = np.random.default_rng(seed)
    pos = np.full((n, 4), 0.34, np.float32)
    u = r.random((n, 3)) * (1.0, lower, 1.0) - 0.5
    pos[:, :3] = (u * box).astype(np.float32)
    if outside:
        pos[n // 2, :3] = 40.0
    if tall is not None:  # the particles in `box`, the settings' box a cube
        box = (tall, tall, tall)
    vel = np.zeros((n, 4), np.float32)
    vel[:, :3] = (r.random((n, 3)) - 0.5).astype(np.float32)
    return W.Scene("random", W.scene_params(h=H, rho0=8 / H**3, box=box), n, n, pos, vel, 1)


def _clump(n, cells, seed=2):
    sc = _scene(n, 8.0, seed)
    r = np.random.default_rng(seed)
    sc.pos[:, :3] = (r.random((n, 3)) * (H * cells)).astype(np.float32)
    return sc


def _oracle(sc, updates):
    O.set_threads(16)
    return O.update(orc_params(sc.params), DT, sc.pos, sc.vel, T=sc.n, substeps=updates)


def _same(got, want, what):
    for g, w, c, part in zip(got, want, (3, 3, 2), ("positions", "velocities", "densities")):
        assert_bitexact(g[:, :c], w[:, :c], f"{what}: {part}")


CASES = {
    "wide lanes, 12 a cell": lambda: _scene(5003, 12.0),
    "wide lanes, 24": lambda: _scene(5003, 24.0),
    "wide lanes, 40, one outside": lambda: _scene(5003, 40.0, outside=True),
    "16-bit slots, 24": lambda: _scene(40001, 24.0),
    "16-bit slots, 40": lambda: _scene(40001, 40.0),
    "17-bit slots, 12": lambda: _scene(65537, 12.0),
    "17-bit slots, 24": lambda: _scene(70001, 24.0),
    "17-bit slots, 40, one outside": lambda: _scene(70001, 40.0, outside=True),
    "17-bit slots, two planes": lambda: _scene(110000, None, box=(0.3, 23.0, 23.0)),
    "17-bit slots, one plane": lambda: _scene(126001, None, box=(0.15, 25.0, 25.0)),
    "17-bit slots, three cells in a row": lambda: _scene(90001, None, box=(23.0, 23.0, 0.3)),
    "a grid that wraps along z": lambda: _scene(70001, None, box=(30.0, 30.0, 0.5), tall=30.0),
    "a grid that wraps": lambda: _scene(70001, None, box=(6.0, 6.0, 6.0), tall=30.0),
    "a grid that wraps along x": lambda: _scene(70001, None, box=(0.5, 30.0, 30.0), tall=30.0),
    "sparse, 1": lambda: _scene(20001, 1.0),
    "sparse, 4": lambda: _scene(70001, 4.0),
    "sparse, 6": lambda: _scene(33001, 6.0),
    "the last size": lambda: _scene(127000, 16.0),
    "the first size of the masks": lambda: _scene(127001, 16.0),
    "eight cells": lambda: _clump(3001, 2),
    "one cell": lambda: _clump(1500, 1),
    "64 cells, narrow lanes": lambda: _clump(17000, 4),
}


@pytest.mark.parametrize("key", [S.TABLE_GRID, S.TABLE_REFERENCE], ids=["grid", "reference"])
@pytest.mark.parametrize("case", sorted(CASES))
def test_lists_past_their_ends_bitexact(case, key):
    sc = CASES[case]()
    announce("coop overflow", case, key)
    with S.Sim(sc.params, sc.n, key) as sim:
        sim.upload(sc.pos, sc.vel)
        for _ in range(2):
            sim.update(DT)
        _same(sim.download(), _oracle(sc, 2), case)


@pytest.mark.parametrize("reference", [False, True])
@pytest.mark.parametrize("n", [2003, 9001, 25013])
def test_batches_past_their_ends_bitexact(n, reference):
    scenes = [_scene(n, 12.0, 3), _scene(n // 2, 24.0, 4), _scene(n, 8.0, 5), _clump(701, 1, 6), _scene(n, 40.0, 7)]
    announce("coop overflow batch", n, reference)
    tables = [sc.n for sc in scenes] if reference else None
    with S.Batch([sc.params for sc in scenes], [sc.n for sc in scenes], tables) as b:
        for s, sc in enumerate(scenes):
            b.upload(s, sc.pos, sc.vel)
        b.step(2 * DT, 2)
        got = [b.download(s) for s in range(len(scenes))]
    for s, sc in enumerate(scenes):
        _same(got[s], _oracle(sc, 2), f"scene {s}")


@pytest.mark.parametrize("n,per_cell", [(16384, 12.0), (16385, 24.0), (40960, 24.0), (40961, 24.0), (65536, 8.2),
                                        (65536, 12.0), (65536, 16.0), (65536, 40.0)])
def test_noalloc_rows_bitexact(n, per_cell):
    sc = _scene(n, per_cell)
    announce("coop overflow noalloc", n, per_cell)
    _same(N._noalloc(N._Hip(), sc, DT), _oracle(sc, 1), "noalloc")
