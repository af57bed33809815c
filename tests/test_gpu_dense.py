"""Fluid compressed past what a neighbour record holds, in part of a scene:
those particles are walked 64 slots of a row at a time, and the XCDs take the
scene in pieces.  Single updates equal the oracle's bit for bit, updates with
recorded buckets equal the reference key's."""
import numpy as np
import pytest

import pyoracle as O
import sph_amd as S
from helpers import announce, assert_bitexact
from sph_amd import workloads as W
from test_gpu_gridkey import _oracle, _sub_dt

pytestmark = pytest.mark.gpu

N = 150_001  # past the forms with several work-items per particle


def _scene(per_cell, outside):
    """A third of the particles at per_cell to a cell in a block, the others loose around it."""
    h, r = 0.2, np.random.default_rng(7)
    dense = N // 3
    side = h * (dense / per_cell) ** (1.0 / 3.0)
    loose = h * ((N - dense) / 6.0) ** (1.0 / 3.0)
    box = (side + loose + 1.0,) * 3
    pos = np.full((N, 4), 0.34, np.float32)
    pos[:dense, :3] = (r.random((dense, 3)) - 0.5) * side
    pos[dense:, :3] = (r.random((N - dense, 3)) - 0.5) * loose
    pos[dense:, 0] += np.float32(0.3 * loose)
    if outside:  # no bucket owned by one cell: the walk tests the float hash
        pos[-50:, 1] += np.float32(2.0 * box[1])
    vel = np.zeros((N, 4), np.float32)
    vel[:, :3] = r.random((N, 3)) - 0.5
    order = r.permutation(N)
    p = W.scene_params(h=h, box=box)
    return W.Scene("dense part", p, N, N, pos[order], vel[order], 1)


# runs of three cells around 64 slots, past two pieces of 64, past the staged range
@pytest.mark.parametrize("per_cell,outside", [(20, False), (26, True), (60, False), (60, True)])
def test_dense_part(per_cell, outside):
    O.set_threads(16)
    sc = _scene(per_cell, outside)
    dt = _sub_dt()
    ref = _oracle(sc, dt)
    announce("dense part", per_cell, outside)
    with S.Sim(sc.params, sc.n, S.TABLE_GRID) as sim:
        for _ in range(2):  # the second time in pieces in every pass
            sim.upload(sc.pos, sc.vel)
            sim.update(dt)
            pos_g, vel_g, dens_g = sim.download()
            assert_bitexact(dens_g, ref["dens"], "density")
            assert_bitexact(vel_g[:, :3], ref["vel"][:, :3], "velocity")
            assert_bitexact(pos_g[:, :3], ref["pos"][:, :3], "position")
        sim.upload(sc.pos, sc.vel)
        sim.step(W.DT, 4)
        got = sim.download()
    with S.Sim(sc.params, sc.n, S.TABLE_REFERENCE) as sim:
        sim.upload(sc.pos, sc.vel)
        sim.step(W.DT, 4)
        want = sim.download()
    for g, w, what in zip(got, want, ("position", "velocity", "density")):
        assert_bitexact(g, w, what + " after a step")
