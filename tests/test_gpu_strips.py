"""Grid key with the bucket order in strips (scenes whose planes of cells hold
more than some 24,000 particles): a scene three cells thick takes that form at
300,000 particles.  Results equal the oracle's (reference key) bit for bit in
every form of the gathers, and the lookup tables are reported in the key's own
order.  124 rows in y: the last strip is a partial one."""
import numpy as np
import pytest

import pyoracle as O
import sph_amd as S
from helpers import announce, assert_bitexact
from sph_amd import workloads as W
from test_gpu_gridkey import _oracle, _sub_dt

pytestmark = pytest.mark.gpu

N = 300_000


def _plate(outside):
    box = (0.6, 24.0, 24.0)
    r = np.random.default_rng(5)
    pos = np.full((N, 4), 0.34, np.float32)
    vel = np.zeros((N, 4), np.float32)
    pos[:, :3] = ((r.random((N, 3)) - 0.5) * box).astype(np.float32)
    vel[:, :3] = (r.random((N, 3)) - 0.5).astype(np.float32)
    if outside:  # cells outside the grid's box wrap onto it
        pos[:200, 1:3] += np.float32(24.0)
        pos[200:300, 0] -= np.float32(3.0)
    p = W.scene_params(h=0.2, box=box)
    return W.Scene("plate", p, N, N, pos, vel, 1)


@pytest.mark.parametrize("outside", [False, True])
def test_strips_bitexact(outside):
    O.set_threads(16)
    sc = _plate(outside)
    dt = _sub_dt()
    ref = _oracle(sc, dt)
    announce("strips", sc.n, outside)
    with S.Sim(sc.params, sc.n, S.TABLE_GRID) as sim:
        grid, gdim, lo = sim.key()
        assert grid and sc.n // gdim[0] > 24576 and gdim[1] % 8 != 0
        default = sim.variants
        walk = {"work": 0, "list": 0, "block": 256, "rows": False}
        for form in (default, {"density": walk, "pressure": walk, "viscosity": walk, "nbr": 0},
                     {"density": dict(walk, list=1), "pressure": walk, "viscosity": dict(walk, list=1), "nbr": 0}):
            sim.variants = form
            sim.upload(sc.pos, sc.vel)
            sim.update(dt)
            pos_g, vel_g, dens_g = sim.download()
            assert_bitexact(dens_g, ref["dens"], f"density {form}")
            assert_bitexact(vel_g[:, :3], ref["vel"][:, :3], f"velocity {form}")
            assert_bitexact(pos_g[:, :3], ref["pos"][:, :3], f"position {form}")
        sp_g = sim.debug_spatial()
        T = sim.table
        with O.grid_key(gdim, lo):
            sp = O.spatial(ref["xp"], T, ref["op"].h)
        np.testing.assert_array_equal(sp_g["hash_id"], sp.hash_id)
        np.testing.assert_array_equal(sp_g["key_id"], sp.key_id)
        np.testing.assert_array_equal(sp_g["sorted_idx"], sp.sorted_idx)
        np.testing.assert_array_equal(sp_g["start"], sp.start)
        # steps, with buckets recorded by the update before, equal the reference key's
        sim.variants = default
        sim.upload(sc.pos, sc.vel)
        for _ in range(2):
            sim.step(W.DT, W.SUBSTEPS)
        got = sim.download()
    with S.Sim(sc.params, sc.n, S.TABLE_REFERENCE) as sim:
        sim.upload(sc.pos, sc.vel)
        for _ in range(2):
            sim.step(W.DT, W.SUBSTEPS)
        want = sim.download()
    for g, w, what in zip(got, want, ("position", "velocity", "density")):
        assert_bitexact(g, w, what + " after two steps")
