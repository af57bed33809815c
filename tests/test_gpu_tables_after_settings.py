"""sph_debug_spatial reports the lookup of the last update, whatever settings
have been given since: a change of box or radius turns the bucket order in
strips (scenes whose planes of cells hold more than some 24,000 particles) into
other strips, takes it away or brings it, and the tables stay those of the
update until the next one."""
import numpy as np
import pytest

import sph_amd as S
from helpers import announce
from sph_amd import workloads as W
from test_gpu_gridkey import _sub_dt

pytestmark = pytest.mark.gpu

N = 300_000
PLATE, OTHER_PLATE, FLAT = (0.6, 24.0, 24.0), (0.6, 12.0, 48.0), (24.0, 24.0, 0.6)


def _tables(sim):
    return {k: v.copy() for k, v in sim.debug_spatial().items()}


@pytest.mark.parametrize("first,second", [
    ((PLATE, 0.2), (OTHER_PLATE, 0.2)),  # strips -> strips over another grid
    ((PLATE, 0.2), (PLATE, 0.4)),        # -> strips over larger cells
    ((PLATE, 0.2), (FLAT, 0.2)),         # strips -> none
    ((FLAT, 0.2), (PLATE, 0.2)),         # none -> strips
])
def test_tables_are_the_last_updates(first, second):
    announce("tables after settings", first, second)
    (box, h), (box2, h2) = first, second
    r = np.random.default_rng(7)
    pos = np.full((N, 4), 0.34, np.float32)
    pos[:, :3] = ((r.random((N, 3)) - 0.5) * box).astype(np.float32)
    vel = np.zeros((N, 4), np.float32)
    with S.Sim(W.scene_params(h=h, box=box), N, S.TABLE_GRID) as sim:
        sim.upload(pos, vel)
        sim.update(_sub_dt())
        want = _tables(sim)
        sim.params = W.scene_params(h=h2, box=box2)
        sim.params = W.scene_params(h=h, box=OTHER_PLATE)  # (a second change before the update)
        sim.params = W.scene_params(h=h2, box=box2)
        got = _tables(sim)
        for k in want:
            np.testing.assert_array_equal(got[k], want[k], err_msg=k)
        # and after the next update those of its settings
        x, v, _ = sim.download()
        sim.update(_sub_dt())
        after = _tables(sim)
        table = sim.table
    with S.Sim(W.scene_params(h=h2, box=box2), N, S.TABLE_GRID) as fresh:
        fresh.upload(x, v)
        fresh.update(_sub_dt())
        np.testing.assert_array_equal(after["hash_id"], fresh.debug_spatial()["hash_id"])
    assert sorted(after["sorted_idx"]) == list(range(N)) and (after["key_id"] < table).all()
