"""Render buffers after steps of several updates: only a step's last update
has to write them (particle order, 16 bytes at a time), and what they hold
after the step is the state and colours of that update."""
import numpy as np
import pytest

import pyoracle as O
import sph_amd as S
from helpers import announce, assert_bitexact
from sph_amd import workloads as W
from test_gpu_resident import _read_f4

pytestmark = pytest.mark.gpu


# both forms of the gathers (several work-items per particle, one), both keys
@pytest.mark.parametrize("n,table", [(1000, S.TABLE_GRID), (140_000, S.TABLE_GRID), (3001, S.TABLE_REFERENCE)])
@pytest.mark.parametrize("substeps", [2, 3])
def test_render_buffers_after_steps(n, table, substeps):
    sc = W.dam_break(n=n)
    announce("render buffers after steps", f"{n} {substeps}")
    with S.Sim(sc.params, sc.n, table) as sim:
        sim.set_colors(enable=True)
        pos_ptr, col_ptr = sim.render_buffers()
        sim.upload(sc.pos, sc.vel)
        shown = None
        # the first step has no recorded buckets; a step after an update does;
        # the second length of run is one of its own
        for run in (substeps, substeps, 1, substeps + 1):
            sim.step(W.DT, run)
            pos, vel, _ = sim.download()
            assert shown is None or not np.array_equal(shown, pos)
            shown = pos
            assert_bitexact(_read_f4(pos_ptr, sc.n), pos, f"positions after {run} updates")
            assert_bitexact(_read_f4(col_ptr, sc.n), O.speed_colors(vel), f"colours after {run} updates")
