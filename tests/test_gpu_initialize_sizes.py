"""sph_initialize's densities and tables under the reference key on either side
of the size at which its density pass goes back to one work-item per particle,
and the updates that follow."""
import numpy as np
import pytest

import pyoracle as O
import sph_amd as S
from helpers import announce, assert_bitexact, orc_params
from sph_amd import workloads as W

pytestmark = pytest.mark.gpu
DT = float(np.float32(np.float32(W.DT) / np.float32(W.SUBSTEPS)))


@pytest.mark.parametrize("n", [700000, 700001])
def test_initialize_reference_key_bitexact(n):
    announce("initialize", n)
    O.set_threads(16)
    box = (14.0, 14.0, 14.0)
    p = W.scene_params(h=0.2, box=box)
    pos, vel = S.generate(S.INIT_UNIFORM_LOWER, 5, n, box)
    op = orc_params(p)
    with S.Sim(p, n, S.TABLE_REFERENCE) as sim:
        sim.initialize(S.INIT_UNIFORM_LOWER, 5, box)
        _, _, dens = sim.download()
        at_rest = orc_params(p)
        at_rest.lookahead = 0.0
        at_rest.gravity_on = 0
        assert_bitexact(dens, O.update(at_rest, 0.0, pos, vel, T=n)[2], "densities")
        sim.update(DT)
        got = sim.download()
    want = O.update(op, DT, pos, vel, T=n)
    for g, w, c, what in zip(got, want, (3, 3, 2), ("positions", "velocities", "densities")):
        assert_bitexact(g[:, :c], w[:, :c], what)
