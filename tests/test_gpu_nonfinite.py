"""Particles at NaN or infinity and particles with infinite velocities: every
other particle's result is the oracle's, in every form of the gathers, on either
side of the size at which the masks' one-sided test begins."""
import numpy as np
import pytest

import pyoracle as O
import sph_amd as S
from helpers import announce, assert_bitexact, orc_params
from test_gpu_fast_arithmetic import _masks, _scene

pytestmark = pytest.mark.gpu
BAD = [17, 23, 29, 31, 37]


@pytest.mark.parametrize("n", [6000, 70000])
@pytest.mark.parametrize("form", ["grid", "masks", "reference"])
def test_the_other_particles_match_the_oracle(form, n):
    announce("non-finite", form, n)
    O.set_threads(16)
    pos, vel, p = _scene(0.2, n=n)
    pos[17, 0] = np.nan
    pos[23, 2] = np.inf
    vel[29, 1] = np.inf
    vel[31, 2] = -np.inf
    vel[37, 0] = np.nan
    dt = float(np.float32(1.0 / 360.0))
    with S.Sim(p, n, S.TABLE_REFERENCE if form == "reference" else S.TABLE_GRID) as sim:
        if form == "masks":
            sim.variants = _masks(sim)
        sim.upload(pos, vel)
        for _ in range(2):
            sim.update(dt)
        got = sim.download()
    want = O.update(orc_params(p), dt, pos, vel, T=n, substeps=2)
    rest = np.setdiff1d(np.arange(n), BAD)
    assert np.isfinite(want[0][rest, :3]).all() and np.isfinite(want[1][rest, :3]).all()
    for g, w, c in zip(got, want, (3, 3, 2)):
        assert_bitexact(g[rest, :c], w[rest, :c], "the other particles")
