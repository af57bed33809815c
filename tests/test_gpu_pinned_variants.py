"""Variants carry the choice of one work-item per particle where they equal the
defaults, whose form else follows the scene's size: read, set again on the same
or another handle, and refused nowhere that the defaults are taken; results are
the defaults' bit for bit."""
import numpy as np
import pytest

import sph_amd as S
from helpers import announce, assert_bitexact
from sph_amd import workloads as W

pytestmark = pytest.mark.gpu


def _run(sim, sc):
    sim.upload(sc.pos, sc.vel)
    for _ in range(2):
        sim.step(W.DT, W.SUBSTEPS)
    return sim.download()


@pytest.mark.parametrize("key", [S.TABLE_GRID, S.TABLE_REFERENCE])
def test_pinned_variants_round_trip(key):
    announce("pinned variants", key)
    sc = W.dam_break(n=5000)
    with S.Sim(sc.params, sc.n, key) as a, S.Sim(sc.params, sc.n, key) as b:
        default = a.variants
        assert "pinned" not in default and not default["fused"]
        want = _run(a, sc)
        a.variants = dict(default, pinned=True)
        assert a.variants == dict(default, pinned=True)
        b.variants = a.variants
        assert b.variants == a.variants
        for sim in (a, b):
            for g, w, what in zip(_run(sim, sc), want, ("positions", "velocities", "densities")):
                assert_bitexact(g, w, what)
        a.variants = default
        assert a.variants == default


@pytest.mark.parametrize("key", [S.TABLE_GRID, S.TABLE_REFERENCE])
def test_tuned_variants_round_trip(key):
    sc = W.dam_break(n=3000)
    announce("tuned variants", key)
    with S.Sim(sc.params, sc.n, key) as a, S.Sim(sc.params, sc.n, key) as b:
        a.upload(sc.pos, sc.vel)
        a.autotune(W.DT / W.SUBSTEPS, 2)
        tuned = a.variants
        b.variants = tuned
        assert b.variants == tuned
        # a pick equal to the defaults that is not pinned is the defaults' own form
        assert np.array_equal(_run(a, sc)[0], _run(b, sc)[0])
