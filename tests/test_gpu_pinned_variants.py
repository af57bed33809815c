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
        assert a.form == (16, 16)
        a.variants = dict(default, pinned=True)
        assert a.variants == dict(default, pinned=True) and a.form == (1, 0)
        b.variants = a.variants
        assert b.variants == a.variants and b.form == (1, 0)
        for sim in (a, b):
            for g, w, what in zip(_run(sim, sc), want, ("positions", "velocities", "densities")):
                assert_bitexact(g, w, what)
        a.variants = default
        assert a.variants == default and a.form == (16, 16)


@pytest.mark.parametrize("key", [S.TABLE_GRID, S.TABLE_REFERENCE])
def test_tuned_variants_round_trip(key):
    sc = W.dam_break(n=3000)
    announce("tuned variants", key)
    with S.Sim(sc.params, sc.n, key) as a, S.Sim(sc.params, sc.n, key) as b:
        a.upload(sc.pos, sc.vel)
        a.autotune(W.DT / W.SUBSTEPS, 2)
        tuned = a.variants
        b.variants = tuned
        assert b.variants == tuned and b.form == a.form
        assert np.array_equal(_run(a, sc)[0], _run(b, sc)[0])


@pytest.mark.parametrize("n,grid,reference", [
    (1, (16, 16), (16, 16)), (16384, (16, 16), (16, 16)), (16385, (8, 16), (8, 16)), (65536, (8, 16), (8, 16)),
    (65537, (8, -16), (8, 32)), (127000, (8, -16), (8, 32)), (127001, (1, 0), (8, 32)),
])
def test_default_form_by_size(n, grid, reference):
    announce("form by size", n)
    p = W.scene_params()
    with S.Sim(p, n, S.TABLE_GRID) as a, S.Sim(p, n, S.TABLE_REFERENCE) as b:
        assert a.form == grid and b.form == reference
        p.prefilter_r2 = 2.0 ** -62  # outside the fast arithmetic's range
        a.params = b.params = p
        assert a.form == b.form == (1, 0)
