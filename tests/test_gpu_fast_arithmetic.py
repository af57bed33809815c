"""The arithmetic that the record-reading kernels use in place of IEEE square
roots and divisions, and the walk's one-sided distance test: the root equals
IEEE sqrt on its whole range, and updates stay bit-exact against the oracle
where the range proofs end -- radii at and past the limits, settings that make
forces tiny or huge, lattices whose neighbours lie at exactly h, particles on
the coordinate planes."""
import numpy as np
import pytest

import pyoracle as O
import sph_amd as S
from helpers import announce, assert_bitexact, orc_params
from sph_amd import workloads as W

pytestmark = pytest.mark.gpu


def _bits(x):
    return int(np.float32(x).view(np.uint32))


def test_root_equals_ieee_on_its_range():
    announce("root_rn")
    bad, first = S.debug_root_mismatches(_bits(2.0 ** -100), _bits(2.0 ** 100))
    assert bad == 0, f"{bad} floats differ, the first {first:#x}"
    assert S.debug_root_mismatches(0, 0) == (0, 0xFFFFFFFF)  # sqrt(0)


def _masks(sim):
    """Explicit variants: one work-item per particle over neighbour masks."""
    v = sim.variants
    for k, b in zip(("density", "pressure", "viscosity"), (256, 128, 256)):
        v[k] = {"work": False, "list": False, "block": b, "rows": True}
    v.update(nbr=True, fused=False)
    return v


def _scene(h, n=6000, jitter=0.01, seed=5, centred=False):
    m = int(np.ceil(n ** (1.0 / 3.0)))
    box = (1.5 * m * 0.5 * h,) * 3
    pos, vel = S.generate(S.INIT_CENTRED_BLOCK if centred else S.INIT_DAM_BREAK, seed, n, box, 0.5 * h, jitter * h)
    return pos, vel, W.scene_params(h=h, rho0=8.0 / h ** 3, box=box)


def _check(pos, vel, p, masks, dt=1.0 / 360.0, updates=3):
    n = len(pos)
    O.set_threads(16)
    with S.Sim(p, n, S.TABLE_GRID) as sim:
        if masks:
            sim.variants = _masks(sim)
        sim.upload(pos, vel)
        for _ in range(updates):
            sim.update(dt)
        got = sim.download()
    want = O.update(orc_params(p), float(np.float32(dt)), pos, vel, T=n, substeps=updates)
    assert_bitexact(got[0][:, :3], want[0][:, :3], "positions")
    assert_bitexact(got[1][:, :3], want[1][:, :3], "velocities")
    assert_bitexact(got[2], want[2], "densities")


@pytest.mark.parametrize("masks", [False, True])
@pytest.mark.parametrize("h", [2.0 ** -18, 2.0 ** -16, 1e-3, 0.35, 8.0, 100.0, 5000.0])
def test_radii_bitexact(h, masks):
    announce("radius", h, masks)
    pos, vel, p = _scene(h)
    p.prefilter_r2 = 2.0 * h * h
    # the motion of the h = 0.2 scene in units of h (at fixed k a small radius throws
    # the particles past the cells that an int32 holds)
    p.pressure_mult, p.near_pressure_mult = 300.0 * (h / 0.2) ** 2, 20.0 * (h / 0.2) ** 2
    p.gravity_scale = 9.81 * h / 0.2
    _check(pos, vel, p, masks)


@pytest.mark.parametrize("masks", [False, True])
@pytest.mark.parametrize("k,kn", [(0.0, 0.0), (1e-12, 1e-15), (1e-3, 1e9), (1e12, 1e12), (-300.0, 20.0)])
def test_pressure_scales_bitexact(k, kn, masks):
    announce("pressure scale", k, kn, masks)
    pos, vel, p = _scene(0.2)
    p.pressure_mult, p.near_pressure_mult = k, kn
    _check(pos, vel, p, masks, dt=1e-6 if max(abs(k), kn) > 1e6 else 1.0 / 360.0)


# spacing h / 2 without jitter: neighbours at exactly h in exact arithmetic, on either side of it in float32;
# the smaller prefilters put the cut inside the support; a centred block has particles on the coordinate planes
@pytest.mark.parametrize("masks", [False, True])
@pytest.mark.parametrize("centred", [False, True])
@pytest.mark.parametrize("r2", [0.35 * 0.35, 0.04, 0.03, 0.01])
def test_lattice_neighbours_at_the_cut_bitexact(r2, centred, masks):
    announce("lattice", r2, centred, masks)
    pos, vel, p = _scene(0.2, n=6859, jitter=0.0, centred=centred)
    p.prefilter_r2 = r2
    _check(pos, vel, p, masks)


@pytest.mark.parametrize("masks", [False, True])
def test_infinite_and_nan_particles_match_the_oracle(masks):
    """A particle at NaN and one moving at infinity: every other particle's result is the oracle's."""
    announce("non-finite", masks)
    pos, vel, p = _scene(0.2)
    pos[17, 0] = np.nan
    n = len(pos)
    with S.Sim(p, n, S.TABLE_GRID) as sim:
        if masks:
            sim.variants = _masks(sim)
        sim.upload(pos, vel)
        sim.update(1.0 / 360.0)
        got = sim.download()
    want = O.update(orc_params(p), float(np.float32(1.0 / 360.0)), pos, vel, T=n, substeps=1)
    rest = np.arange(n) != 17
    assert np.isfinite(want[0][rest, :3]).all()
    for g, w, c in zip(got, want, (3, 3, 2)):
        assert_bitexact(g[rest, :c], w[rest, :c], "the other particles")
