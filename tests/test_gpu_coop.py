"""The gathers with sixteen or eight work-items per particle, which the default
variants take for small scenes and under the reference key: bit-exact against
the oracle at the edges of their group and size ranges (one particle, partial
waves and workgroups, the sizes where the lanes per particle, the rows' index
width and the form change), where lists and rows overflow, over scene
boundaries inside a wave, and across a change of variants in mid-run."""
import numpy as np
import pytest

import pyoracle as O
import sph_amd as S
from helpers import announce, assert_bitexact, orc_params
from sph_amd import workloads as W

pytestmark = pytest.mark.gpu


def _sub_dt():
    return float(np.float32(np.float32(W.DT) / np.float32(W.SUBSTEPS)))


def _lattice(n, spacing, box, seed=3):
    pos, vel = S.generate(S.INIT_DAM_BREAK, seed, n, box, spacing, 0.01 * spacing)
    vel[:, 0] = np.float32(0.3) * np.sin(pos[:, 1] * 9).astype(np.float32)
    return pos, vel


def _check(p, pos, vel, table, updates=2):
    n = len(pos)
    with S.Sim(p, n, table) as sim:
        sim.upload(pos, vel)
        sim.step(_sub_dt() * updates, updates)
        got = sim.download()
    dt = float(np.float32(np.float32(_sub_dt() * updates) / np.float32(updates)))
    want = O.update(orc_params(p), dt, pos, vel, T=n, substeps=updates)
    assert_bitexact(got[0][:, :3], want[0][:, :3], "positions")
    assert_bitexact(got[1][:, :3], want[1][:, :3], "velocities")
    assert_bitexact(got[2], want[2], "densities")


@pytest.fixture(scope="module", autouse=True)
def _threads():
    O.set_threads(16)


@pytest.mark.parametrize("key", ["grid", "reference"])
@pytest.mark.parametrize("n", [1, 3, 16, 17, 255, 4099, 16384, 16385, 65536, 65537, 131072, 131073])
def test_sizes_bitexact(n, key):
    announce("coop sizes", n, key)
    L = 0.1 * (4 * n) ** (1.0 / 3.0) + 1.0
    pos, vel = _lattice(n, 0.1, (L, L, L))
    _check(W.scene_params(box=(L, L, L)), pos, vel, S.TABLE_GRID if key == "grid" else max(1, n))


# spacing: neighbours within h = 0.2 about 33.5 (0.1 / spacing)^3 -- past the 48 terms held at once, the 96
# entries of the LDS list, the 128 entries of a 16-bit row and the 64 of a 32-bit one, runs past 32 slots
@pytest.mark.parametrize("key", ["grid", "reference"])
@pytest.mark.parametrize("n,spacing", [(5000, 0.085), (5000, 0.06), (5000, 0.04), (20011, 0.07), (20011, 0.045),
                                       (70001, 0.075), (70001, 0.05)])
def test_dense_bitexact(n, spacing, key):
    announce("coop dense", n, spacing, key)
    pos, vel = _lattice(n, spacing, (6.0, 6.0, 6.0))
    _check(W.scene_params(box=(6.0, 6.0, 6.0)), pos, vel, S.TABLE_GRID if key == "grid" else n, updates=1)


# the one-launch sort: tables of a few buckets (thousands of records each), not a multiple of the workgroups'
# ranges, and on both sides of its limit
@pytest.mark.parametrize("n,table", [(3000, 1), (3000, 7), (9001, 4097), (9001, 65535), (9001, 65536), (9001, 65537),
                                     (16384, 65536), (16384, 30011), (16385, 65536)])
def test_sort_tables_bitexact(n, table):
    announce("small sort", n, table)
    L = 0.1 * (4 * n) ** (1.0 / 3.0) + 1.0
    pos, vel = _lattice(n, 0.1, (L, L, L))
    p = W.scene_params(box=(L, L, L))
    _check(p, pos, vel, table, updates=4)
    with S.Sim(p, n, table) as sim:
        sim.upload(pos, vel)
        sim.update(_sub_dt())
        got = sim.debug_spatial()
    _, xp = O.predict(orc_params(p), _sub_dt(), pos, vel)
    want = O.spatial(xp, table, p.smoothing_radius)
    for k in ("hash_id", "key_id", "sorted_idx", "start"):
        np.testing.assert_array_equal(got[k], getattr(want, k))


@pytest.mark.parametrize("counts", [(5, 1, 130, 64, 4000), (9000, 7, 12345, 3)])
@pytest.mark.parametrize("reference", [False, True])
def test_scene_boundaries_bitexact(counts, reference):
    announce("coop batch", counts, reference)
    scenes = [W.batch_scene(n, 0.1 + 0.03 * q, 0.05 * q, 11 + q) for q, n in enumerate(counts)]
    tables = list(counts) if reference else None
    with S.Batch([sc.params for sc in scenes], list(counts), tables) as b:
        for q, sc in enumerate(scenes):
            b.upload(q, sc.pos, sc.vel)
        b.step(W.DT, W.SUBSTEPS)
        got = [b.download(q) for q in range(len(scenes))]
    for q, sc in enumerate(scenes):
        want = O.update(orc_params(sc.params), _sub_dt(), sc.pos, sc.vel, T=sc.n, substeps=W.SUBSTEPS)
        for g, w, what in zip(got[q], want, ("positions", "velocities", "densities")):
            c = 2 if what == "densities" else 3
            assert_bitexact(g[:, :c], w[:, :c], f"scene {q} {what}")


@pytest.mark.parametrize("key", ["grid", "reference"])
def test_variants_changed_between_updates_bitexact(key):
    """Default (by size), then an explicit variant, then the defaults again."""
    announce("coop variants", key)
    sc = W.dam_break(n=6000)
    with S.Sim(sc.params, sc.n, S.TABLE_GRID if key == "grid" else sc.n) as sim:
        default = sim.variants
        other = {k: dict(default[k], block=64, list=True, rows=False, work=key != "grid")
                 for k in ("density", "pressure", "viscosity")}
        other.update(nbr=False, fused=False)
        sim.upload(sc.pos, sc.vel)
        for v in (default, other, default):
            sim.variants = v
            assert sim.variants == v
            sim.step(W.DT, W.SUBSTEPS)
        got = sim.download()
    want = O.update(orc_params(sc.params), _sub_dt(), sc.pos, sc.vel, T=sc.n, substeps=3 * W.SUBSTEPS)
    assert_bitexact(got[0][:, :3], want[0][:, :3], "positions")
    assert_bitexact(got[1][:, :3], want[1][:, :3], "velocities")
    assert_bitexact(got[2], want[2], "densities")


def test_noalloc_sizes_and_sparse_boxes_bitexact():
    """sph_update_noalloc over its forms of the sort (a small table, a table past the one-launch sort's limit) and a
    radius that takes the walking kernels, in turn: each call leaves the shared scratch as the next one needs it."""
    import test_zz_no_alloc as N
    hip = N._Hip()
    cases = [(1000, 0.2, 4.0), (5000, 0.2, 9.0), (20000, 0.2, 8.0), (5000, 2.0 ** -18, 2.0 ** -12), (5000, 0.2, 12.0),
             (1, 0.2, 4.0), (65536, 0.2, 8.0)]
    for n, h, box in cases:
        announce("noalloc", n, h, box)
        pos, vel = S.generate(S.INIT_DAM_BREAK, n, n, (box,) * 3, 0.5 * h, 0.005 * h)
        p = W.scene_params(h=h, rho0=8.0 / h ** 3, box=(box,) * 3)
        p.prefilter_r2 = 2.0 * h * h
        p.pressure_mult, p.near_pressure_mult = 300.0 * (h / 0.2) ** 2, 20.0 * (h / 0.2) ** 2
        p.gravity_scale = 9.81 * h / 0.2
        sc = W.Scene("noalloc", p, n, n, pos, vel, 1)
        got = N._noalloc(hip, sc, _sub_dt(), wait=n % 2)
        want = O.update(orc_params(p), _sub_dt(), pos, vel, T=n)
        assert_bitexact(got[0][:, :3], want[0][:, :3], "positions")
        assert_bitexact(got[1][:, :3], want[1][:, :3], "velocities")
        assert_bitexact(got[2], want[2], "densities")


def test_reference_key_past_a_million():
    """The lists' forms at a size that only the reference key takes them for, against the walking forms."""
    n = (1 << 20) + 77
    sc = W.uniform_lower(n=n, table=2 * n)
    announce("reference key", n)
    got = []
    with S.Sim(sc.params, n, 2 * n) as sim:
        walk = {"work": 0, "list": 0, "block": 128, "rows": False}
        for form in (sim.variants, {"density": walk, "pressure": walk, "viscosity": walk, "nbr": 0}):
            sim.variants = form
            sim.upload(sc.pos, sc.vel)
            sim.step(W.DT, 2)
            got.append(sim.download())
    for a, b, what in zip(*got, ("positions", "velocities", "densities")):
        assert_bitexact(a, b, what)
