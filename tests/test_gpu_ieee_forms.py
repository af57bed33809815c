"""The mask kernels' forms with IEEE roots and divisions, taken while a scene of
the layout lies outside the fast arithmetic's range (radius outside
[2^-16, 2^26], or a cut below 2^-60): equal to the oracle, alone, in a batch
beside usual scenes, fused and in separate launches, and while such a scene
comes and goes between the steps."""
import numpy as np
import pytest

import pyoracle as O
import sph_amd as S
from helpers import announce, assert_bitexact, orc_params
from sph_amd import workloads as W
from test_gpu_fused import _rows

pytestmark = pytest.mark.gpu
DT = float(np.float32(np.float32(W.DT) / np.float32(W.SUBSTEPS)))


def _close_pairs(n=3001, h=0.2):
    """Particles that see only what lies within 2^-31 of them: a third coincide with another, a third lie 2^-32 from one."""
    r = np.random.default_rng(3)
    box = (4.0, 4.0, 4.0)
    pos = np.full((n, 4), 0.34, np.float32)
    pos[:, :3] = ((r.random((n, 3)) - 0.5) * 3.0).astype(np.float32)
    third = n // 3
    pos[third:2 * third, :3] = pos[:third, :3]
    pos[2 * third:, :3] *= np.float32(2.0 ** -20)  # (differences of 2^-32 are floats there)
    q = pos[2 * third:2 * third + (n - 2 * third) // 2 * 2, :3]
    q[1::2] = q[0::2]
    q[1::2, 0] += np.float32(2.0 ** -32)
    vel = np.zeros((n, 4), np.float32)
    vel[:, :3] = (r.random((n, 3)) - 0.5).astype(np.float32)
    p = W.scene_params(h=h, box=box, gravity=False)
    p.prefilter_r2 = 2.0 ** -62
    p.lookahead = 0.0
    return W.Scene("close pairs", p, n, n, pos, vel, 1)


def _sparse(h, n=4099):
    """No particle within h of another (at these radii a pair overflows or underflows)."""
    q = np.arange(n)
    pos = np.full((n, 4), 0.34, np.float32)
    pos[:, :3] = (np.stack([q // 256, (q // 16) % 16, q % 16], 1) - 8).astype(np.float32) * np.float32(1.5 * h)
    vel = np.zeros((n, 4), np.float32)
    p = S.default_params(smoothing_radius=h, gravity_on=0, pressure_mult=0.0, near_pressure_mult=0.0, viscosity=0.0,
                         bounds=(64 * h, 64 * h, 64 * h))
    p.prefilter_r2 = 2.0 * h * h
    return W.Scene("sparse", p, n, n, pos, vel, 1)


ODD = {"close": _close_pairs, "small": lambda: _sparse(2.0 ** -18), "large": lambda: _sparse(2.0 ** 27)}


def _oracle(sc, updates):
    return O.update(orc_params(sc.params), DT, sc.pos, sc.vel, T=sc.n, substeps=updates)


def _same(got, want, what):
    for g, w, c, part in zip(got, want, (3, 3, 2), ("positions", "velocities", "densities")):
        assert_bitexact(g[:, :c], w[:, :c], f"{what}: {part}")


@pytest.mark.parametrize("form", ["default", "separate", "fused"])
@pytest.mark.parametrize("odd", sorted(ODD))
def test_alone(odd, form):
    O.set_threads(16)
    sc = ODD[odd]()
    announce("ieee alone", odd, form)
    with S.Sim(sc.params, sc.n, S.TABLE_GRID) as sim:
        if form != "default":
            sim.variants = _rows(form == "fused")
        sim.upload(sc.pos, sc.vel)
        for _ in range(3):
            sim.update(DT)
        _same(sim.download(), _oracle(sc, 3), f"{odd} {form}")


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("odd", sorted(ODD))
def test_beside_usual_scenes_coming_and_going(odd, fused):
    O.set_threads(16)
    scenes = [W.batch_scene(5003, 0.2, 0.05, 31), ODD[odd](), W.batch_scene(2049, 0.15, 0.1, 32)]
    announce("ieee batch", odd, fused)
    with S.Batch([sc.params for sc in scenes], [sc.n for sc in scenes]) as b:
        b.variants = _rows(fused)
        for s, sc in enumerate(scenes):
            b.upload(s, sc.pos, sc.vel)
        for _ in range(2):  # IEEE forms
            b.step(W.DT, W.SUBSTEPS)
        _same(b.download(1), _oracle(scenes[1], 6), odd)
        L, h = S.lib(), b._h
        for q in (scenes[0].params, scenes[1].params):  # the fast forms, then the IEEE ones again
            assert L.sph_batch_set_params(h, 1, S.ctypes.byref(q)) == 0
            b.upload(1, scenes[1].pos, scenes[1].vel)
            b.step(W.DT, W.SUBSTEPS)
        _same(b.download(1), _oracle(scenes[1], 3), odd + " again")
        for s in (0, 2):
            _same(b.download(s), _oracle(scenes[s], 12), f"scene {s} beside {odd}")
