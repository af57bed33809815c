"""Bucket order in strips inside a multi-scene layout: a scene that takes it
beside scenes that do not, in separate launches and in the fused update, and
across a change of settings that takes the strips away and brings them back.
Equal to the same scenes under the reference key, bit for bit."""
import numpy as np
import pytest

import sph_amd as S
from helpers import announce, assert_bitexact
from sph_amd import workloads as W
from test_gpu_fused import _rows

pytestmark = pytest.mark.gpu
PLATE, FLAT = (0.6, 24.0, 24.0), (24.0, 24.0, 0.6)


def _random(n, box, seed):
    r = np.random.default_rng(seed)
    pos = np.full((n, 4), 0.34, np.float32)
    pos[:, :3] = ((r.random((n, 3)) - 0.5) * box).astype(np.float32)
    vel = np.zeros((n, 4), np.float32)
    vel[:, :3] = (r.random((n, 3)) - 0.5).astype(np.float32)
    return W.Scene("random", W.scene_params(h=0.2, box=box), n, n, pos, vel, 1)


def _run(scenes, reference, fused):
    tables = [sc.n for sc in scenes] if reference else None
    with S.Batch([sc.params for sc in scenes], [sc.n for sc in scenes], tables) as b:
        if not reference:
            b.variants = _rows(fused)
        for s, sc in enumerate(scenes):
            b.upload(s, sc.pos, sc.vel)
        out = []
        for box in (PLATE, FLAT, PLATE):
            p = W.scene_params(h=0.2, box=box)
            assert S.lib().sph_batch_set_params(b._h, 1, S.ctypes.byref(p)) == 0
            b.step(W.DT, W.SUBSTEPS)
            out += [b.download(s) for s in range(len(scenes))]
        return out


@pytest.mark.parametrize("fused", [False, True])
def test_strips_beside_other_scenes_bitexact(fused):
    announce("strips in a batch", fused)
    scenes = [_random(20011, (3.0, 3.0, 3.0), 1), _random(300000, PLATE, 2), _random(1003, (2.0, 1.0, 2.0), 3),
              _random(300001, PLATE, 4)]
    for q, (got, want) in enumerate(zip(_run(scenes, False, fused), _run(scenes, True, fused))):
        for g, w, what in zip(got, want, ("positions", "velocities", "densities")):
            assert_bitexact(g, w, f"step {q // 4} scene {q % 4} {what}")
