"""sph_update_noalloc recorded into a caller's graph: the scratch array's counts
are what the calls run before a replay leave, not what they were when it was
recorded.  Every call and replay equals the handle path, bit for bit, with
calls of both forms (several work-items per particle; walking, taken for a
radius outside the fast arithmetic's range) around them."""
import ctypes

import numpy as np
import pytest

import sph_amd as S
import test_zz_no_alloc as N
from helpers import announce, assert_bitexact
from sph_amd import workloads as W

pytestmark = pytest.mark.gpu

DT = float(np.float32(np.float32(W.DT) / np.float32(W.SUBSTEPS)))


def _tiny_radius():
    h, n = 1.0e-5, 700
    q = np.arange(n)  # a lattice of spacing 2 h, 9 a side: the poly6 factor of a pair would overflow
    pos = np.full((n, 4), 0.34, np.float32)
    pos[:, :3] = (np.stack([q // 81, (q // 9) % 9, q % 9], 1) - 4) * (2 * h)
    vel = np.zeros((n, 4), np.float32)
    p = S.default_params(smoothing_radius=h, gravity_on=0, pressure_mult=0.0, near_pressure_mult=0.0, viscosity=0.0,
                         bounds=(20 * h, 20 * h, 20 * h))
    return W.Scene("tiny radius", p, n, n, pos, vel, 1)


class _Graph:
    """A call on its own stream, recorded; run() replays it and returns its outputs."""

    def __init__(self, hip, sc):
        self.hip, self.sc, n = hip, sc, sc.n
        self.bufs = [hip.put(sc.pos), hip.put(sc.vel), hip.malloc(16 * n), hip.malloc(16 * n), hip.malloc(8 * n)]
        self.stream, graph, self.exec = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
        L = hip.L
        assert L.hipStreamCreate(ctypes.byref(self.stream)) == 0
        assert L.hipStreamBeginCapture(self.stream, 1) == 0  # hipStreamCaptureModeThreadLocal
        p = sc.params
        rc = N._entry()(ctypes.byref(p), n, DT, *self.bufs, self.stream, 0)
        assert L.hipStreamEndCapture(self.stream, ctypes.byref(graph)) == 0
        assert rc == 0, S.last_error()
        assert L.hipGraphInstantiate(ctypes.byref(self.exec), graph, None, None, ctypes.c_size_t(0)) == 0

    def run(self):
        L, n = self.hip.L, self.sc.n
        assert L.hipGraphLaunch(self.exec, self.stream) == 0
        assert L.hipStreamSynchronize(self.stream) == 0
        return tuple(self.hip.get(b, (n, w), np.float32) for b, w in zip(self.bufs[2:], (4, 4, 2)))


def _same(got, want, what):
    for g, w, part in zip(got, want, ("positions", "velocities", "densities")):
        assert_bitexact(g, w, f"{what}: {part}")


def test_recorded_calls_and_calls_around_them():
    hip = N._Hip()
    for f in ("hipStreamCreate", "hipStreamSynchronize"):
        getattr(hip.L, f).argtypes = [ctypes.c_void_p]
    hip.L.hipGraphLaunch.argtypes = [ctypes.c_void_p] * 2
    hip.L.hipStreamBeginCapture.argtypes = [ctypes.c_void_p, ctypes.c_int]
    hip.L.hipStreamEndCapture.argtypes = [ctypes.c_void_p] * 2
    small, large, tiny = W.dam_break(n=3000), W.dam_break(n=20000), _tiny_radius()
    want = {sc.name + str(sc.n): N._handle(sc, DT) for sc in (small, large, tiny)}

    def call(sc, what):
        announce("noalloc", what, sc.n)
        _same(N._noalloc(hip, sc, DT), want[sc.name + str(sc.n)], what)

    call(small, "first")
    call(tiny, "walking form")
    graphs = {"several": _Graph(hip, large), "walking": _Graph(hip, tiny)}
    call(small, "after recording, before any replay")
    for _ in range(3):
        for name, sc in (("several", large), ("walking", tiny)):
            announce("noalloc replay", name)
            _same(graphs[name].run(), want[sc.name + str(sc.n)], f"replay, {name}")
            call(small, f"after the replay, {name}")
            call(tiny, "walking form")
            _same(graphs[name].run(), want[sc.name + str(sc.n)], f"replay after the walking form, {name}")
