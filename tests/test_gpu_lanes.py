"""GPU: which steps take four lanes per particle: by the slots of the active
scenes, counted by what their pairs cost (plain, viscosity or tension, the same
with stencil rows of more than 32 slots at rest density)."""
import ctypes as C

import pytest

from libfluid_amd import _lib as L
from libfluid_amd import configs

pytestmark = pytest.mark.gpu


def params(kind):
    p = configs.scaled_c1(2, 2, 2).params  # eight particles a cell at rest density
    if kind != "plain":
        p.viscosity, p.surface_tension = (0.2, 0.0) if kind == "viscous" else (0.0, 1.0)
    if kind == "long":                      # twelve
        p.mass *= 8.0 / 12.0
    return p


# (kind, particles) per scene, scenes paused, lanes
CASES = [([("plain", 61_440)], (), 4), ([("plain", 61_441)], (), 1),
         ([("viscous", 65_536)], (), 4), ([("tense", 65_537)], (), 1),
         ([("long", 98_304)], (), 4), ([("long", 98_305)], (), 1),
         ([("plain", 4000)] * 12 + [("tense", 500)], (), 4),     # a small full scene does not move
         ([("plain", 4000)] * 16 + [("tense", 500)], (), 1),     # a plain launch past its limit
         ([("plain", 4000)] * 16 + [("viscous", 4000)] * 8, (), 1),
         ([("plain", 30_720), ("viscous", 32_768)], (), 4), ([("plain", 30_721), ("viscous", 32_768)], (), 1),
         ([("tense", 4000)] * 24, (), 1), ([("tense", 4000)] * 24, range(0, 24, 2), 4),
         ([("plain", 4000)] * 24, range(1, 24, 2), 4), ([("plain", 4000)] * 28, range(1, 28), 4),
         ([("plain", 4000)] * 28, range(0, 27), 1)]              # the last one alone: a launch over every slot


@pytest.mark.parametrize("k", range(len(CASES)))
def test_lanes_by_active_slots(gpu, k):
    scenes, paused, want = CASES[k]
    slots = sum((n + 511) // 512 * 512 for _, n in scenes)
    with gpu.Batch(slots, sum(params(t).ncells + 1 for t, _ in scenes), len(scenes)) as b:
        ids = [b.add(params(t), n, 1e-4) for t, n in scenes]
        for i in paused:
            b.set_active(ids[i], False)
        got = C.c_int(0)
        L.check(L.lib.lf_batch_debug_lanes(b._h, C.byref(got)), "lanes")
        assert got.value == want
