"""Emission order: a trace of many photons emits them sorted by direction (or origin, for
a collimated light) instead of by index. The film is an integer sum over photons that
each depend on their index alone, so it must hold the same fixed-point words, and the
counters the same values, as the same photons traced in pieces too small to be sorted.
Exact equality: no tolerance."""
import numpy as np
import pytest

import goodphotons_amd as gp
from goodphotons_amd import abi, scenes

pytestmark = pytest.mark.gpu


def _two_lights():
    # a cosine and a collimated emitter: the sort key holds the emitter, each its own draws
    sd = scenes.cornell_c0(40)
    sd.emitters.append(scenes.quad_emitter((0.3, 0.9, 0.3), (0.2, 0, 0), (0, 0, 0.2), (0, -1, 0),
                                           sd.emitters[0].spd, collimated=True, beam=(0, -1, 0)))
    return sd


@pytest.mark.parametrize("make,n,queue", [
    (lambda: scenes.cornell_c0(48), (1 << 21) + 77, None),      # one refill, odd count
    (lambda: scenes.caustics_c1(48), (1 << 21) + 1, 1 << 18),   # refills that are sorted
    (lambda: scenes.cornell_c0(32), 1 << 21, 1 << 16),          # refills around the least sorted size
    (_two_lights, (1 << 21) + 12345, None),
], ids=["c0", "c1_refills", "least_refill", "two_lights"])
def test_sorted_emission_traces_the_same_photons(gplib, make, n, queue):
    sd = make()
    gs = gp.GpuScene(sd, gplib)
    saved = gplib.tuning()
    keys = ("photons", "segments", "connections", "splats", "direct_connections")
    try:
        if queue:
            gplib.set_tuning(queue_capacity=queue)
        whole = gp.Film(sd.camera.res_x, sd.camera.res_y, max_photons=n, lib=gplib)
        _, st = gp.trace(gs, sd.camera, whole, n, seed_base=31, max_depth=6)
        parts = gp.Film(sd.camera.res_x, sd.camera.res_y, max_photons=n, lib=gplib)
        sums = dict.fromkeys(keys, 0)
        for at in range(0, n, 60000):
            _, sp = gp.trace(gs, sd.camera, parts, min(60000, n - at), seed_base=31 + at, max_depth=6)
            for k in keys:
                sums[k] += getattr(sp, k)
        assert {k: getattr(st, k) for k in keys} == sums and st.photons == n
        a, b = whole.raw(), parts.raw()
        assert a[1] == b[1] and np.array_equal(a[0], b[0])
        whole.close()
        parts.close()
    finally:
        gplib.set_tuning(**{k: getattr(saved, k) for k, _ in abi.Tuning._fields_})
        gs.close()
