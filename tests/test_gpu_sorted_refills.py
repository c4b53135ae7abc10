"""Traces that refill the queue and sort every refill (a queue of 2^20 slots, the smallest
that does), and traces through the next smaller queue, which keep index order: the film's
words and the counters of the same photons traced in pieces too small to be sorted.
Exact equality: no tolerance."""
import numpy as np
import pytest

import goodphotons_amd as gp
from goodphotons_amd import abi, scenes

pytestmark = pytest.mark.gpu

KEYS = ("photons", "segments", "connections", "splats", "direct_connections")


@pytest.mark.parametrize("make", [lambda: scenes.cornell_c0(32), lambda: scenes.caustics_c1(48)], ids=["c0", "c1"])
def test_refills_trace_the_same_photons(gplib, make):
    sd, n = make(), (1 << 21) + (1 << 19) + 77
    gs = gp.GpuScene(sd, gplib)
    saved = gplib.tuning()
    want = None
    try:
        for queue, piece in ((saved.queue_capacity, 60000), (1 << 20, n), (1 << 19, n)):
            gplib.set_tuning(queue_capacity=queue)
            film = gp.Film(sd.camera.res_x, sd.camera.res_y, max_photons=n, lib=gplib)
            sums = dict.fromkeys(KEYS, 0)
            for at in range(0, n, piece):
                _, st = gp.trace(gs, sd.camera, film, min(piece, n - at), seed_base=31 + at, max_depth=6)
                for k in KEYS:
                    sums[k] += getattr(st, k)
            words, ledger = film.raw()
            if want is None:
                want = (words.copy(), ledger, sums)
            assert sums == want[2] and ledger == want[1], queue
            assert np.array_equal(words, want[0]), queue
            film.close()
    finally:
        gplib.set_tuning(**{k: getattr(saved, k) for k, _ in abi.Tuning._fields_})
        gs.close()
