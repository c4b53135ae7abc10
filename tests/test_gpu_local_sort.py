"""k_shade places the survivors of each workgroup round sorted by a local key. Whatever
the grid and the queue make of the rounds (one partial round, many rounds per workgroup,
a queue smaller than one round of the grid), the traced photons are the same, so film
words and counters are equal. A trace that fits the queue runs without the scheduling
kernel, in chunks of 32 iterations (the deep case has two); one that does not is refilled.
Exact equality: no tolerance."""
import numpy as np
import pytest

import goodphotons_amd as gp
from goodphotons_amd import abi, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make,depth", [(lambda: scenes.glossy_box(40), 7), (lambda: scenes.caustics_c1(40), 40)],
                         ids=["glossy", "c1_deep"])
def test_rounds_of_the_local_sort_change_nothing(gplib, make, depth):
    sd = make()
    gs = gp.GpuScene(sd, gplib)
    n = 300_001
    saved = gplib.tuning()
    got = []
    try:
        for queue, waves in ((1 << 23, 64), (1 << 20, 4), (1 << 12, 4), (1 << 16, 5)):
            gplib.set_tuning(queue_capacity=queue, grid_waves_per_cu=waves)
            film = gp.Film(sd.camera.res_x, sd.camera.res_y, max_photons=n, lib=gplib)
            e, st = gp.trace(gs, sd.camera, film, n, seed_base=5, max_depth=depth)
            got.append((film.raw()[0], [getattr(st, k) for k in ("photons", "segments", "connections", "splats")],
                        e.as_dict()))
            film.close()
    finally:
        gplib.set_tuning(**{k: getattr(saved, k) for k, _ in abi.Tuning._fields_})
        gs.close()
    for words, counts, energy in got[1:]:
        assert np.array_equal(words, got[0][0]) and counts == got[0][1] and energy == got[0][2]
