"""Ray queries run in batches through pinned memory: the answers of one call, at sizes around
the direct size (65536 rays), a batch (1048576) and past it, equal those of the same rays in
small calls, for both queries, trees that fit the LDS stack and trees that spill."""
import numpy as np
import pytest

import goodphotons_amd as gp
from goodphotons_amd import scenes
from tests.parity import seeded_rays

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[5, 60_000], ids=["lds", "spill"])
def probe(request, gplib):
    sd = scenes.soup(request.param, 9, res=16)
    scene, rays = gp.GpuScene(sd, gplib), seeded_rays(sd, 1_400_003, 3)
    tmax = np.random.default_rng(4).uniform(0.05, 2.0, len(rays)).astype(np.float32)
    cut = list(range(0, len(rays), 40_000))
    small = [scene.closest_hit(rays[a:a + 40_000]) for a in cut]
    occ = [scene.any_hit(rays[a:a + 40_000], tmax[a:a + 40_000]) for a in cut]
    return scene, rays, tmax, np.concatenate([p for p, _ in small]), np.concatenate([t for _, t in small]), \
        np.concatenate(occ)


@pytest.mark.parametrize("n", [1, 63, 65, 65536, 65537, 87382, 262144, 524289, 600_011, 1_048_576, 1_048_577, 1_400_003])
def test_batches_answer_alike(probe, n):
    scene, rays, tmax, prim, t, occ = probe
    for first in (0, 1_400_003 - n):
        part = slice(first, first + n)
        p, d = scene.closest_hit(rays[part])
        assert np.array_equal(p, prim[part]) and np.array_equal(d, t[part])
        assert np.array_equal(scene.any_hit(rays[part], tmax[part]), occ[part])


def test_no_rays(probe):
    scene = probe[0]
    p, d = scene.closest_hit(np.zeros((0, 6), np.float32))
    assert len(p) == len(d) == len(scene.any_hit(np.zeros((0, 6), np.float32), np.zeros(0, np.float32))) == 0
