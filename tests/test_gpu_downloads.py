"""Films reach the host through pinned slots of 2 MB: totals, hit counts and words of films
below, at and above a slot, and of several slots, are the words scaled on the host, bit for
bit; two threads may download at once."""
import threading

import numpy as np
import pytest

import goodphotons_amd as gp
from goodphotons_amd import scenes

pytestmark = pytest.mark.gpu
SIZES = [(1, 1), (255, 257), (256, 256), (257, 256), (331, 199), (700, 800)]


def _film(lib, size, seed):
    sd = scenes.cornell_c0(16).with_camera_res(*size)
    scene, film, n = gp.GpuScene(sd, lib), gp.Film(*size, max_photons=1 << 20, lib=lib), size[0] * size[1]
    r = np.random.default_rng([seed, n])
    film.seed(scene, sd.camera, 1 << 16, r.random((n, 3)) * 1e-3, np.floor(r.random(n) * 1e6))
    return film


def _check(film):
    words, scale = film.raw()
    xyz, hits = film.download()
    assert words[:, 3].any()
    assert np.array_equal(xyz, words[:, :3].astype(np.float64) * (1.0 / scale))
    assert np.array_equal(hits, words[:, 3].astype(np.float64))
    assert np.array_equal(film.download_hits(), hits)


@pytest.mark.parametrize("size", SIZES, ids=str)
def test_totals_are_the_words(gplib, size):
    _check(_film(gplib, size, 1))


def test_two_threads(gplib):
    films, errors = [_film(gplib, s, 2) for s in SIZES[2:]], []

    def work(part):
        try:
            for _ in range(5):
                for f in part:
                    _check(f)
        except BaseException as e:   # noqa: BLE001
            errors.append(e)
    threads = [threading.Thread(target=work, args=(films[k::2],)) for k in range(2)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not errors
