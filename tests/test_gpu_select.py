"""The exposure anchor is the exact order statistic of the film's channels: films around the
sizes of a histogram's workgroups, of equal pixels, of black pixels, and of values over many
powers of two, against the sorted values of the downloaded film, bit for bit; the linear image
at sizes around a pinned slot; both tone-map entry points."""
import numpy as np
import pytest

import goodphotons_amd as gp
from goodphotons_amd import scenes

pytestmark = pytest.mark.gpu
M = np.array([[3.2406, -1.5372, -0.4986], [-0.9689, 1.8758, 0.0415], [0.0557, -0.2040, 1.0570]])


def _ybar_sum():
    w = np.arange(360.0, 831.0)

    def lobe(mu, a, b):
        t = (w - mu) * np.where(w < mu, a, b)
        return np.exp(-0.5 * t * t)
    s = 0.0
    for v in 0.821 * lobe(568.8, 0.0213, 0.0247) + 0.286 * lobe(530.9, 0.0613, 0.0322):
        s += v
    return s


@pytest.mark.parametrize("size", [(1, 1), (2, 1), (16, 32), (27, 19), (511, 513), (417, 419), (1000, 700)], ids=str)
@pytest.mark.parametrize("kind", ["spread", "equal", "black"])
def test_anchor_and_linear(gplib, size, kind):
    sd = scenes.cornell_c0(16).with_camera_res(*size)
    scene, n, photons = gp.GpuScene(sd, gplib), size[0] * size[1], 1 << 20
    film = gp.Film(*size, max_photons=photons, lib=gplib)
    r = np.random.default_rng([n, len(kind)])
    scale = scene.info()["total_power"] * photons * 0.02
    lum = {"spread": np.exp2(r.uniform(-30.0, 0.0, n)), "equal": np.full(n, 0.25), "black": np.zeros(n)}[kind]
    film.seed(scene, sd.camera, photons, lum[:, None] * scale * np.array([0.95, 1.0, 1.09]), np.zeros(n))
    xyz, _ = film.download()
    c = xyz * (1.0 / (photons * _ybar_sum()))
    # the library's order of operations, without contraction
    lin = np.stack([(m[0] * c[:, 0] + m[1] * c[:, 1]) + m[2] * c[:, 2] for m in M], axis=1)
    got = film.to_linear(photons).reshape(-1, 3)
    # one ulp of float for the host's own sum of ybar
    assert np.allclose(got, lin, rtol=2.0 ** -23, atol=2.0 ** -23 * np.abs(lin).max())
    top = np.sort(np.maximum(lin.max(axis=1), 0.0))[int(0.99 * (n - 1))]
    img, exposure, anchor = film.tonemap(photons, exposure_comp=1.0)
    # double arithmetic, a few roundings apart through the host's sum of ybar
    assert anchor == pytest.approx(0.9 / top if top > 0 else 1.0, rel=1e-14) and exposure == anchor
    img2, exposure2, anchor2 = film.tonemap(photons, exposure_comp=1.0, no_alloc=True)
    assert anchor2 == anchor and exposure2 == exposure and np.array_equal(img, img2)
