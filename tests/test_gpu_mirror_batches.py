"""Connections through mirror planes are listed and traced 64 at a time: the counts equal the
oracle's and the film its float rounding, for photon counts that leave part of a batch over,
with several cameras (against each camera alone, bit for bit) and every stack depth."""
import numpy as np
import pytest

import goodphotons_amd as gp
from goodphotons_amd import scenes
from tests.parity import image_metrics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 64, 1025, 50021])
def test_counts_equal_the_oracles(gplib, orc, n):
    sd = scenes.mirror_box(24)
    x, h, _, st = gp.render_forward(gp.GpuScene(sd, gplib), sd.camera, n, hero_c=4, max_depth=8)
    cx, ch, _, cst = orc.render(orc.scene(sd), sd.camera, n, hero_c=4, max_bounce=8, threads=8)
    assert (st["segments"], st["connections"], st["splats"]) == (cst["segments"], cst["connections"], cst["splats"])
    assert np.array_equal(h, ch)
    # float32 transport against the double oracle: 2^-24 per operation, about 100 of them a splat
    assert image_metrics(x, cx, n, n, res=(24, 24))["rel_rmse_max"] < 1e-5


@pytest.mark.parametrize("lds", [8, 12, 32])
def test_cameras_together_and_alone(gplib, lds):
    sd = scenes.mirror_box(24)
    c = sd.camera
    cams = [c] + [scenes.camera((c.eye[0] + 0.05 * k, c.eye[1], c.eye[2]), tuple(c.target), tuple(c.up),
                                c.fov_y_deg, 20 + 3 * k, 31) for k in (1, 2)]
    scene, n, before = gp.GpuScene(sd, gplib), 30011, gplib.tuning().lds_stack
    try:
        gplib.set_tuning(lds_stack=lds)
        both, _, st = gp.render_forward_shared(scene, cams, n, hero_c=4, max_depth=8)
        for (x, h), cam in zip(both, cams):
            ax, ah, _, _ = gp.render_forward(scene, cam, n, hero_c=4, max_depth=8)
            assert np.array_equal(h, ah)
            # the films' scales depend on their own camera only
            assert np.array_equal(x, ax)
    finally:
        gplib.set_tuning(lds_stack=before)
