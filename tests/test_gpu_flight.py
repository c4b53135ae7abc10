"""Small traces fly in one kernel; the same photons through the wavefront's kernels (kernel
timing switched on selects them) give the same film words, ledger and counters, bit for bit:
one photon, counts around the lanes of a wave and of the launch, more photons than lanes,
up to the last count that flies; several cameras; every stack depth; each number of
wavelengths."""
import numpy as np
import pytest

import goodphotons_amd as gp
from goodphotons_amd import scenes

pytestmark = pytest.mark.gpu
KEYS = ("photons", "segments", "connections", "splats", "direct_connections")


def _cams(sd, count):
    c = sd.camera
    return [c] + [scenes.camera((c.eye[0] + 0.02 * k, c.eye[1], c.eye[2]), tuple(c.target), tuple(c.up),
                                c.fov_y_deg, 17 + k, 23) for k in range(1, count)]


def _both(lib, sd, n, cams=1, hero=4, depth=8, rr=0, **tuning):
    scene, views, got = gp.GpuScene(sd, lib), _cams(sd, cams), []
    before = lib.tuning()
    keep = {k: getattr(before, k) for k in ("profile", "lds_stack", "queue_capacity")}
    try:
        for profile in (0, 1):
            lib.set_tuning(profile=profile, **tuning)
            films = [gp.Film(c.res_x, c.res_y, max_photons=n, lib=lib) for c in views]
            e, st = gp.trace_shared(scene, views, films, n, seed_base=77, hero_c=hero, max_depth=depth, rr_depth=rr)
            assert (sum(st.as_dict()["kernel_launches"]) > 0) == bool(profile)
            got.append(([f.raw()[0] for f in films], e.as_dict(), {k: getattr(st, k) for k in KEYS}))
    finally:
        lib.set_tuning(**keep)
    (fa, ea, sa), (fb, eb, sb) = got
    assert sa == sb and sa["photons"] == n and ea == eb
    assert all(np.array_equal(a, b) for a, b in zip(fa, fb))


@pytest.mark.parametrize("n", [1, 3, 63, 3071, 3073, 6145, 98305, 262143, 262145, 393216])
def test_photon_counts(gplib, n):
    _both(gplib, scenes.cornell_c0(48), n, rr=3)


@pytest.mark.parametrize("hero", [1, 2, 3, 4])
@pytest.mark.parametrize("make", [scenes.caustics_c1, scenes.glossy_box], ids=["glass", "glossy"])
def test_materials_and_wavelengths(gplib, make, hero):
    _both(gplib, make(40), 30011, hero=hero, depth=16)


@pytest.mark.parametrize("cams,n", [(2, 40009), (6, 130003), (16, 5003)])
def test_cameras(gplib, cams, n):
    _both(gplib, scenes.caustics_c1(32), n, cams=cams, depth=16)


@pytest.mark.parametrize("lds", [8, 12, 16, 24, 32])
@pytest.mark.parametrize("tris", [5, 60_000])
def test_stack_depths(gplib, tris, lds):
    _both(gplib, scenes.soup(tris, 4, res=24), 20011, lds_stack=lds)
