"""The device builder's box levels, heights and input checks at the sizes where they can go
wrong: a triangle or two past a leaf, one below, at and above the 512 leaves a workgroup
folds and its square, and inputs that must be refused."""
import numpy as np
import pytest

import goodphotons_amd as gp
from goodphotons_amd import scenes
from tests.parity import seeded_rays

pytestmark = pytest.mark.gpu


def _first(sd, k):
    return scenes.SceneData(f"{sd.name}_{k}", sd.verts[:k].copy(), sd.mat_ids[:k].copy(), sd.materials,
                            sd.emitters, sd.camera)


@pytest.mark.parametrize("k", [1, 5, 6, 511, 512, 513, 1023, 1025, 262143, 262145])
def test_closest_hits_equal_the_host_trees(gplib, k):
    sd = _first(scenes.soup(300_000, 5, res=32), k)
    rays = seeded_rays(sd, 20_000, k)
    host, dev = gp.GpuScene(sd, gplib), gp.GpuScene(sd, gplib, builder="device")
    hp, ht = host.closest_hit(rays)
    dp, dt = dev.closest_hit(rays)
    # equal distances bit for bit: a hit does not depend on the tree, a lost box loses hits
    assert np.array_equal(ht, dt)
    assert np.mean(hp != dp) < 1e-4      # only exact ties may name another triangle
    assert (k == 1) or dev.info()["bvh_depth"] >= np.ceil(np.log2(k / 4))


@pytest.mark.parametrize("at", [0, 299, 700])
@pytest.mark.parametrize("what", ["material_low", "material_high", "nan", "inf"])
def test_bad_triangles_are_refused(gplib, what, at):
    sd = _first(scenes.soup(1000, 5, res=32), 701)
    if what.startswith("material"):
        sd.mat_ids[at] = -1 if what.endswith("low") else len(sd.materials)
    else:
        sd.verts[at].reshape(-1)[4] = np.nan if what == "nan" else -np.inf
    with pytest.raises(gp.GpError, match="material id" if what.startswith("material") else "non-finite"):
        gp.GpuScene(sd, gplib, builder="device")
