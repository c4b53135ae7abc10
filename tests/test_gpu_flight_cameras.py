"""Several cameras in flight, up to the most photons that fly with them in a small tree (box)
and in a deep one (glass sphere), and one photon more (on the wavefront): each as
test_gpu_flight compares the two routes. Exact equality: no tolerance."""
import pytest

from goodphotons_amd import scenes
from tests import test_gpu_flight as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cams,n", [(2, 139022), (3, 75674), (4, 49152), (6, 26754), (6, 26755), (7, 5003)])
def test_small_tree(gplib, cams, n):
    F._both(gplib, scenes.cornell_c0(32), n, cams=cams, depth=8)


@pytest.mark.parametrize("depth,cams,n", [(8, 3, 235929), (8, 6, 79776), (8, 6, 79777), (8, 16, 14336), (8, 16, 14337),
                                          (16, 16, 28672), (16, 16, 28673),
                                          (5, 3, 134532), (5, 6, 11891), (5, 6, 11892), (5, 16, 384)])
def test_deep_tree(gplib, depth, cams, n):
    F._both(gplib, scenes.caustics_c1(32), n, cams=cams, depth=depth)
