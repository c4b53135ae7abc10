"""Several cameras in flight, up to the most photons that fly with them, and one photon more
(on the wavefront): each as test_gpu_flight compares the two routes. Exact equality: no
tolerance."""
import pytest

from goodphotons_amd import scenes
from tests import test_gpu_flight as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make", [scenes.cornell_c0, scenes.caustics_c1], ids=["box", "glass"])
@pytest.mark.parametrize("cams,n", [(2, 139022), (3, 75674), (4, 49152), (6, 26754), (6, 26755), (7, 5003)])
def test_cameras_in_flight(gplib, make, cams, n):
    F._both(gplib, make(32), n, cams=cams, depth=9)
