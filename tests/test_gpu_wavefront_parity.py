"""The small films of the oracle comparison through the wavefront's kernels: traces of so
few photons fly in one kernel by themselves, so kernel timing (which keeps them from flying)
and a small queue (refills, replayed graphs) send them there. Same bounds."""
import pytest

from goodphotons_amd import abi
from tests import test_gpu_parity as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("route", [dict(profile=1), dict(queue_capacity=1 << 14)], ids=["one_refill", "refilled"])
@pytest.mark.parametrize("name,builder,n,depth,rr", P.FILM_CASES, ids=[c[0] for c in P.FILM_CASES])
def test_film_matches_oracle(gplib, orc, name, builder, n, depth, rr, route):
    saved = gplib.tuning()
    try:
        gplib.set_tuning(**route)
        P.test_film_matches_oracle(gplib, orc, name, builder, n, depth, rr)
    finally:
        gplib.set_tuning(**{k: getattr(saved, k) for k, _ in abi.Tuning._fields_})
