"""Ray binning on a server: it is a tuning, which is refused while jobs run and taken between
two drains of the same server; the films are those of a server that never bins. Exact
equality: no tolerance."""
import numpy as np
import pytest

import goodphotons_amd as gp
from goodphotons_amd import abi, scenes

pytestmark = pytest.mark.gpu


def test_binning_switched_between_drains(gplib):
    specs = [(scenes.cornell_c0(48), 1 << 17, 8, 3, 11), (scenes.icosphere_c2(4, 32), 1 << 15, 12, 0, 66)]
    gss = [gp.GpuScene(sd, gplib) for sd, *_ in specs]
    saved = gplib.tuning()
    res = []
    try:
        for sorts in ((0, 0, 0), (0, 1, 0)):
            gplib.set_tuning(queue_capacity=1 << 14, ray_sort=sorts[0])
            srv = gp.Server(hbm_budget_bytes=1 << 30, max_live_jobs=8, lib=gplib)
            got = []
            for k, sort in enumerate(sorts):
                gplib.set_tuning(ray_sort=sort)
                ids = [srv.submit(gs, sd.camera, n, seed_base=seed + k, max_depth=depth, rr_depth=rr)
                       for (sd, n, depth, rr, seed), gs in zip(specs, gss)]
                srv.step(max_iterations=4)
                with pytest.raises(gp.GpError):
                    gplib.set_tuning(ray_sort=1 - sort)
                srv.step()
                got += [srv.take(j, sd.camera.res_x, sd.camera.res_y) for j, (sd, *_) in zip(ids, specs)]
            srv.close()
            res.append(got)
        for (ra, xa, ha), (rb, xb, hb) in zip(*res):
            assert np.array_equal(xa, xb) and np.array_equal(ha, hb)
            assert ra.stats.segments == rb.stats.segments and ra.stats.splats == rb.stats.splats
    finally:
        gplib.set_tuning(**{k: getattr(saved, k) for k, _ in abi.Tuning._fields_})
        for gs in gss:
            gs.close()
