"""Depth limits far beyond the longest path, and paths longer than a chunk of iterations.

A trace that fits the queue looks for its end every iters_per_graph iterations, one that
flies in a single kernel reports the iterations that the wavefront would have run, and both
trace the photons of a trace that is refilled. Exact equality: no tolerance."""
import numpy as np
import pytest

import goodphotons_amd as gp
from goodphotons_amd import abi, scenes

pytestmark = pytest.mark.gpu
KEYS = ("photons", "segments", "connections", "splats", "direct_connections")


def _trace(lib, gs, sd, n, depth, **tuning):
    saved = lib.tuning()
    try:
        lib.set_tuning(**tuning)
        f = gp.Film(sd.camera.res_x, sd.camera.res_y, max_photons=n, lib=lib)
        e, st = gp.trace(gs, sd.camera, f, n, seed_base=3, max_depth=depth)
        words = f.raw()[0]
        f.close()
        return words, e.as_dict(), {k: getattr(st, k) for k in KEYS}, st.iterations
    finally:
        lib.set_tuning(**{k: getattr(saved, k) for k, _ in abi.Tuning._fields_})


@pytest.mark.parametrize("make", [scenes.caustics_c1, scenes.mirror_box, scenes.glossy_box],
                         ids=["glass", "mirror", "glossy"])
@pytest.mark.parametrize("n", [700, 100_003])
@pytest.mark.parametrize("chunk", [2, 8, 32])
def test_ends_with_the_last_path(gplib, make, n, chunk):
    sd = make(40)
    gs = gp.GpuScene(sd, gplib)
    try:
        a = _trace(gplib, gs, sd, n, 250, iters_per_graph=chunk)
        b = _trace(gplib, gs, sd, n, 250, iters_per_graph=chunk, profile=1)      # no flight
        c = _trace(gplib, gs, sd, n, 250, iters_per_graph=chunk, queue_capacity=4096)
        assert np.array_equal(a[0], b[0]) and a[1:] == b[1:]
        assert np.array_equal(a[0], c[0]) and a[1:3] == c[1:3]
        assert a[3] == 250 or (a[1]["residual"] == 0 and a[3] % chunk == 0)
        if a[3] > chunk:   # a chunk earlier paths were alive
            assert _trace(gplib, gs, sd, n, a[3] - chunk, iters_per_graph=chunk)[1]["residual"] > 0
    finally:
        gs.close()


def test_chunks_of_a_trace_that_fits_the_queue(gplib):
    # 40 iterations on the wavefront (too many photons to fly) in chunks of 8 and of 64,
    # against the same photons refilled through a small queue
    sd = scenes.caustics_c1(40)
    gs = gp.GpuScene(sd, gplib)
    n = 900_001
    try:
        a = _trace(gplib, gs, sd, n, 40, iters_per_graph=8)
        b = _trace(gplib, gs, sd, n, 40, iters_per_graph=64)
        c = _trace(gplib, gs, sd, n, 40, queue_capacity=1 << 14)
        for x in (b, c):
            assert np.array_equal(a[0], x[0]) and a[1:3] == x[1:3]
        assert a[3] > 8 and b[3] == 40
    finally:
        gs.close()
