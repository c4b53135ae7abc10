"""Calls of other threads while one thread traces: film downloads, seeding and the image
calls use the engine's stream without its lock; checkpoints, new scenes and the program's
own transfers make synchronous copies. The tracing thread makes a new graph for every trace
here (setting the tuning drops the last one). Every result equals the one the same call
gives alone. Exact equality: no tolerance."""
import threading

import numpy as np
import pytest
import torch

import goodphotons_amd as gp
from goodphotons_amd import abi, scenes

pytestmark = pytest.mark.gpu


def test_calls_beside_the_making_of_graphs(gplib, tmp_path):
    sd = scenes.cornell_c0(96)
    gs = gp.GpuScene(sd, gplib)
    saved = gplib.tuning()
    n = 300_000
    films = [gp.Film(96, 96, max_photons=4 * n, lib=gplib) for _ in range(4)]
    try:
        for k, f in enumerate(films):
            gp.trace(gs, sd.camera, f, n, seed_base=k * n, max_depth=6)
        alone = [f.download() for f in films]
        raw = films[1].raw()
        lin, img = films[2].to_linear(n), films[3].tonemap(n)

        def trace():
            gplib.set_tuning(queue_capacity=1 << 16)
            f = gp.Film(96, 96, max_photons=n, lib=gplib)
            _, st = gp.trace(gs, sd.camera, f, n, seed_base=99, max_depth=6)
            words = f.raw()[0]
            f.close()
            return words, [getattr(st, k) for k in ("photons", "segments", "connections", "splats")]

        want = trace()
        done, bad = threading.Event(), []

        def side(k):
            try:
                while not done.is_set():
                    x, h = films[k].download()
                    ok = np.array_equal(x, alone[k][0]) and np.array_equal(h, alone[k][1])
                    films[k].save_checkpoint(str(tmp_path / f"film{k}"), n)
                    gp.GpuScene(sd, gplib, builder=("host", "device")[k & 1]).close()
                    ok = ok and np.array_equal(torch.from_numpy(x).cuda().cpu().numpy(), x)
                    if k == 0:
                        f = gp.Film(96, 96, max_photons=4 * n, lib=gplib)
                        f.seed(gs, sd.camera, n, x, h, max_depth=6)
                        ok = ok and np.array_equal(f.download_hits(), h)
                        f.close()
                    if k == 1:
                        ok = ok and np.array_equal(films[1].raw()[0], raw[0])
                    if k == 2:
                        ok = ok and np.array_equal(films[2].to_linear(n), lin)
                    if k == 3:
                        got = films[3].tonemap(n)
                        ok = ok and np.array_equal(got[0], img[0]) and got[1:] == img[1:]
                    if not ok:
                        bad.append(k)
                        return
            except gp.GpError as e:
                bad.append((k, str(e)))

        threads = [threading.Thread(target=side, args=(k,)) for k in range(4)]
        for t in threads:
            t.start()
        try:
            got = [trace() for _ in range(20)]
        finally:
            done.set()
            for t in threads:
                t.join()
        assert not bad
        assert all(np.array_equal(w, want[0]) and c == want[1] for w, c in got)
    finally:
        gplib.set_tuning(**{k: getattr(saved, k) for k, _ in abi.Tuning._fields_})
        for f in films:
            f.close()
        gs.close()
