"""Test infrastructure only: the engine's host code through the emulation build (child
process, started with the AddressSanitizer runtime preloaded by
tests/test_emulated_engine.py). argv: the scenario. Prints JSON on the last line."""
import ctypes as C
import json
import os
import sys
import tempfile
import threading

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path.insert(0, ROOT)

import goodphotons_amd as gp  # noqa: E402
from goodphotons_amd import scenes  # noqa: E402

lib = gp.Library(os.environ["EMU_LIB"])
emu = lib.lib
emu.emu_launches.restype = C.c_longlong
emu.emu_launches.argtypes = [C.c_char_p]
emu.emu_stream_syncs.restype = C.c_longlong
emu.emu_event_records.restype = C.c_longlong
KEYS = ("photons", "segments", "connections", "splats")


def counts(st):
    return [int(getattr(st, k)) for k in KEYS]


def film_of(sd, n):
    return gp.Film(sd.camera.res_x, sd.camera.res_y, max_photons=n, lib=lib)


def graph():
    """A film is downloaded and saved, another seeded and a scene created by a second thread
    while the first makes the graph of a trace that is refilled."""
    lib.set_tuning(queue_capacity=4096, grid_waves_per_cu=4, iters_per_graph=2)
    sd = scenes.cornell_c0(32)
    gs = gp.GpuScene(sd, lib)
    other = film_of(sd, 1000)
    gp.trace(gs, sd.camera, other, 1000, max_depth=4)
    xyz, hits = other.download()
    seen = {}

    def side():
        try:
            x, h = other.download()
            fresh = film_of(sd, 1000)
            fresh.seed(gs, sd.camera, 1000, xyz, hits, max_depth=4)
            y, g = fresh.download()
            gp.GpuScene(sd, lib).close()
            with tempfile.TemporaryDirectory() as d:
                other.save_checkpoint(os.path.join(d, "film"), 1000)
            seen["same"] = bool(np.array_equal(x, xyz) and np.array_equal(h, hits) and np.array_equal(g, hits))
        except gp.GpError as e:
            seen["error"] = str(e)

    def during():
        t = threading.Thread(target=side)
        t.start()
        t.join()

    cb = C.CFUNCTYPE(None)(during)
    emu.emu_on_graph(cb)
    n = 5001
    got = []
    for _ in range(2):   # made, then replayed
        f = film_of(sd, n)
        _, st = gp.trace(gs, sd.camera, f, n, max_depth=4)
        got.append((f.raw()[0], counts(st)))
    return {"seen": seen, "counts": got[0][1], "hits": got[0][0][:, 3].tolist(),
            "same": bool(np.array_equal(got[0][0], got[1][0]) and got[0][1] == got[1][1])}


def nest(n):
    """n triangles, each half the size of the last, nested into a corner: a tree that grows
    by about a level a triangle."""
    sd = scenes.soup(n, 4, res=8)
    corner = np.array([1, 0, 0, 1.2, 0.2, 0, 1, 0.2, 0.2])
    v = np.array(sd.verts, np.float32).reshape(-1, 9)
    v[:n] = corner[None] * (0.4 * 0.5 ** np.arange(n))[:, None] + 0.5
    sd.verts = v.reshape(np.shape(sd.verts))
    return sd


def reshape():
    """A server that is given a deeper tree at every step, with chunks in flight (EMU_ASYNC:
    the emulator aborts if a graph is destroyed under one); then steps that change nothing."""
    lib.set_tuning(queue_capacity=4096, grid_waves_per_cu=4, iters_per_graph=2, lds_stack=12)
    depths, same = [], True
    sds = [nest(n) for n in (8, 12, 14, 16, 18, 20, 22, 24, 28, 32)]
    gss = [gp.GpuScene(sd, lib, builder="device") for sd in sds]
    srv = gp.Server(lib=lib)
    ids = []
    for sd, gs in zip(sds, gss):
        depths.append(gs.info()["bvh_depth"])
        ids.append(srv.submit(gs, sd.camera, 64, max_depth=3))
        srv.step(max_iterations=2)
    srv.step()
    for sd, gs, j in zip(sds, gss, ids):
        r, x, h = srv.take(j, 8, 8)
        xa, ha, _, _ = gp.render_forward(gs, sd.camera, 64, max_depth=3)
        same = same and r.status == 0 and bool(np.array_equal(x, xa) and np.array_equal(h, ha))
    # steps of one scene whose stack needs 9..24 entries
    waits = []
    for k in (1, 5):
        sd, gs = sds[k], gss[k]
        j = srv.submit(gs, sd.camera, 64, max_depth=4)
        srv.step(max_iterations=2)
        before = emu.emu_stream_syncs()
        srv.step(max_iterations=2)
        waits.append(emu.emu_stream_syncs() - before)
        srv.step()
        srv.take(j, 8, 8)
    srv.close()
    return {"depths": depths, "same": same, "waits": waits}


def deep():
    """Paths that end long before the depth limit: iterations of a trace on the wavefront
    (mirrors) and of one that flies, and what is still alive an iteration chunk earlier."""
    lib.set_tuning(queue_capacity=4096, grid_waves_per_cu=4, iters_per_graph=4)
    out = {}
    for name, sd in (("mirror", scenes.mirror_box(8)), ("box", scenes.cornell_c0(8))):
        gs = gp.GpuScene(sd, lib)

        def run(depth):
            f = film_of(sd, 64)
            e, st = gp.trace(gs, sd.camera, f, 64, max_depth=depth)
            return [int(st.iterations), float(e.residual), counts(st)]

        flown = emu.emu_launches(b"k_flight")
        whole = run(60)
        out[name] = {"whole": whole, "before": run(whole[0] - 4) if whole[0] > 4 else None,
                     "flown": emu.emu_launches(b"k_flight") - flown}
        lib.set_tuning(profile=1)
        out[name]["wavefront"] = run(60)
        lib.set_tuning(profile=0)
    return out


def autotune():
    """Kernels that gp_autotune times with a budget small enough to fly, and a trace of it."""
    sd = scenes.cornell_c0(8)
    gs = gp.GpuScene(sd, lib)
    lib.set_tuning(queue_capacity=4096, grid_waves_per_cu=4)
    best = gp.abi.Tuning()
    p = gp.trace_params(32, max_depth=1)
    lib.check(emu.gp_autotune(gs.h, C.byref(sd.camera), C.byref(p), C.byref(best)))
    out = {"flown": emu.emu_launches(b"k_flight"), "extended": emu.emu_launches(b"k_extend"),
           "installed": lib.tuning().queue_capacity == best.queue_capacity}
    lib.set_tuning(queue_capacity=4096)
    gp.trace(gs, sd.camera, film_of(sd, 32), 32, max_depth=1)
    out["trace_flown"] = emu.emu_launches(b"k_flight") - out["flown"]
    return out


def views(sd, count):
    c = sd.camera
    return [c] + [scenes.camera((c.eye[0] + 0.02 * k, c.eye[1], c.eye[2]), tuple(c.target), tuple(c.up),
                                c.fov_y_deg, 9 + k, 11) for k in range(1, count)]


def flight():
    """Traces that fly, with the stack in LDS and spilling, one camera and three, against
    the wavefront's kernels (kernel timing on) for the same photons."""
    out = {}
    for name, sd, n, cams, lds in (("c1_8", scenes.caustics_c1(32), 1500, 1, 8),
                                   ("c1_12", scenes.caustics_c1(32), 1500, 1, 12),
                                   ("c0_cams", scenes.cornell_c0(32), 590, 3, 12)):
        gs, cs, got = gp.GpuScene(sd, lib), views(sd, cams), []
        for profile in (0, 1):
            lib.set_tuning(queue_capacity=4096, grid_waves_per_cu=4, lds_stack=lds, profile=profile)
            films = [gp.Film(c.res_x, c.res_y, max_photons=n, lib=lib) for c in cs]
            before = emu.emu_launches(b"k_flight")
            e, st = gp.trace_shared(gs, cs, films, n, max_depth=8)
            got.append([[f.raw()[0].tolist() for f in films], e.as_dict(), counts(st)])
            out.setdefault(name, {}).setdefault("flown", []).append(emu.emu_launches(b"k_flight") - before)
        out[name].update(same=got[0] == got[1], counts=got[0][2], hits=[w[3] for w in got[0][0][0]])
    return out


def sort():
    """Sorted emission (a build with low thresholds) of a trace with two lights, and of two
    jobs on a server, against traces of the same photons that fly."""
    lib.set_tuning(queue_capacity=4096, grid_waves_per_cu=4, iters_per_graph=2)
    sd = scenes.cornell_c0(16)
    sd.emitters.append(scenes.quad_emitter((0.3, 0.9, 0.3), (0.2, 0, 0), (0, 0, 0.2), (0, -1, 0),
                                           sd.emitters[0].spd, collimated=True, beam=(0, -1, 0)))
    gs = gp.GpuScene(sd, lib)
    n = 2003
    whole, parts = film_of(sd, n), film_of(sd, n)
    _, st = gp.trace(gs, sd.camera, whole, n, max_depth=4)
    sorts = emu.emu_launches(b"k_emit_perm")
    sums = np.zeros(len(KEYS), np.int64)
    for at in range(0, n, 700):
        _, sp = gp.trace(gs, sd.camera, parts, min(700, n - at), seed_base=at, max_depth=4)
        sums += counts(sp)
    out = {"sorts": sorts, "more_sorts": emu.emu_launches(b"k_emit_perm") - sorts, "counts": counts(st),
           "trace": bool(np.array_equal(whole.raw()[0], parts.raw()[0]) and counts(st) == sums.tolist())}
    srv = gp.Server(lib=lib)
    srv.submit(gs, sd.camera, 1203, max_depth=1)
    before = emu.emu_launches(b"k_emit_perm")
    srv.step()
    out["one_job_sorts"] = emu.emu_launches(b"k_emit_perm") - before
    jobs = [(gs, sd, 1203, 7), (gs, sd, 350, 9000)]
    ids = [srv.submit(g, d.camera, k, seed_base=s, max_depth=2) for g, d, k, s in jobs]
    srv.step()
    same = True
    for j, (g, d, k, s) in zip(ids, jobs):
        r, x, h = srv.take(j, 16, 16)
        f = film_of(d, k)
        for at in range(0, k, 700):
            gp.trace(g, d.camera, f, min(700, k - at), seed_base=s + at, max_depth=2)
        hs = f.download_hits()
        same = same and r.status == 0 and bool(np.array_equal(h, hs))
    srv.close()
    out["server"] = same
    out["two_job_sorts"] = emu.emu_launches(b"k_emit_perm") - sorts
    return out


def refill():
    """Which traces sort their emission (a build with low thresholds): photons that the queue
    of 4096 slots holds at once, and more than it holds; the films against traces that fly."""
    lib.set_tuning(queue_capacity=4096, grid_waves_per_cu=4, iters_per_graph=2)
    sd = scenes.cornell_c0(16)
    gs = gp.GpuScene(sd, lib)
    out = {}
    for n in (3200, 6100):
        whole, parts = film_of(sd, n), film_of(sd, n)
        before = emu.emu_launches(b"k_emit_perm")
        gp.trace(gs, sd.camera, whole, n, max_depth=2)
        sorts = emu.emu_launches(b"k_emit_perm") - before
        for at in range(0, n, 700):
            gp.trace(gs, sd.camera, parts, min(700, n - at), seed_base=at, max_depth=2)
        out[n] = [sorts, bool(np.array_equal(whole.raw()[0], parts.raw()[0]))]
    return out


def route():
    """Which traces fly (1024 resident lanes): small tree or deep, segments, cameras, photons."""
    lib.set_tuning(queue_capacity=4096, grid_waves_per_cu=4)
    out = []
    for deep, sd, runs in ((0, scenes.cornell_c0(8), ((1, 1, 1536), (1, 1, 1537), (1, 2, 543), (1, 2, 544), (1, 6, 104),
                                                      (1, 6, 105), (1, 7, 40), (1, 16, 40), (12, 6, 156), (12, 6, 157))),
                           (1, nest(24), ((2, 1, 1536), (2, 1, 1537), (2, 3, 525), (2, 3, 526), (2, 6, 46), (2, 6, 47),
                                          (8, 6, 311), (8, 6, 312), (8, 16, 55), (8, 16, 57), (20, 16, 111), (20, 16, 113)))):
        gs = gp.GpuScene(sd, lib, builder="device")
        for depth, cams, n in runs:
            cs = views(sd, cams)
            films = [gp.Film(c.res_x, c.res_y, max_photons=n, lib=lib) for c in cs]
            before = emu.emu_launches(b"k_flight")
            gp.trace_shared(gs, cs, films, n, max_depth=depth)
            out.append([deep, depth, cams, n, emu.emu_launches(b"k_flight") - before])
    return out


def seeding():
    """Events that seeding a film records (65536 pixels fill a staging slot), and whether its
    words are the rounded doubles."""
    sd0, out = scenes.cornell_c0(8), []
    gs = gp.GpuScene(sd0, lib)
    for rx, ry in ((1, 1), (16, 16), (1024, 64), (4099, 16)):
        cam = sd0.with_camera_res(rx, ry).camera
        rng = np.random.default_rng(rx)
        h = np.floor(rng.uniform(0, 50, rx * ry))
        x = rng.uniform(0, 1e12, (rx * ry, 3))
        f = gp.Film(rx, ry, max_photons=1000, lib=lib)
        before = emu.emu_event_records()
        f.seed(gs, cam, 1000, x, h, max_depth=4)
        events = emu.emu_event_records() - before
        w, scale = f.raw()
        out.append([rx * ry, events, bool(np.array_equal(w[:, :3], np.rint(x * scale).astype(np.int64))
                                          and np.array_equal(w[:, 3], h) and w[:, :3].any())])
        f.close()
    return out


def totals():
    """Launches of the conversion kernel by film size, and whether the doubles are the words."""
    sd0, out = scenes.cornell_c0(8), []
    gs = gp.GpuScene(sd0, lib)
    for rx, ry in ((1, 1), (32, 32), (64, 48), (439, 7)):
        f = gp.Film(rx, ry, max_photons=200, lib=lib)
        gp.trace(gs, sd0.with_camera_res(rx, ry).camera, f, 200, max_depth=2)
        w, scale = f.raw()
        before = emu.emu_launches(b"k_film_totals")
        x, h = f.download()
        only = f.download_hits()
        out.append([rx * ry, emu.emu_launches(b"k_film_totals") - before,
                    bool(np.array_equal(x, w[:, :3] * (1.0 / scale)) and np.array_equal(h, w[:, 3])
                         and np.array_equal(only, h) and h.any())])
    return out


def films():
    """Films of a server's jobs of several sizes, with scratch to convert them in and without
    (allocations fail after those of the films), against the same traces."""
    lib.set_tuning(queue_capacity=4096, grid_waves_per_cu=4, iters_per_graph=2)
    sd0, out = scenes.cornell_c0(8), []
    gs = gp.GpuScene(sd0, lib)
    cams = [sd0.with_camera_res(*r).camera for r in ((9, 5), (160, 110), (128, 128), (16385, 1))]
    emu.emu_fail_async_allocations.argtypes = [C.c_longlong]
    for allowed in (-1, len(cams)):
        srv = gp.Server(lib=lib)
        emu.emu_fail_async_allocations(allowed)
        before = emu.emu_launches(b"k_film_totals")
        ids = [srv.submit(gs, c, 64, seed_base=7 * k, max_depth=2) for k, c in enumerate(cams)]
        srv.step()
        converted = emu.emu_launches(b"k_film_totals") - before
        emu.emu_fail_async_allocations(-1)
        same = True
        for k, (j, c) in enumerate(zip(ids, cams)):
            r, x, h = srv.take(j, c.res_x, c.res_y)
            xa, ha, _, _ = gp.render_forward(gs, c, 64, seed_base=7 * k, max_depth=2)
            same = same and r.status == 0 and bool(np.array_equal(x, xa) and np.array_equal(h, ha))
        srv.close()
        out.append([converted, same])
    return out


def chunks():
    """Iterations that a server runs for small jobs in chunks of two (EMU_ASYNC), drained at
    once and in steps, and for one that is refilled; films against the same traces."""
    lib.set_tuning(queue_capacity=4096, grid_waves_per_cu=4, iters_per_graph=2)
    sd = scenes.cornell_c0(8)
    gs, out = gp.GpuScene(sd, lib), []
    for jobs, depth, step in (((300,), 3, 0), ((300,), 3, 2), ((200, 500), 2, 0), ((4500,), 2, 0)):
        srv = gp.Server(lib=lib)
        before = emu.emu_launches(b"k_schedule")
        ids = [srv.submit(gs, sd.camera, n, seed_base=1000 * k, max_depth=depth) for k, n in enumerate(jobs)]
        for _ in range(4 if step else 0):
            srv.step(max_iterations=step)
        srv.step()
        ran = emu.emu_launches(b"k_schedule") - before
        same = True
        for k, (j, n) in enumerate(zip(ids, jobs)):
            r, x, h = srv.take(j, 8, 8)
            xa, ha, _, st = gp.render_forward(gs, sd.camera, n, seed_base=1000 * k, max_depth=depth)
            same = same and r.status == 0 and bool(np.array_equal(h, ha)) and r.stats.segments == st["segments"]
        srv.close()
        out.append([ran, same])
    return out


def probes():
    """Events of an occlusion call just past the directly answered ones, and its answers
    against those."""
    sd = scenes.cornell_c0(8)
    gs = gp.GpuScene(sd, lib)
    n = 65600
    rng = np.random.default_rng(3)
    rays = np.concatenate([rng.uniform(-0.1, 1.1, (n, 3)), rng.normal(size=(n, 3))], 1).astype(np.float32)
    tmax = rng.uniform(0.1, 1.0, n).astype(np.float32)
    before = emu.emu_event_records()
    whole = gs.any_hit(rays, tmax)
    events = emu.emu_event_records() - before
    ends = [gs.any_hit(rays[:300], tmax[:300]), gs.any_hit(rays[-300:], tmax[-300:])]
    return {"events": events, "same": bool(np.array_equal(whole[:300], ends[0]) and np.array_equal(whole[-300:], ends[1])),
            "hit": int(whole.sum())}


print(json.dumps({"probes": probes, "chunks": chunks, "films": films, "totals": totals, "seeding": seeding, "route": route, "flight": flight, "sort": sort, "refill": refill, "autotune": autotune, "graph": graph, "reshape": reshape, "deep": deep}[sys.argv[1]]()))
