"""The engine's host code and the kernels that the other emulated cases do not reach, on
the CPU under AddressSanitizer (tests/emu): what the host may do to streams and graphs
while work runs on them, and which kernels a call runs.

Exact equality throughout, except where the oracle's film is compared.
"""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

from goodphotons_amd import scenes
from tests.emu import build as emu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.skipif(not emu.available(), reason="clang++ with AddressSanitizer not found")


def _run(scenario, libs, cus, preempt=0, run_async=0, variant=""):
    env = dict(os.environ)
    env.update({"LD_PRELOAD": emu.asan_runtime(), "ASAN_OPTIONS": "detect_leaks=0", "EMU_CUS": str(cus),
                "EMU_PREEMPT": str(preempt), "EMU_ASYNC": str(run_async), "EMU_LIB": libs[variant]})
    return subprocess.Popen([sys.executable, os.path.join(ROOT, "tests", "emu", "run_engine.py"), scenario],
                            stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, env=env)


# Each scenario is a child process of its own; all are started at once.
CASES = {
    "autotune": dict(cus=1),
    "graph": dict(cus=1),
    "reshape": dict(cus=1, run_async=1),
    "deep": dict(cus=1),
    "flight": dict(cus=2, preempt=3),
    "sort": dict(cus=1, variant="sort"),
    "refill": dict(cus=1, variant="refill"),
    "route": dict(cus=1),
    "seeding": dict(cus=1),
    "totals": dict(cus=1),
    "films": dict(cus=1),
    "chunks": dict(cus=1, run_async=1),
    "probes": dict(cus=1),
}
# emission sorted from 64 photons on, in traces of 1000 and on servers with 1500 in all
VARIANTS = {"": (), "sort": ("GP_EMIT_COLS=16", "GP_EMIT_ORDER_MIN=64", "GP_EMIT_ORDER_JOB_MIN=1000",
                             "GP_EMIT_ORDER_SERVER_MIN=1500"),
            "refill": ("GP_EMIT_COLS=16", "GP_EMIT_ORDER_MIN=64", "GP_EMIT_ORDER_JOB_MIN=3000",
                       "GP_EMIT_ORDER_SERVER_MIN=3500")}


@pytest.fixture(scope="module")
def runs():
    libs = {v: emu.build(v, d) for v, d in VARIANTS.items()}
    procs = {k: _run(k, libs, **kw) for k, kw in CASES.items()}
    yield procs
    for p in procs.values():
        if p.poll() is None:
            p.kill()
            p.wait()


_done = {}


def _result(runs, key):
    if key not in _done:
        out, err = runs[key].communicate(timeout=900)
        assert runs[key].returncode == 0, err[-3000:]
        _done[key] = json.loads(out.strip().splitlines()[-1])
    return _done[key]


def test_calls_of_another_thread_stay_out_of_a_graph(runs, orc):
    # film calls, synchronous ones among them, and a new scene that fall into the making of a
    # trace's graph neither fail nor end up in the graph, and the trace holds the oracle's
    # photons
    out = _result(runs, "graph")
    assert out["seen"] == {"same": True}
    assert out["same"]
    sd = scenes.cornell_c0(32)
    _, h, _, st = orc.render(orc.scene(sd), sd.camera, 5001, hero_c=4, max_bounce=4, threads=8)
    assert out["counts"] == [5001] + [st[k] for k in ("segments", "connections", "splats")]
    assert np.array_equal(np.array(out["hits"]), h)


def test_a_server_waits_for_its_chunks_before_the_engine_changes_shape_and_only_then(runs):
    # the emulator aborts where a graph is destroyed under a running chunk; a step that
    # changes nothing synchronises no stream
    out = _result(runs, "reshape")
    need = [3 * ((d + 1) // 2) for d in out["depths"]]
    assert need == sorted(need) and set(need) >= set(range(12, 37, 3))
    assert out["same"]
    assert out["waits"] == [0, 0]


@pytest.mark.parametrize("name", ["mirror", "box"])
def test_a_deep_trace_ends_with_the_chunk_that_ends_its_last_path(runs, name):
    # iters_per_graph = 4: a chunk less leaves paths alive, and a trace that flies counts
    # the iterations that the wavefront runs
    out = _result(runs, "deep")[name]
    iters, residual, counts = out["whole"]
    assert (out["flown"] > 0) == (name == "box")
    assert 4 < iters < 60 and iters % 4 == 0 and residual == 0
    assert out["before"][1] > 0
    assert out["wavefront"] == out["whole"]


def test_autotune_times_the_wavefronts_kernels_with_a_small_budget(runs):
    # 18 shapes and the sorting modes, each warmed and timed
    out = _result(runs, "autotune")
    assert out["flown"] == 0 and out["extended"] >= 2 * 19 and out["installed"]
    assert out["trace_flown"] == 1


@pytest.mark.parametrize("name", ["c1_8", "c1_12", "c0_cams"])
def test_flight_with_interleaved_lanes(runs, orc, name):
    # every access of k_flight checked: the wavefront's words, ledger and counters, and the
    # oracle's photons
    out = _result(runs, "flight")[name]
    assert out["flown"] == [1, 0] and out["same"]
    sd = scenes.cornell_c0(32) if name == "c0_cams" else scenes.caustics_c1(32)
    n = out["counts"][0]
    _, h, _, st = orc.render(orc.scene(sd), sd.camera, n, hero_c=4, max_bounce=8, threads=8)
    assert out["counts"][1] == st["segments"] and np.array_equal(np.array(out["hits"]), h)
    if name != "c0_cams":
        assert out["counts"][2:] == [st["connections"], st["splats"]]


def test_sorted_emission(runs, orc):
    # k_emit_keys, k_emit_perm and the ordered k_emit with every access checked: one sort of
    # the trace's 2003 photons of two lights, then a server with two jobs in the order; one
    # job of 1203 photons is too few for a server
    out = _result(runs, "sort")
    assert out["one_job_sorts"] == 0 and out["two_job_sorts"] > 0
    assert out["sorts"] == 1 and out["more_sorts"] == 0
    assert out["trace"] and out["server"]


def test_refills_of_a_small_queue_keep_index_order(runs):
    # a trace is sorted if the queue holds it at once, or holds twice the least sorted trace
    # (6000 photons in this build)
    out = _result(runs, "refill")
    assert out["3200"][0] >= 1 and out["3200"][1]
    assert out["6100"] == [0, True]


def test_which_traces_of_several_cameras_fly(runs):
    # 1024 resident lanes: one camera up to 1.5 photons a lane; in a small tree less by
    # cameras^1.5, and six cameras; in a deep one by cameras^1.75, or ^3.5 for paths of few
    # segments; up to twice as many for long paths
    for deep, depth, cams, n, flown in _result(runs, "route"):
        fits = n * (2 + cams) <= 4.5 * 1024
        more = min(max(depth, 8), 16) / 8
        if not deep:
            fits = fits and cams <= 6 and n * cams ** 1.5 <= 1.5 * 1024 * more
        elif depth < 8:
            fits = fits and n * cams ** 3.5 <= 24 * 1024
        else:
            fits = fits and n * cams ** 1.75 <= 7 * 1024 * more
        assert flown == (1 if fits else 0), (deep, depth, cams, n)


def test_seeding_a_film_of_up_to_a_slot_is_one_synchronous_copy(runs):
    # no event and no staging ring; the words are the rounded doubles on either side of a slot
    out = _result(runs, "seeding")
    assert [npx for npx, *_ in out] == [1, 256, 65536, 65584]
    assert all(same for *_, same in out)
    assert [events > 0 for _, events, _ in out] == [False, False, False, True]


def test_small_downloads_are_converted_on_the_host(runs):
    # the same doubles on either side of the limit
    out = _result(runs, "totals")
    assert all(same for *_, same in out)
    assert [launches for _, launches, _ in out] == [0, 0, 0, 2]   # 3073 pixels: both calls


def test_a_servers_films_with_and_without_scratch_to_convert_them_in(runs):
    # on the device from 16385 pixels on, where there is scratch
    assert _result(runs, "films") == [[2, True], [0, True]]


def test_a_server_runs_no_chunk_after_the_one_that_ends_its_jobs(runs):
    # chunks of two iterations: three or two for small jobs, however they are stepped
    out = _result(runs, "chunks")
    assert all(same for _, same in out)
    assert [ran for ran, _ in out[:3]] == [4, 4, 2]
    assert out[3][0] <= 8   # refilled: 4500 photons through 4096 slots, two iterations each


def test_a_ray_query_of_few_slots_records_no_event(runs):
    out = _result(runs, "probes")
    assert out["events"] == 0 and out["same"] and 0 < out["hit"] < 65600
