"""bench.py prints counters of committed profiles only for the kernels they were taken on: the
same sources apart from comments, tuning and photon count."""
import json
import os
import shutil

import pytest

import bench

TUNING = {"queue_capacity": 8, "ray_sort": 2}


@pytest.fixture
def record(tmp_path, monkeypatch):
    monkeypatch.setattr(bench, "PROFILES", str(tmp_path))

    def write(**kw):
        rec = {"sources": bench.kernel_sources_digest(), "photons": 7, "tuning": TUNING,
               "kernels": {"k_extend": {"hbm_bytes_per_dispatch": 5, "valu_insts_per_dispatch": 1000,
                                        "lane_utilization": 0.5}}, **kw}
        for kind in ("traffic", "valu"):
            with open(tmp_path / f"c9_{kind}.json", "w") as f:
                json.dump({k: v for k, v in rec.items() if v is not None}, f)
    return write


def _found():
    t, src = bench.measured_traffic("c9", "k_extend", TUNING, 7)
    v = bench.measured_valu("c9", "k_extend", TUNING, 7, 1.0)
    assert (t is None) == (src is None) == (v is None)
    return t == 5 and v["lane_utilization"] == 0.5 if t is not None else None


def test_a_matching_record_is_used(record):
    record()
    assert _found()


@pytest.mark.parametrize("change", [{"sources": "0" * 16}, {"sources": None}, {"photons": 8},
                                    {"tuning": {**TUNING, "ray_sort": 1}}, {"kernels": {}}], ids=str)
def test_any_other_is_not(record, change):
    record(**change)
    assert _found() is None


def test_the_digest_follows_the_code_and_not_its_comments(tmp_path):
    csrc = os.path.join(bench.ROOT, "goodphotons_amd", "csrc")
    for name in bench.KERNEL_SOURCES:
        shutil.copy(os.path.join(csrc, name), tmp_path / name)
    same = bench.kernel_sources_digest(csrc)
    assert bench.kernel_sources_digest(str(tmp_path)) == same
    with open(tmp_path / "gp_device.hpp", "a") as f:
        f.write("\n   // a remark\n")
    assert bench.kernel_sources_digest(str(tmp_path)) == same
    with open(tmp_path / "gp_device.hpp", "a") as f:
        f.write("constexpr int kMore = 1;\n")
    assert bench.kernel_sources_digest(str(tmp_path)) != same
