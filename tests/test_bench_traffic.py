"""bench.py's measured HBM traffic: the counters of the kernels that the roofline line names
and of no others.  The profiler's runs are replaced by its result."""
import argparse

import pytest

import bench

GIB_KIB = float(1 << 20)
KERNELS = {"__amd_rocclr_copyBuffer": [95.0, GIB_KIB / 2], "void (anonymous namespace)::k_draw<false>(unsigned int*)": [4000.0],
           "void (anonymous namespace)::k_coverage<128>(CovArgs)": [100.0, 300.0],
           "void (anonymous namespace)::k_coverage<512>(CovArgs)": [50.0], "(anonymous namespace)::k_coverage_many(CovArgs)": [70.0],
           "void (anonymous namespace)::k_draw<3u>(unsigned int*)": [1.0], "void (anonymous namespace)::k_expand<16>(ExpandArgs)": [8.0]}


@pytest.mark.parametrize("name,kib", [("draw_items", 4000.0), ("coverage", 520.0 / 4), ("expand", 8.0)])
def test_live_traffic_of_the_named_kernel(monkeypatch, name, kib):
    import shutil
    import subprocess
    monkeypatch.setattr(shutil, "which", lambda _: "rocprofv3")
    monkeypatch.setattr(subprocess, "run", lambda *a, **k: argparse.Namespace(returncode=0))
    monkeypatch.setattr(bench, "_counter_per_dispatch", lambda d, counter: KERNELS)
    got = bench.live_traffic(argparse.Namespace(size=64, paths=2, seed=0), name)
    # the copy of 1 GiB counts half, so each counter is scaled by two
    assert got["fetch_bytes"] == got["write_bytes"] == round(2 * kib * 1024)
    assert got["bytes_per_launch"] == 2 * got["fetch_bytes"]


def test_other_kernels_have_none(monkeypatch):
    import shutil
    monkeypatch.setattr(shutil, "which", lambda _: "rocprofv3")
    assert bench.live_traffic(argparse.Namespace(size=64, paths=2, seed=0), "box_blur_round") is None
