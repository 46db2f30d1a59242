"""bench.py prices the face stage by the counters committed under profiles/: its
kernels are found there, and the bound it names is the busier unit."""
import os
import re
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


def test_face_stage_is_priced():
    kernel = bench.face_kernels("learned")
    r = bench.roofline(kernel, 2.75e-3, 1e9, 400.0)
    assert r["kernel"] == kernel and r["traffic"] > 1e9
    assert r["bound"] in ("valu", "vector_memory_addressing")
    others = [v["frac"] for v in r.values() if isinstance(v, dict)]
    assert 0.0 < max(others) <= r["frac"] < 1.0
    assert r["achieved"] / r["peak"] == pytest.approx(r["frac"])


def test_stage_figures_are_the_kernels_sums():
    names = bench.face_kernels("learned").split(" + ")
    for key in ("traffic_bytes_per_launch", "valu_instr_per_launch", "ta_busy_cycles_per_launch"):
        each = [bench.profiled(key, k) for k in names]
        assert bench.profiled(key, " + ".join(names)) == pytest.approx(sum(each))


def test_unknown_kernel_is_not_given_a_bound():
    r = bench.roofline("k_nothing<3>", 1e-3, 1e9, 400.0)
    assert r["bound"] == "not measured" and r["traffic"] is None


def test_names_are_those_the_step_launches():
    """the particles per wavefront in the names follow kPairGroup"""
    src = open(os.path.join(ROOT, "meshlesshydro_amd", "csrc", "hydro_impl.h")).read()
    fp32, fp64 = map(int, re.search(r"kPairGroup = sizeof\(T\) == 4 \? (\d+) : (\d+);", src).groups())
    assert "k_face_pairs<3, float, true, %d>" % fp32 in bench.face_kernels("learned")
    assert "k_face_deferred<3, %d>" % fp32 in bench.face_kernels("learned")
    assert bench.profiled("valu_instr_per_launch", "k_face_pairs<3, double, false, %d>" % fp64) > 0


def test_algorithmic_bytes_hold_the_fluxes():
    """56 entries in FP32: 28 fluxes of 20 bytes written, 56 read"""
    with_rows = bench.face_kernel_bytes(3, 4, 56.0) - bench.face_kernel_bytes(3, 4, 0.0)
    assert with_rows == pytest.approx(28 * 20 + 56 * 20 + 84 * 4)
