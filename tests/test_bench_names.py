"""bench.py's names and bytes of the profiled kernel classes against the
sources and the committed counter profile: every class of the profiled paths
that the profile has by base name is there under kernel_name()'s full name, the
factorisation's three instantiations have the template parameters ilu.hip
launches, and the residual's kind follows flux.hip's lines between its two
routes."""
import json
import os
import re

import pytest

import bench

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _source(name):
    return open(os.path.join(ROOT, "kfun3d_amd", "csrc", name)).read()


@pytest.fixture(scope="module")
def profile():
    return json.load(open(os.path.join(ROOT, "profiles", "traffic_c5.json")))["kernels"]


@pytest.mark.parametrize("prec,dom", [("fp64", d) for d in ("grad", "edge_flux", "fill", "ilu", "trsv_lower", "trsv_upper")] +
                         [("bf16", d) for d in ("fill", "ilu", "trsv_lower", "trsv_upper")])
def test_profiled_class_is_in_the_counter_profile(profile, prec, dom):
    name = bench.kernel_name(dom, prec, 7, True, 2654208)
    assert name in profile, (name, sorted(profile))


def test_factorisation_names_are_the_launched_ones():
    calls = re.findall(r"launch_ilu<([^>]*)>\(c, c->a", _source("ilu.hip"))
    launched = {"k_ilu_rows<%s>" % c.replace("uint16_t", "unsigned short") for c in calls}
    named = {bench.kernel_name("ilu", p, 7, True, 2654208) for p in ("fp64", "fp32", "bf16")}
    assert named == launched - {"k_ilu_rows<double, false, double>"}   # the paths factor FP64 exactly


def test_residual_routes_follow_the_source():
    src = _source("flux.hip")
    one, wide = (int(re.search(r"#define FLUX_%s_ROWS (\d+)u" % w, src).group(1)) for w in ("ONE", "WIDE"))
    assert (bench.FLUX_ONE_ROWS, bench.FLUX_WIDE_ROWS) == (one, wide)
    for n, name, kind in ((wide, "k_flux_residual<16, false, true>", "flux_residual_fd"),
                          (wide + 1, "k_flux_residual<4, false, true>", "flux_residual_fd"),
                          (one, "k_flux_residual<4, false, true>", "flux_residual_fd"),
                          (one + 1, "k_residual<false, true>", "residual_fd")):
        assert bench.kernel_name("residual", "fp64", 7, True, n) == name
        assert bench.profile_kind("residual", n) == kind


def test_factorisation_bytes_count_its_copies():
    n = 1000
    base = {p: bench.alg_bytes("ilu", 0, 0, 0, 0, n, bench.value_bytes("ilu", p), 0) for p in ("fp64", "fp32", "bf16")}
    assert base == {"fp64": 260 * n, "fp32": 132 * n, "bf16": 132 * n}
    for prec, sweeps, more in (("fp64", 0, 0), ("fp64", 2, 128), ("fp32", 0, 0), ("fp32", 2, 64), ("bf16", 0, 32),
                               ("bf16", 2, 64)):
        got = bench.alg_bytes("ilu", 0, 0, 0, 0, n, bench.value_bytes("ilu", prec), bench.ilu_copies(prec, sweeps))
        assert got == base[prec] + more * n, (prec, sweeps)
