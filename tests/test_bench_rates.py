"""Rates of the benchmark's JSON line, from the stub library's 10 ms per kernel group.

M2L: the bytes are every multipole read and every local written once, and the
parents' locals of the levels whose M2L and L2L are one kernel -- the leaf alone,
or every level from 3 on, whichever the solver was told.

Near field: achieved and frac count the dense blocks' flops; the matrix cores run
a quarter of the complex multiplications, of 24 FP16 flops each in the split
kernel and 6 otherwise, and executed / executed_frac say so.
"""
import pytest

from test_bench_flow import ROOT, run_bench


@pytest.fixture
def bench(monkeypatch):
    monkeypatch.syspath_prepend(ROOT)
    import bench as m
    return m


NS = [280, 180, 120, 90, 72, 68]  # samples of six levels


def test_m2l_bytes_count_the_parents_of_the_fused_levels(bench):
    b = 8
    plain = 2 * b * (16 * 120 + 64 * 90 + 256 * 72 + 1024 * 68)
    assert bench.m2l_bytes_per_rhs(6, NS, b) == plain
    assert bench.m2l_bytes_per_rhs(6, NS, b, 5) == plain + b * 256 * 72
    assert bench.m2l_bytes_per_rhs(6, NS, b, 3) == plain + b * (16 * 120 + 64 * 90 + 256 * 72)


def test_fused_levels_follow_the_choice_and_the_rule(bench):
    assert bench.fused_from(6, 0, 64) is None
    assert bench.fused_from(6, 1, 64) == 5
    assert bench.fused_from(6, -1, 6) == 5 and bench.fused_from(6, -1, 7) == 3
    assert bench.fused_from(8, -1, 1) == 3  # the single-system FP64 path at 1024^2
    assert bench.fused_from(3, -1, 64) is None


def test_json_line_counts_the_leaf_alone(bench, monkeypatch):
    """The stub's solvers fuse the leaf (1): 2 steps x 250 FP32 products in 10 ms."""
    d = run_bench(monkeypatch, "--workload", "dbim-256", "--steps", "2", "--warmup", "0", "--cpu-baseline", "off",
                  "--ref-geometry", "off")
    ns = [4 * (8 + i) for i in range(6)]
    want = 500 * bench.m2l_bytes_per_rhs(6, ns, 8, 5) / 10e-3 / 1e9
    assert abs(d["m2l"]["achieved_GBs"] - want) < 0.1
    assert d["m2l"]["leaf_l2l_fused"] is True and d["m2l"]["fused_from_level"] == 5


@pytest.mark.parametrize("split,per_dense", [(128, 24 / 32), (0, 6 / 32)])
def test_executed_rate_counts_the_symmetric_products(monkeypatch, split, per_dense):
    r = run_bench(monkeypatch, "--workload", "dbim-256", "--steps", "2", "--warmup", "0", "--cpu-baseline", "off",
                  "--ref-geometry", "off", split=split)["roofline"]
    assert abs(r["executed"] - per_dense * r["achieved"]) < 0.02
    assert abs(r["executed_frac"] - r["executed"] / r["peak"]) < 1e-3
    assert r["executed_frac"] < r["frac"]
