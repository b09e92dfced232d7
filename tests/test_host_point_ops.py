"""The operation counts behind bench.py's point-kernel roofline are those of the code: the crystal-frame form is
run on a number type that counts (tests/cpu_point/op_count.cpp)."""
import importlib.util
import os
import subprocess

import pytest

from conftest import ROOT

SRC = os.path.join(ROOT, "tests", "cpu_point", "op_count.cpp")


@pytest.fixture(scope="module")
def bench():
    spec = importlib.util.spec_from_file_location("bench_ops", os.path.join(ROOT, "bench.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def test_counts_are_those_of_the_code(bench, tmp_path):
    exe = str(tmp_path / "op_count")
    subprocess.run(["g++", "-O1", "-std=c++17", "-o", exe, SRC], check=True)
    lines = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split("\n")
    counted = [tuple(map(int, line.split())) for line in lines if line]
    order = ("residual", "elastic_residual", "jacobian", "setup", "outputs", "tangent")
    assert set(order) == set(bench.POINT_OPS)
    for name, (c12, c24) in zip(order, counted):
        per, fixed = bench.POINT_OPS[name]
        assert (12 * per + fixed, 24 * per + fixed) == (c12, c24), name


def test_elastic_residuals_and_first_steps_run_no_slip_loop(bench):
    """One point with k iterations and k + 1 residuals: k with slip, and k - 1 Jacobians."""
    res, jac = 94 * 24 + 137 + 12, 85 * 24 + 529
    f = [bench.point_ops(24, 1, 0, k, k + 1) for k in (1, 2, 5)]
    assert f[1] - f[0] == res + jac
    assert f[2] - f[0] == 4 * (res + jac)
    assert f[0] == 144 + (3 * 24 + 136) + 80 + 381 + res
    assert bench.point_ops(24, 10, 10, 50, 60) == 10 * bench.point_ops(24, 1, 1, 5, 6)
