"""profiles/traffic.json, which bench.py reports as each launch's HBM traffic: the launches
that the plans run, with the values of the counter summary beside it."""
import json
import os
import re

import pytest

from conftest import REPO

PROFILES = os.path.join(REPO, "profiles")


def _traffic():
    with open(os.path.join(PROFILES, "traffic.json")) as f:
        return json.load(f)


@pytest.mark.parametrize("workload,launches", [
    ("adjoint_16x4096x4096_fwd", {"row_r2c", "column_c2c"}),   # columns of 2^12 rows: one launch
    ("adjoint_16x4096x4096_adj", {"row_c2r", "column_c2c"}),
    ("f64_16384x16384", {"row_r2c", "column_phase_a", "column_phase_b"}),
    ("batched_512_seed4", {"batched_rows", "batched_columns"})])
def test_launches(workload, launches):
    assert set(_traffic()[workload]) == launches


def test_values_are_the_summary():
    with open(os.path.join(PROFILES, "bench_legs_hbm_traffic.txt")) as f:
        listed = {(m[1], m[2]): float(m[3]) for m in re.finditer(r"^  (\S+) +(\S+) +FETCH .* HBM +([\d.]+) GB", f.read(), re.M)}
    have = {(w, k): v / 1e9 for w, d in _traffic().items() for k, v in d.items()}
    assert set(listed) == set(have)
    for k, v in have.items():
        assert abs(listed[k] - v) <= 6e-5, k
