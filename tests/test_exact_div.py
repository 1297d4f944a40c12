"""Quotients from shared reciprocals (csrc/exact_div.h) on the CPU."""
import os
import re
import subprocess

import pytest

NATIVE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")


def _run(tmp_path, plant):
    exe = str(tmp_path / "exact_div_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-mfma",
                    "-DEXACT_DIV_PLANT=%d" % plant, os.path.join(NATIVE, "exact_div_check.cpp"),
                    "-o", exe], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    m = re.search(r"reciprocals (\d+), quotients (\d+), mismatches (\d+) (\d+)", r.stdout)
    assert m, r.stdout
    return [int(v) for v in m.groups()]


def test_reciprocals_and_quotients_are_rounded_to_nearest(tmp_path):
    """Every significand with estimates up to one ulp off, and 40 M quotients
    (a quarter next to rounding boundaries), against fp32 division."""
    recips, quots, bad_r, bad_q = _run(tmp_path, 0)
    assert bad_r == 0 and bad_q == 0
    assert recips > 45000000 and quots > 30000000


@pytest.mark.parametrize("plant", [1, 2])
def test_check_catches_planted_mistakes(tmp_path, plant):
    """An all-ones significand accepted, or the quotient left uncorrected."""
    assert sum(_run(tmp_path, plant)[2:]) > 0
