"""The closed form of the DDA's crossing sequences (csrc/dda_terms.h) on the
CPU: every fit it accepts gives the sequential fp32 sums bit for bit."""
import os
import re
import subprocess

import pytest

NATIVE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")


def _run(tmp_path, plant):
    exe = str(tmp_path / "dda_terms_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-DDDA_TERMS_PLANT=%d" % plant,
                    os.path.join(NATIVE, "dda_terms_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    m = re.search(r"tried (\d+), one binade (\d+), one crossing (\d+), mismatches (\d+)", r.stdout)
    assert m, r.stdout
    return [int(v) for v in m.groups()]


def test_accepted_fits_equal_the_sums(tmp_path):
    """Six sequences of 20000 lines and 2 M arbitrary sums and steps (ties,
    powers of two, zeros, infinities, subnormals): no term differs, and the
    fits cover nearly all of the lines' chunks."""
    tried, one, two, bad = _run(tmp_path, 0)
    assert bad == 0
    assert one + two > 0.8 * tried and two > 100000


@pytest.mark.parametrize("plant", [1])
def test_check_catches_an_unchecked_first_step(tmp_path, plant):
    """Without the test of the first step against the second the same check
    finds wrong terms."""
    assert _run(tmp_path, plant)[3] > 0
