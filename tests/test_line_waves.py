"""How many wavefronts walk a line, by the tuning and the frame (CPU)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def waves(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("line_waves") / "check")
    subprocess.run(["g++", "-O2", "-std=c++17", os.path.join(HERE, "native", "line_waves_check.cpp"),
                    "-o", exe], check=True)

    def run(*args):
        r = subprocess.run([exe], input=" ".join(map(str, args)), stdout=subprocess.PIPE, text=True,
                           check=True)
        return int(r.stdout)

    return run


# 4 at 1920x1080 took two wavefronts before there was a form with three,
# which is slower there.
@pytest.mark.parametrize("setting,lines,width,want", [
    (0, 441, 320, 3), (0, 1792, 1366, 3), (0, 1793, 1366, 2), (0, 3000, 2560, 2),
    (0, 500, 2561, 1), (0, 9000, 3840, 1),
    (1, 441, 320, 1), (1, 9000, 3840, 1),
    (2, 441, 320, 2), (2, 9000, 3840, 2), (3, 441, 320, 2), (3, 9000, 3840, 2),
    (4, 441, 320, 3), (4, 1792, 1366, 3), (4, 1793, 1366, 2), (4, 2048, 1920, 2),
    (4, 500, 2561, 2), (4, 9000, 3840, 2)])
def test_waves_per_line(waves, setting, lines, width, want):
    assert waves(setting, lines, width, 21040) == want


# LDS of a line with a run cache of 24, 40 and 56 words, and at the edges of
# the unit in which it is given out: seven, six, five lines a compute unit.
@pytest.mark.parametrize("lds,most", [(21040, 1792), (25136, 1536), (29232, 1280), (23040, 1792),
                                      (23041, 1536), (26880, 1536), (26881, 1280)])
def test_three_waves_while_every_line_is_resident(waves, lds, most):
    for setting in (0, 4):
        assert waves(setting, most, 1366, lds) == 3
        assert waves(setting, most + 1, 1366, lds) == 2
