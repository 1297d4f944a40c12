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
    assert waves(setting, lines, width) == want
