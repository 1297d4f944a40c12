"""What a group of steps can touch (csrc/walk_skip.h), on the CPU: against the
walk's own sums, and against the oracle's full walk at mip distances up to
the whole walk."""
import os
import re
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "rle-based-voxel-raycasting_amd", "csrc")


def _build(tmp_path, name, defines, lib=False):
    exe = str(tmp_path / name)
    srcs = [os.path.join(HERE, "native", name + ".cpp")]
    if lib:
        srcs += [os.path.join(CSRC, f) for f in ("host.cpp", "raymap.cpp", "scene.cpp")]
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fopenmp", "-pthread",
                    "-Wno-subobject-linkage"] + ["-D" + d for d in defines] + srcs + ["-o", exe],
                   check=True)
    return exe


def _run(exe, *args):
    r = subprocess.run([exe] + [str(a) for a in args], stdout=subprocess.PIPE, text=True,
                       env=dict(os.environ, OMP_NUM_THREADS="4"))
    assert r.returncode == 0, r.stdout
    return r.stdout


def _range(tmp_path, plant, mip, steps=20000000):
    out = _run(_build(tmp_path, "walk_range_check", ["WALK_RANGE_PLANT=%d" % plant]), mip, steps)
    m = re.search(r"groups (\d+), of two blocks a side (\d+), below lo (\d+), above hi (\d+), "
                  r"outside (\d+)", out)
    assert m, out
    return dict(zip(("groups", "near", "below", "above", "outside"), map(int, m.groups())))


@pytest.mark.parametrize("mip", [300, 1024, 4096, 16384, 65536, 262144])
def test_every_step_is_in_its_groups_blocks(tmp_path, mip):
    """No step's cell lies outside the blocks its group looks up, and no
    step ends beyond the group's distances, however long the level."""
    r = _range(tmp_path, 0, mip)
    assert r["groups"] > 200000 and r["near"] > 0.05 * r["groups"]
    assert r["outside"] == 0 and r["above"] == 0


@pytest.mark.parametrize("mip", [16384, 65536])
def test_range_check_catches_a_missing_offset(tmp_path, mip):
    assert _range(tmp_path, 1, mip)["outside"] > 0


@pytest.mark.parametrize("mip", [30, 1024, 4096])
def test_no_step_is_nearer_than_its_group(tmp_path, mip):
    """Near an axis too, where the guessed split of a group's steps between
    the two kinds of crossing is off."""
    assert _range(tmp_path, 0, mip, 100000000)["below"] == 0


def _reach(exe, scene, mip):
    out = _run(exe, scene, mip, 30)
    m = re.search(r"steps (\d+), hidden (\d+), violations (\d+)", out)
    assert m, out
    return [int(v) for v in m.groups()]


@pytest.mark.parametrize("scene", [0, 1])
def test_no_hidden_step_acts_on_long_levels(tmp_path, scene):
    """Over 30 views a mip distance no step of a hidden group draws or moves
    the window (rough terrain, and flat ground with towers)."""
    exe = _build(tmp_path, "walk_reach_check", ["WALK_REACH_PLANT=0"], lib=True)
    for mip in (0, 4096, 8192, 16384, 65536, 262144):
        steps, hidden, violations = _reach(exe, scene, mip)
        assert violations == 0, mip
        assert hidden > 0.4 * steps, mip


@pytest.mark.parametrize("scene", [0, 1])
def test_reach_check_catches_a_missing_offset(tmp_path, scene):
    exe = _build(tmp_path, "walk_reach_check", ["WALK_REACH_PLANT=1"], lib=True)
    assert _reach(exe, scene, 65536)[2] > 0
