"""Three wavefronts per line (GPU): the rings' edges (lines of few chunks and
of many, lines that end early, frames without a drawn pixel), every run-cache
depth, and the automatic choice on either side of its line limit.  Against
the oracle, bit for bit."""
import pytest

pytestmark = pytest.mark.gpu

import rlevox  # noqa: E402
import workloads  # noqa: E402
from test_gpu_parity import assert_same, gpu_stages  # noqa: E402


@pytest.fixture(scope="module")
def dev(ctx, c1_scene):
    s = ctx.upload(c1_scene.mips)
    yield s
    s.free()


def check(ctx, oracle, dscene, mips, pose, W, H, mip, far, **tuning):
    rm = rlevox.raymap(pose, W, H, mip, far)
    rb, clip, _ = oracle.raycast(mips, oracle.raymap(pose, W, H, mip, far))
    ctx.set_tuning(**tuning)
    try:
        got = gpu_stages(ctx, dscene, rm)
    finally:
        ctx.set_tuning()
    assert_same("line clip", got["clip"][:max(rm.map_line_count, 1)], clip[:max(rm.map_line_count, 1)])
    assert_same("ray buffer", got["raybuf"], rb)
    return rm.map_line_count


# altitude above the surface, pitch, yaw, mip distance, far distance
VIEWS = [
    (30.0, 0.2, 0.4, 0, 0),
    (3.0, 0.02, 2.2, 700, 20000),     # long lines along the ground
    (200.0, 1.2, 1.0, 0, 0),          # straight down: full early
    (60.0, -0.9, 0.3, 0, 0),          # the sky
    (25.0, 0.1, 3.0, 8, 40),          # less than a chunk
    (25.0, 0.1, 5.0, 20, 3000),       # a mip switch every few chunks
]


@pytest.mark.parametrize("size", [(64, 48), (321, 243)])
@pytest.mark.parametrize("depth", [24, 40, 56])
@pytest.mark.parametrize("view", range(len(VIEWS)))
def test_three_waves(ctx, oracle, c1_scene, dev, view, depth, size):
    alt, pitch, yaw, mip, far = VIEWS[view]
    row = workloads.surface_row(c1_scene.mips[0], 300.0, 200.0)
    pose = workloads.pose(300.0, alt - row, 200.0, pitch, yaw)
    check(ctx, oracle, dev, c1_scene.mips, pose, size[0], size[1], mip, far, waves_per_block=4,
          run_cache=depth)


def test_automatic_choice(ctx, oracle, c1_scene, dev):
    row = workloads.surface_row(c1_scene.mips[0], 300.0, 200.0)
    pose = workloads.pose(300.0, 30.0 - row, 200.0, 0.25, 0.4)
    lines = [check(ctx, oracle, dev, c1_scene.mips, pose, W, H, 0, 0)
             for W, H in [(640, 480), (1920, 1080)]]
    assert lines[0] <= 1792 < lines[1]
