"""The chunked walk where its closed form changes form (GPU): eyes on cell
corners and at negative coordinates, rays along an axis and on the diagonal,
mip distances from a few chunks to the whole walk.  Every kernel against the
oracle, bit for bit."""
import math

import pytest

pytestmark = pytest.mark.gpu

import workloads  # noqa: E402
from test_gpu_parity import check_view  # noqa: E402


@pytest.fixture(scope="module")
def dev(ctx, c1_scene):
    s = ctx.upload(c1_scene.mips)
    yield s
    s.free()


EYES = [(300.0, 200.0), (300.5, 200.25), (-41.3, -77.8), (-64.0, 512.0), (100000.4, 3.1)]
YAWS = [0.0, math.pi / 4, math.pi / 2, 3 * math.pi / 4, math.pi, 1e-4, 2.0]


@pytest.mark.parametrize("k", range(len(EYES) * len(YAWS)))
def test_eye_positions_and_headings(ctx, oracle, c1_scene, dev, k):
    x, z = EYES[k // len(YAWS)]
    yaw = YAWS[k % len(YAWS)]
    row = workloads.surface_row(c1_scene.mips[0], x, z)
    alt, pitch = [(30.0, 0.2), (4.0, 0.05), (150.0, 0.6), (12.0, -0.1)][k % 4]
    mip, far = [(0, 0), (40, 6000), (700, 3000), (8000, 20000)][(k // 4) % 4]
    check_view(ctx, oracle, dev, c1_scene.mips, workloads.pose(x, alt - row, z, pitch, yaw), 224, 161,
               mip, far)
