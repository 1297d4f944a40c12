"""The kernels that render by default (three wavefronts per line, two and one,
24-word run caches) and the automatic choice, at the edges of the walk: eyes
on cell corners and at negative coordinates, rays along an axis and on the
diagonal, from high above and inside the terrain, mip distances from a few
chunks to the whole walk.  Against the oracle, bit for bit."""
import math

import pytest

pytestmark = pytest.mark.gpu

import test_gpu_parity  # noqa: E402
import workloads  # noqa: E402
from test_gpu_parity import check_view  # noqa: E402

DEFAULTS = [(1, 4, 24), (1, 2, 24), (1, 1, 24), (1, 0, 0)]


@pytest.fixture(autouse=True)
def kernels(monkeypatch):
    monkeypatch.setattr(test_gpu_parity, "KERNELS", DEFAULTS)


@pytest.fixture(scope="module")
def dev(ctx, c1_scene):
    s = ctx.upload(c1_scene.mips)
    yield s
    s.free()


EYES = [(300.0, 200.0), (300.5, 200.25), (-41.3, -77.8), (-64.0, 512.0), (100000.4, 3.1)]
YAWS = [0.0, math.pi / 4, math.pi / 2, 3 * math.pi / 4, math.pi, 1e-4, 2.0]
# altitude above the surface, pitch; mip and far distance
LOOKS = [(30.0, 0.2), (4.0, 0.05), (1500.0, 1.2), (-10.0, 0.1), (12.0, -0.1)]
DISTANCES = [(0, 0), (40, 6000), (700, 3000), (8000, 20000), (65536, 0)]


@pytest.mark.parametrize("k", range(len(EYES) * len(YAWS)))
def test_eyes_and_headings(ctx, oracle, c1_scene, dev, k):
    x, z = EYES[k // len(YAWS)]
    alt, pitch = LOOKS[k % len(LOOKS)]
    mip, far = DISTANCES[(k // 2) % len(DISTANCES)]
    row = workloads.surface_row(c1_scene.mips[0], x, z)
    pose = workloads.pose(x, alt - row, z, pitch, YAWS[k % len(YAWS)])
    check_view(ctx, oracle, dev, c1_scene.mips, pose, 224, 161, mip, far)


@pytest.mark.parametrize("W,H", [(1024, 768), (1366, 768), (1920, 1080), (2560, 1440), (3840, 2160)])
def test_sizes_on_both_sides_of_the_choice(ctx, oracle, c1_scene, dev, W, H):
    for p in workloads.random_views(c1_scene.mips[0], 2, seed=W):
        check_view(ctx, oracle, dev, c1_scene.mips, p, W, H)
