"""Long walks at one mip level (GPU): mip distances up to the whole walk over
flat ground with sparse towers, where a stretch of the walk judged by the
wrong columns loses a tower.  Every wavefront kernel and the batch against the
oracle, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import rlevox  # noqa: E402
import workloads  # noqa: E402
from test_gpu_parity import assert_same, gpu_stages  # noqa: E402

SIZE, HEIGHT, GROUND = 512, 64, 60


@pytest.fixture(scope="module")
def towers():
    rng = np.random.default_rng(9)
    solid = np.zeros((SIZE, HEIGHT, SIZE), np.uint8)  # z, y, x
    solid[:, GROUND:, :] = 1
    for _ in range(60):
        x, z = rng.integers(0, SIZE - 1, 2)
        solid[z:z + 2, int(rng.integers(2, 52)):, x:x + 2] = 1
    colour = (np.arange(solid.size, dtype=np.uint32) % 60000).astype(np.uint16).reshape(solid.shape)
    return rlevox.encode_dense(solid, colour, nmips=3)


@pytest.fixture(scope="module")
def dev(ctx, towers):
    s = ctx.upload(towers.mips)
    yield s
    s.free()


@pytest.mark.parametrize("mip", [8192, 65536, 262144])
def test_towers_at_long_mip_distances(ctx, oracle, towers, dev, mip):
    rng = np.random.default_rng(mip)
    W, H = 512, 384
    for k in range(8):
        x, z = rng.uniform(0, SIZE, 2)
        alt = rng.uniform(1.0, 20.0 if k % 2 else 300.0)
        row = workloads.surface_row(towers.mips[0], float(x), float(z))
        p = workloads.pose(float(x), float(alt) - row, float(z), float(rng.uniform(0.01, 0.2)),
                           float(rng.uniform(0, 6.28)))
        rm = rlevox.raymap(p, W, H, mip, 0)
        ref_rb, ref_clip, _ = oracle.raycast(towers.mips, oracle.raymap(p, W, H, mip, 0))
        n = max(rm.map_line_count, 1)
        for wpb in (0, 1, 2, 4):
            ctx.set_tuning(waves_per_block=wpb)
            try:
                got = gpu_stages(ctx, dev, rm)
            finally:
                ctx.set_tuning()
            tag = " [view %d, waves_per_block %d]" % (k, wpb)
            assert_same("line clip" + tag, got["clip"][:n], ref_clip[:n])
            assert_same("ray buffer" + tag, got["raybuf"], ref_rb)
        dc, dd = ctx.alloc(W * H * 2), ctx.alloc(W * H * 4)
        ctx.render_batch([rlevox.make_view(dev, p, W, H, dc, dd)],
                         params=rlevox.RenderParams(mip, 0, 0, 0))
        ctx.sync()
        col, dep = oracle.compose(oracle.raymap(p, W, H, mip, 0), ref_rb, ref_clip)
        assert_same("batch depth %d" % k, dd.download(np.int32, W * H).reshape(H, W), dep)
        assert_same("batch colour %d" % k, dc.download(np.uint16, W * H).reshape(H, W),
                    oracle.gapfill(col, dep))
        dc.free()
        dd.free()
