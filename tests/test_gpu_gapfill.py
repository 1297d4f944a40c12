"""Gap-fill where its tap sets change (GPU): depths at and around the limits
of the 2x2, 3x3, 4x4 and 5x5 sets, of the staged border and of the taps'
reach, alone and mixed, on sizes with inner, clamped and partial tiles.
Bit for bit against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIMITS = [1, 2, 24, 25, 26, 122, 123, 124, 203, 204, 205, 366, 367, 368, 609, 610, 611, 615, 616, 1874,
          1875, 40000, 0x7fffffff]


def run(ctx, oracle, col, dep):
    H, W = col.shape
    b = [ctx.alloc(W * H * 2), ctx.alloc(W * H * 4), ctx.alloc(W * H * 2)]
    b[0].upload(col)
    b[1].upload(dep)
    ctx.gapfill(W, H, b[0], b[1], b[2])
    ctx.sync()
    got = b[2].download(np.uint16, W * H).reshape(H, W)
    for x in b:
        x.free()
    want = oracle.gapfill(col, dep)
    assert np.array_equal(got, want), "%d pixels differ" % int((got != want).sum())


@pytest.mark.parametrize("W,H", [(256, 96), (250, 61), (64, 4), (131, 133)])
@pytest.mark.parametrize("k", range(len(LIMITS)))
def test_depths_at_a_limit(ctx, oracle, W, H, k):
    """One depth and its neighbours over the whole image, other depths
    sprinkled in: tap sets of one kind, and of two or three."""
    rng = np.random.default_rng(100 * k + W)
    col = rng.integers(0, 65536, (H, W)).astype(np.uint16)
    dep = np.full((H, W), LIMITS[k], np.int32)
    for share, pool in ((0.2, LIMITS[max(k - 1, 0):k + 2]), (0.02, LIMITS)):
        m = rng.random((H, W)) < share
        dep[m] = rng.choice(np.array(pool, np.int32), int(m.sum()))
    run(ctx, oracle, col, dep)


def test_far_and_near_tiles(ctx, oracle):
    """Whole tiles beyond the taps' reach beside near ones."""
    rng = np.random.default_rng(5)
    H, W = 300, 516
    col = rng.integers(0, 65536, (H, W)).astype(np.uint16)
    dep = np.where(rng.random((H // 30, W // 43)) < 0.5, 700, 90).repeat(30, 0).repeat(43, 1)
    dep = (dep + rng.integers(0, 60, (H, W))).astype(np.int32)
    run(ctx, oracle, col, dep)
