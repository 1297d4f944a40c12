"""The device memory a resident scene reports (GPU): pointer maps, slabs and
the tops of each level's 16x16 blocks of columns."""
import pytest

pytestmark = pytest.mark.gpu


def test_device_bytes_count_every_table(ctx, c1_scene):
    mips = c1_scene.mips
    s = ctx.upload(mips)
    try:
        arrays = sum(m["ptrmap"].nbytes + m["slabs"].nbytes for m in mips)
        blocks = sum(max(m["sx"] // 16, 1) * max(m["sz"] // 16, 1) for m in mips)
        # each level's slabs are padded by 512 to 767 bytes; the descriptor and
        # the levels' own tops take less than 1 KB
        pad = s.device_bytes - arrays - 4 * blocks
        assert 512 * len(mips) < pad < 768 * len(mips) + 1024
    finally:
        s.free()
