"""The tiled GEMM's plan (csrc/gemm_plan.cpp) on the CPU: what it may not do whatever the fitted costs say."""
import random

import pytest

from plan_util import gemm_plan, stream_us


def test_plans_fit_their_room_and_the_kernels():
    r = random.Random(3)
    for _ in range(4000):
        m, k = r.randint(1, 9000), 8 * r.randint(1, 2200)
        n = [8 * r.randint(1, 2200) for _ in range(r.choice([1, 3]))]
        room = r.choice([0, 256, 80 << 10, 4 << 20, 64 << 20, 2 ** 62])
        p = gemm_plan(m, k, n, room=room)
        assert p.bytes <= room
        assert (p.bm, p.bn) in {(256, 256), (256, 128), (128, 128), (128, 64), (64, 64), (32, 64)}
        tiles = -(-m // p.bm) * sum(-(-x // p.bn) for x in n)
        steps = -(-k // 64)
        assert not (p.tail and p.ks > 1)
        if p.tail:
            assert p.bn == 256 and steps >= 4 and p.tail == tiles % 256 and 2 * p.tail <= 256
        if p.ks > 1:
            assert p.bn != 256 and 0 < p.split_tiles <= tiles and p.split_tiles <= 16384 and steps // p.ks >= 3
        assert bool(p.bytes) == bool(p.tail or p.ks > 1)


# measured the other way round in time: rows that do not begin on 64 bytes
@pytest.mark.parametrize("m,k,n", [(5977, 3112, (7184,)), (2882, 5608, (17488, 1168, 1168)), (2027, 4712, (14256,)),
                                   (2694, 8528, (17360,)), (5288, 3056, (8704, 2040, 2040)), (6769, 272, (5048,))])
def test_unaligned_rows_keep_the_large_tiles(m, k, n):
    assert gemm_plan(m, k, n).bn == 256


# products that the smaller tiles run 1.05 times faster or more
@pytest.mark.parametrize("m,k,n", [(4096, 4096, (8192, 1024, 1024)), (1000, 4096, (8192, 1024, 1024)), (1355, 10992, (7880, 1608, 1608)),
                                   (3932, 1664, (4592, 592, 592)), (890, 4008, (2328,)), (2040, 9520, (856,))])
def test_smaller_tiles_where_they_were_faster(m, k, n):
    assert gemm_plan(m, k, n).bn < 256


# rows, k, 16-column blocks, us streamed, us tiled (output projections, weights from HBM, one MI355X): the estimates take
# the faster
@pytest.mark.parametrize("m,k,ncb,streamed,tiled", [
    (1, 12288, 512, 36.2, 44.2), (1, 8192, 512, 25.4, 29.3), (1, 8192, 1024, 46.7, 52.0), (1, 12288, 1280, 83.8, 92.9),
    (1, 4096, 512, 14.5, 17.0), (1, 4096, 1280, 29.8, 33.5), (1, 4096, 1792, 39.7, 51.0),
    (1, 1024, 1792, 31.5, 13.5), (8, 1024, 320, 11.1, 6.4), (8, 2048, 576, 17.4, 10.4), (8, 4096, 640, 20.2, 16.9),
    (8, 4096, 272, 13.9, 10.7), (12, 8192, 640, 46.9, 31.1), (8, 3072, 1024, 23.9, 18.5), (12, 12288, 1024, 93.4, 70.6),
    (1, 6144, 512, 23.7, 19.4), (1, 5120, 1280, 49.2, 41.0),
])
def test_few_rows_take_the_faster_kernel(m, k, ncb, streamed, tiled):
    assert (stream_us(m, k, ncb) <= gemm_plan(m, k, (16 * ncb,)).us) == (streamed < tiled)
