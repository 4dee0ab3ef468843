"""The split bounces' hand-out of the ray queue (path tracer, ray_fetch 2 and 4):
records equal to the fused bounces', and no cost for blocks beyond what the
device holds."""
import time

import pytest
import torch

from fledge_amd import _native as N
from fledge_amd import api

pytestmark = pytest.mark.gpu


def sphere(ctx, level):
    v, i = api.gen_octasphere(level, 0.1, seed=7, base_freq=2.0)
    return api.LBVH.build(ctx, torch.from_numpy(v).cuda(), torch.from_numpy(i).cuda())


# a queue of a few rays, one share a wave, shares of the largest size and more
# of them than waves (one block of 64 a CU: 256 waves of 128 rays)
@pytest.mark.parametrize("w,h,spp", [(5, 3, 1), (96, 64, 2), (400, 300, 2)])
@pytest.mark.parametrize("block,per_cu", [(64, 1), (128, 64), (512, 2)])
@pytest.mark.parametrize("fetch", [2, 4])
def test_hand_out(ctx, w, h, spp, block, per_cu, fetch):
    print("split queue %dx%dx%d block %d x %d fetch %d" % (w, h, spp, block, per_cu, fetch), flush=True)
    bvh = sphere(ctx, 4)
    cam = N.Camera.make((0.0, 0.0, -1.6), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 45.0)
    want = bvh.pathtrace(cam, w, h, spp, 3, record=True, ray_fetch=1)
    got = bvh.pathtrace(cam, w, h, spp, 3, record=True, ray_fetch=fetch, trace_block=block, blocks_per_cu=per_cu,
                        stack_mode=2, ring_depth=8)
    assert got["segments"] == want["segments"] > w * h * spp
    assert torch.equal(got["nseg"], want["nseg"]) and torch.equal(got["seg_id"], want["seg_id"])
    assert torch.equal(got["seg_t"].view(torch.int32), want["seg_t"].view(torch.int32))


@pytest.mark.parametrize("count", [False, True])
def test_blocks_beyond_the_device_cost_nothing(ctx, count):
    """64 blocks of 256 threads a CU against 8, most of which find no ray: 3.6
    times the frame's time when each of their waves asked one counter, and twice
    and more when each added to the visits of a counting frame."""
    bvh = sphere(ctx, 4)
    cam = N.Camera.make((0.0, 0.0, -3.0), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 45.0)

    def frame(per_cu):
        torch.cuda.synchronize()
        t = time.perf_counter()
        bvh.pathtrace(cam, 1280, 720, 4, 8, ray_fetch=2, trace_block=256, blocks_per_cu=per_cu, stack_mode=2,
                      ring_depth=8, count_visits=count)
        torch.cuda.synchronize()
        return time.perf_counter() - t

    times = {n: min(frame(n) for _ in range(8)) for n in (8, 64)}
    print(times, flush=True)
    assert times[64] < 1.5 * times[8]
