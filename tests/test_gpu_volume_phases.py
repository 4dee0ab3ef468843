"""The volume integrator's phased schedule against one lane per path, at the
frame sizes and media where it can go wrong."""
import time

import pytest
import torch

from fledge_amd import _native as N
from fledge_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,spp,depth,film", [(1, 1, 1, 4, 0), (3, 1, 2, 4, 1), (8, 8, 1, 32, 0), (33, 17, 3, 32, 1),
                                                (130, 2, 2, 6, 0)])
@pytest.mark.parametrize("bias", [0.5, 0.02])
def test_phased_schedule_small_frames(ctx, w, h, spp, depth, film, bias):
    """Schedule 2's phases and wave-wide long walks against one lane per path:
    fewer paths than a wave, a part of a wave, the first Halton indices (walks
    of thousands of steps), a nearly empty medium (long ratio walks) and film
    tasks; bits and lookup counts equal."""
    print("phased %dx%d spp %d depth %d film %d bias %g" % (w, h, spp, depth, film, bias), flush=True)
    grid = api.gen_fbm_grid(20, seed=11, bias=bias)
    grid[3:5, 4:9, :] = 0.0
    vol = api.Volume(ctx, torch.from_numpy(grid).cuda(), [0, 0, 0, 1, 1, 1], 6.4, 1.6, 0.3)
    scene = api.vol_scene(N.Camera.make((0.5, 0.5, -1.5), (0.5, 0.5, 0.0), (0.0, 1.0, 0.0), 45.0))
    a, sa = vol.render(scene, w, h, spp, depth, schedule=1, film=film, stats=True)
    b, sb = vol.render(scene, w, h, spp, depth, schedule=2, film=film, stats=True)
    assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    assert sa == sb


@pytest.mark.parametrize("w", [1024, 1025])
def test_paths_claimed_at_once(ctx, w):
    """The largest launch whose waves claim one path per lane on 256 CUs
    (655,360 paths), and one beyond it: bits of one lane per path."""
    print("claims %dx640" % w, flush=True)
    grid = api.gen_fbm_grid(20, seed=11)
    vol = api.Volume(ctx, torch.from_numpy(grid).cuda(), [0, 0, 0, 1, 1, 1], 6.4, 1.6, 0.3)
    scene = api.vol_scene(N.Camera.make((0.5, 0.5, -1.5), (0.5, 0.5, 0.0), (0.0, 1.0, 0.0), 45.0))
    a = vol.render(scene, w, 640, 1, 3, schedule=1)
    b = vol.render(scene, w, 640, 1, 3, schedule=2)
    assert torch.equal(a.view(torch.int32), b.view(torch.int32))


def test_small_frame_of_a_constant_grid_is_not_slower(ctx):
    """65,536 paths whose walks are a step each: the phases had taken 1.4 times
    one lane per path, with two paths a lane in half of the waves."""
    vol = api.Volume(ctx, torch.ones((64, 64, 64), device="cuda"), [0, 0, 0, 1, 1, 1], 6.4, 1.6, 0.3)
    scene = api.vol_scene(N.Camera.make((0.5, 0.5, -1.5), (0.5, 0.5, 0.0), (0.0, 1.0, 0.0), 45.0))

    def frame(schedule):
        torch.cuda.synchronize()
        t = time.perf_counter()
        vol.render(scene, 128, 128, 4, 32, schedule=schedule)
        torch.cuda.synchronize()
        return time.perf_counter() - t

    times = {k: min(frame(k) for _ in range(8)) for k in (1, 2)}
    print(times, flush=True)
    assert times[2] < 1.2 * times[1]
