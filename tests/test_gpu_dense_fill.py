"""A dense volume's grid on the device (flg_volume_create, flg_volume_update):
every voxel, the zero border and the majorant, at the edges of the columns that
a lane fills."""
import time

import pytest
import torch

from fledge_amd import _native as N
from fledge_amd import api

pytestmark = pytest.mark.gpu

BOX = [0, 0, 0, 1, 1, 1]


def scene():
    return api.vol_scene(N.Camera.make((0.5, 0.5, -1.5), (0.5, 0.5, 0.0), (0.0, 1.0, 0.0), 45.0))


# columns of 8 quads for nz + 1 of them: one short, full, one over; thin grids;
# one whose quads are more than 256 MB
@pytest.mark.parametrize("shape", [(6, 5, 5), (7, 3, 9), (8, 9, 2), (1, 1, 1), (300, 1, 1), (1, 300, 1), (1, 1, 300),
                                   (63, 31, 17), (261, 250, 260)])
@pytest.mark.parametrize("peak", [(0, 0, 0), (-1, -1, -1)])
def test_dense_fill(ctx, shape, peak):
    """Radiance and lookups bit-equal to the sparse volume of the same grid,
    whose bricks are stored by another kernel; the greatest voxel in a corner."""
    print("dense fill", shape, peak, flush=True)
    g = torch.rand(shape, generator=torch.Generator().manual_seed(5)) + 0.01
    g[peak] = 3.0
    g = g.cuda()
    dense = api.Volume(ctx, torch.zeros_like(g), BOX, 6.4, 1.6, 0.3)
    dense.update(g)
    sparse = api.Volume.sparse(ctx, *api.leaves_of(g), shape, BOX, 6.4, 1.6, 0.3)
    a, sa = dense.render(scene(), 40, 40, 8, 16, stats=True)
    b, sb = sparse.render(scene(), 40, 40, 8, 16, stats=True)
    assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    assert sa == sb and sa["lookups"] > 0


def test_update_is_bound_by_its_writes(ctx):
    """An update of 512^3 voxels in less than twice the time of writing its quads'
    bytes once (it took 2.8 times that)."""
    g = torch.rand((512, 512, 512), device="cuda")
    vol = api.Volume(ctx, g, BOX, 6.4, 1.6, 0.3)
    quads = torch.empty((513, 513, 514, 4), dtype=torch.float32, device="cuda")

    def best(f):
        times = []
        for _ in range(8):
            torch.cuda.synchronize()
            t = time.perf_counter()
            f()
            torch.cuda.synchronize()
            times.append(time.perf_counter() - t)
        return min(times)

    update, write = best(lambda: vol.update(g)), best(lambda: quads.zero_())
    print(update, write, flush=True)
    assert update < 2.0 * write
