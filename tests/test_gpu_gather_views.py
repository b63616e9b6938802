"""A batch launch that names no number of workgroups (a workgroup per block,
gather_views_kernel: the view is found from the block) against the persistent
launch and the single-view gather: the same bits, for one view, two, and more
than a power of two of them, with ragged extents and a view of one block."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from legitengine_amd import lgx  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from legitengine_amd import device
    device.require_device()
    return device


@pytest.mark.parametrize("sizes", [[(64, 48)], [(16, 16), (333, 187)],
                                   [(96, 64), (16, 16), (130, 70), (257, 33), (64, 64)]])
@pytest.mark.parametrize("tile,grid", [(0, 4), (28, 8)])
def test_block_per_workgroup_equals_persistent(dev, sizes, tile, grid):
    items, refs = [], []
    for i, (w, h) in enumerate(sizes):
        sc = lgx.make_scene(70 + i, 8, 2)
        view, proj = lgx.scene_matrices(sc, w, h)
        g = dev.GBufferDev.alloc(w, h, "mixed").render(sc)
        pyr = dev.PyramidDev(g, 4, lgx.SAMPLER_HIZ_POINT).build()
        ga = dev.Gather(w, h, 4, 0, lgx.SAMPLER_HIZ_POINT, grid=grid, footprint_dirs=64, tile=tile)
        refs.append(ga(view, proj, g, pyr).numpy())
        items.append((ga, g, pyr, dev.DImage(w, h, lgx.RGBA32F), view, proj))
    gb = dev.GatherBatch(items)
    gb.set_tile(tile)
    for wg in (0, 8, 0):
        for it in items:
            it[3].t.fill_(-1.0)
        gb.launch(wg)
        torch.cuda.synchronize()
        for it, ref in zip(items, refs):
            assert it[3].numpy().tobytes() == ref.tobytes(), wg
    gb.close()
