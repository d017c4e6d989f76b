"""Frames whose large-triangle queue is too small: the per-meshlet raster draws
what does not fit, narrow and wide, opaque and alpha-clipped, so keys, shadow
depth bits and covered samples stay the oracle's and nothing is reported lost."""
import pytest

from lighthugger_amd import abi
from lighthugger_amd.frame import ViewConfig
from lighthugger_amd.scene import make_camera, make_uniforms
from oracle.compare import compare_frames, oracle_frame, snapshot

from .test_gpu_raster_edges import H, W, _scene, _soup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alpha", [False, True])
@pytest.mark.parametrize("capacity", [1, 7, 64])
def test_small_large_triangle_queue(capacity, alpha):
    import torch

    from lighthugger_amd.lib import Renderer, get_tuning_classes, set_tuning_classes

    cam = make_camera((0.02, 0.01, 4.0), (0, 0, 0), W, H, sun_dir=(0.2, 0.3, 0.9))
    old = get_tuning_classes()
    try:
        new = get_tuning_classes()
        for t in new:
            t.tile_raster, t.medium_extent_px, t.small_extent_px = 0, 8, 8
        set_tuning_classes(new)
        for extent, count in ((20.0, 300), (66.0, 70), (150.0, 40), (1200.0, 12)):
            print(f"case: capacity {capacity}, {count} triangles of {extent} px, alpha {alpha}", flush=True)
            scene = _scene(_soup(extent, count, 11), alpha)
            orc = oracle_frame(scene, ViewConfig(W, H, 193, statistics=True), make_uniforms(cam, scene.num_instances))
            for stats in (True, False):
                r = Renderer(scene, ViewConfig(W, H, 193, statistics=stats, big_capacity=capacity))
                r.set_camera(cam)
                r.frame()
                torch.cuda.synchronize()
                gpu = snapshot(r.view)
                assert int(gpu["counters"][abi.CNT_OVERFLOW]) == 0
                compare_frames(gpu, orc, scene)
                if stats:
                    for p in range(abi.NUM_PASSES):
                        k = abi.CNT_FRAGMENTS + p
                        assert int(gpu["counters"][k]) == int(orc["counters"][k]), p
    finally:
        set_tuning_classes(old)
