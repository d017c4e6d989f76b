"""The tiled raster's direct list: meshlets over more tiles than a bin entry
may name, which the large-triangle launch draws itself, several waves to each.
Sheets of narrow triangles over a 10x7-tile view, two of them with larger and
clip-crossing ones, against the oracle: keys, shadow depth bits and covered
samples are integers and must be equal."""
import numpy as np
import pytest

from lighthugger_amd import abi
from lighthugger_amd.frame import ViewConfig
from lighthugger_amd.scene import HostScene, Material, make_camera, make_uniforms
from oracle.compare import compare_frames, oracle_frame, snapshot

pytestmark = pytest.mark.gpu

W, H, S = 607, 413, 193


def _sheet(columns, x, y, seed):
    """A jittered sheet of 8x8 vertices (98 triangles, one meshlet) from pixel
    (x, y) of the plane 4 m before the camera, with the given column and row
    widths in pixels."""
    rng = np.random.default_rng(seed)
    m = 2 * 4.0 * np.tan(np.radians(30)) / H
    at = np.concatenate([[0.0], np.cumsum(columns)])
    px = np.stack(np.meshgrid(x + at, y + at), -1) + rng.uniform(-3, 3, (8, 8, 2))
    xy = (px - np.array([W, H]) / 2) * m
    pos = np.concatenate([xy, rng.uniform(-0.05, 0.05, (8, 8, 1))], -1).reshape(-1, 3).astype(np.float32)
    a = (np.arange(7)[:, None] * 8 + np.arange(7)[None]).ravel()
    idx = np.concatenate([np.stack([a, a + 1, a + 9], 1), np.stack([a, a + 9, a + 8], 1)]).astype(np.uint32)
    return pos, None, rng.uniform(0, 2, (64, 2)).astype(np.float32), idx


@pytest.mark.parametrize("hiz", [False, True])
@pytest.mark.parametrize("blocks", [1, 3, 33, 2048])
def test_meshlets_over_many_tiles(blocks, hiz):
    import torch

    from lighthugger_amd.lib import Renderer, get_tuning_classes, set_tuning_classes

    print(f"case: {blocks} blocks, hiz {hiz}", flush=True)
    sheets = [_sheet([45.0] * 7, 20, 10, 1), _sheet([50.0] * 7, 250, 60, 2), _sheet([58.0] * 7, -60, -80, 3),
              _sheet([12.0] * 7, 500, 300, 4), _sheet([40.0] * 6 + [200.0], 100, 40, 5),
              _sheet([50.0] * 6 + [9000.0], 30, 20, 6)]
    scene = HostScene.build(sheets, [Material((0.7, 0.6, 0.5), 0.6, 0.2)],
                            [(i, 0, np.eye(4, dtype=np.float32)) for i in range(len(sheets))])
    cam = make_camera((0.02, 0.01, 4.0), (0, 0, 0), W, H, sun_dir=(0.2, 0.3, 0.9))
    orc = oracle_frame(scene, ViewConfig(W, H, S, statistics=True), make_uniforms(cam, scene.num_instances))
    old = get_tuning_classes()
    try:
        new = get_tuning_classes()
        for t in new:
            t.tile_raster, t.medium_extent_px, t.small_extent_px, t.big_blocks = 1, 64, 8, blocks
        set_tuning_classes(new)
        for stats in (True, False):
            r = Renderer(scene, ViewConfig(W, H, S, statistics=stats, hiz=hiz))
            r.set_camera(cam)
            for _ in range(2):  # the second Hi-Z frame takes the first one's history
                r.frame()
                torch.cuda.synchronize()
                gpu = snapshot(r.view)
                assert int(gpu["counters"][abi.CNT_OVERFLOW]) == 0
                if not hiz:
                    compare_frames(gpu, orc, scene)
                    assert int(gpu["counters"][abi.CNT_TILE_DIRECT]) >= 3
                else:  # the draw lists keep Hi-Z's own order and counts
                    assert np.array_equal(gpu["visbuffer"], orc["visbuffer"])
                    assert np.array_equal(gpu["shadow"], orc["shadow"])
                if stats and not hiz:
                    for p in range(abi.NUM_PASSES):
                        k = abi.CNT_FRAGMENTS + p
                        assert int(gpu["counters"][k]) == int(orc["counters"][k]), p
    finally:
        set_tuning_classes(old)
