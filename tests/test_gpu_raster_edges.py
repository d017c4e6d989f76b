"""The raster's paths at their edges, against the oracle: triangle counts
around one and two rounds of 64 lanes and around a full triangle queue, boxes
around the in-lane limit (4 px), the run length, the medium extents and 64 px
(the widest box of the 24-bit edge functions), slivers and shapes that leave
the target on every side.  Keys, shadow depth bits and covered samples are
integers and must be equal."""
import numpy as np
import pytest

from lighthugger_amd import abi
from lighthugger_amd.frame import ViewConfig
from lighthugger_amd.scene import HostScene, Material, make_camera, make_uniforms
from oracle.compare import compare_frames, oracle_frame, snapshot

from .util import grid_patch

pytestmark = pytest.mark.gpu

W, H = 211, 157


def _soup(extent_px: float, count: int, seed: int):
    """`count` triangles of about `extent_px` pixels in a plane 4 m before the
    camera (60 degrees, H pixels high), some of them slivers, their centres
    spread over the view and a margin outside it; both windings."""
    rng = np.random.default_rng(seed)
    m = 2 * 4.0 * np.tan(np.radians(30)) / H  # metres per pixel at the plane
    centre = rng.uniform(-0.65, 0.65, (count, 1, 2)) * np.array([W, H]) * m
    angle = rng.uniform(0, 2 * np.pi, (count, 1)) + np.array([0, 2.1, 4.2]) * rng.choice([1, -1], (count, 1))
    r = 0.5 * extent_px * m * rng.uniform(0.9, 1.1, (count, 3))
    xy = np.stack([r * np.cos(angle), r * np.sin(angle)], -1)
    thin = rng.random(count) < 0.3
    xy[thin, 2] = xy[thin, 0] * 0.5 + xy[thin, 1] * 0.5 + 0.3 * m  # nearly on the opposite edge
    z = rng.uniform(-0.05, 0.05, (count, 3, 1))
    pos = np.concatenate([centre + xy, z], -1).reshape(-1, 3).astype(np.float32)
    uv = rng.uniform(0, 2, (3 * count, 2)).astype(np.float32)
    return pos, None, uv, np.arange(3 * count, dtype=np.uint32).reshape(-1, 3)


def _check(scene, tuning=None, shadow=193):
    import torch

    from lighthugger_amd.lib import Renderer, get_tuning_classes, set_tuning_classes

    cam = make_camera((0.02, 0.01, 4.0), (0, 0, 0), W, H, sun_dir=(0.2, 0.3, 0.9))
    cfg = ViewConfig(W, H, shadow, statistics=True)
    orc = oracle_frame(scene, cfg, make_uniforms(cam, scene.num_instances))
    old = get_tuning_classes()
    try:
        if tuning:
            new = get_tuning_classes()
            for t in new:
                for k, v in tuning.items():
                    setattr(t, k, v)
            set_tuning_classes(new)
        for stats in (True, False):
            r = Renderer(scene, ViewConfig(W, H, shadow, statistics=stats))
            r.set_camera(cam)
            r.frame()
            torch.cuda.synchronize()
            gpu = snapshot(r.view)
            compare_frames(gpu, orc, scene)
            if stats:
                for p in range(abi.NUM_PASSES):
                    k = abi.CNT_FRAGMENTS + p
                    assert int(gpu["counters"][k]) == int(orc["counters"][k]), p
    finally:
        set_tuning_classes(old)
    assert int(orc["counters"][abi.CNT_FRAGMENTS]) > 0


def _scene(mesh, alpha):
    texture = np.random.default_rng(3).integers(0, 256, (16, 16, 4)).astype(np.uint8)
    mat = Material((0.7, 0.6, 0.5), 0.6, 0.2, base_color_texture=0, alpha_clip=alpha)
    tr = np.eye(4, dtype=np.float32)
    return HostScene.build([mesh], [mat], [(0, 0, tr)], textures=[texture])


@pytest.mark.parametrize("alpha", [False, True])
@pytest.mark.parametrize("extent", [0.7, 1.6, 2.5, 4.4, 8.2, 17.0, 63.0, 64.4, 66.0, 150.0])
def test_triangle_extents(extent, alpha):
    print(f"case: extent {extent} alpha {alpha}", flush=True)
    scene = _scene(_soup(extent, 150, 7), alpha)
    for tuning in ({"tile_raster": 0, "medium_extent_px": 64, "small_extent_px": 8},
                   {"tile_raster": 0, "medium_extent_px": 8, "small_extent_px": 8},
                   {"tile_raster": 1, "medium_extent_px": 64, "small_extent_px": 1}):
        _check(scene, tuning)


@pytest.mark.parametrize("count", [1, 2, 63, 64, 65, 97, 98])
def test_triangle_counts(count):
    print(f"case: {count} triangles", flush=True)
    pos, nrm, uv, idx = grid_patch(7, 7)
    scene = _scene((pos * 1.7, nrm, uv, idx[:count]), False)
    for tile in (0, 1):
        _check(scene, {"tile_raster": tile})
