"""Limits at which the frame changes its way, and what it reports there: the
widest triangles of the 24-bit edge functions, views over 8,192 tiles, full
queues with the tiled raster, without it and in the second occlusion phase, and
instance lists that only a cascade overflows.  Against the oracle, or one
raster against the other: keys, depths and counts are integers."""
import numpy as np
import pytest

from lighthugger_amd import abi
from lighthugger_amd.frame import ViewConfig
from lighthugger_amd.scene import HostScene, make_camera, make_uniforms
from oracle.compare import oracle_frame, snapshot

from .test_gpu_raster_edges import H, W, _check, _scene, _soup

pytestmark = pytest.mark.gpu

OVERFLOW_INSTANCES, OVERFLOW_BIG, OVERFLOW_CLIP = 0x1, 0x4, 0x8


@pytest.fixture
def tuning():
    """Sets fields of every class's tuning; restored afterwards."""
    from lighthugger_amd.lib import get_tuning_classes, set_tuning_classes

    saved = get_tuning_classes()

    def change(**fields):
        new = get_tuning_classes()
        for t in new:
            for k, v in fields.items():
                setattr(t, k, v)
        set_tuning_classes(new)

    yield change
    set_tuning_classes(saved)


def _frame(scene, cam, cfg):
    import torch

    from lighthugger_amd.lib import Renderer

    r = Renderer(scene, cfg)
    r.set_camera(cam)
    r.frame()
    torch.cuda.synchronize()
    return r


def _camera(w=W, h=H):
    return make_camera((0.02, 0.01, 4.0), (0, 0, 0), w, h, sun_dir=(0.2, 0.3, 0.9))


@pytest.mark.parametrize("axis", [0, 1])
def test_extents_around_120_px(axis):
    """Triangles of 120 px and up to 30 subpixels (1/256 px) more or less, so
    that the snapped extents take every value around the limit (30,720)."""
    m = 2 * 4.0 * np.tan(np.radians(30)) / H
    n = 61
    rng = np.random.default_rng(5)
    size = 120.0 + (np.arange(n) - 30) / 256.0
    long = np.stack([np.zeros(n), size, size * rng.uniform(0.1, 0.9, n)], 1)
    short = np.stack([np.zeros(n), rng.uniform(-6, 6, n), rng.uniform(10, 34, n)], 1)
    if axis:
        long, short = long[:, ::-1], short[:, ::-1]  # mirrored, and front-facing again
    at = rng.uniform(0, 1, (n, 1, 2)) * np.array([W - 126, H - 126])
    px = at + np.stack([long, short] if axis == 0 else [short, long], -1) + 3.0
    xy = (px - np.array([W, H]) / 2) * m
    pos = np.concatenate([xy, np.zeros((n, 3, 1))], -1).reshape(-1, 3).astype(np.float32)
    uv = rng.uniform(0, 2, (3 * n, 2)).astype(np.float32)
    mesh = (pos, None, uv, np.arange(3 * n, dtype=np.uint32).reshape(-1, 3))
    for alpha in (False, True):
        for fields in ({"tile_raster": 0, "medium_extent_px": 64}, {"tile_raster": 0, "medium_extent_px": 8},
                       {"tile_raster": 1, "medium_extent_px": 64}):
            print(f"case: axis {axis} alpha {alpha} {fields}", flush=True)
            _check(_scene(mesh, alpha), {**fields, "small_extent_px": 8})


@pytest.mark.parametrize("height", [4096, 4160])  # 8,192 and 8,320 tiles
def test_views_of_8192_tiles_and_more(height, tuning):
    import torch

    scene = HostScene.preset(abi.PRESET_SMALL, num_instances=64)
    w = 8192
    cam = make_camera((0, 20, 60), (0, 0, 0), w, height)
    keys = []
    for tile in (1, 0):
        print(f"case: {w}x{height} tile_raster {tile}", flush=True)
        tuning(tile_raster=tile, medium_extent_px=32)
        r = _frame(scene, cam, ViewConfig(w, height, 64, ldr=False))
        c = r.view.counters()
        assert int(c[abi.CNT_OVERFLOW]) == 0
        assert (int(c[abi.CNT_TILE_ITEMS]) > 0) == (tile == 1)
        o = r.view.offsets["visbuffer"]
        keys.append(r.view.handle[0][o: o + r.view.sizes["visbuffer"]].view(torch.int64).clone())
        del r
    assert bool((keys[0] != -1).any())
    assert torch.equal(keys[0], keys[1])


def test_full_queue_is_reported_where_triangles_are_missing(tuning):
    scene = _scene(_soup(20.0, 300, 11), False)
    tuning(tile_raster=1, medium_extent_px=16, small_extent_px=8)
    c = _frame(scene, _camera(), ViewConfig(W, H, 193, big_capacity=7)).view.counters()
    assert int(c[abi.CNT_OVERFLOW]) == OVERFLOW_BIG
    # over 120 px and neither queue with a place left: a clip overflow
    scene = _scene(_soup(150.0, 40, 11), False)
    tuning(tile_raster=0)
    c = _frame(scene, _camera(), ViewConfig(W, H, 193, big_capacity=1, clip_capacity=1)).view.counters()
    assert int(c[abi.CNT_OVERFLOW]) == OVERFLOW_CLIP
    assert int(c[abi.CNT_BIG]) > 1


@pytest.mark.parametrize("alpha", [False, True])
def test_full_queue_in_both_occlusion_phases(alpha, tuning):
    import torch

    tuning(tile_raster=0)
    for extent, count in ((40.0, 300), (150.0, 40)):
        print(f"case: {count} triangles of {extent} px alpha {alpha}", flush=True)
        scene = _scene(_soup(extent, count, 11), alpha)
        orc = oracle_frame(scene, ViewConfig(W, H, 193), make_uniforms(_camera(), scene.num_instances))
        r = _frame(scene, _camera(), ViewConfig(W, H, 193, big_capacity=7, hiz=True))
        for _ in range(2):
            gpu = snapshot(r.view)
            assert int(gpu["counters"][abi.CNT_OVERFLOW]) == 0
            assert int(gpu["counters"][abi.CNT_BIG + 1]) > 7  # (the second phase empties the main view's count)
            assert np.array_equal(gpu["visbuffer"], orc["visbuffer"])
            assert np.array_equal(gpu["shadow"], orc["shadow"])
            r.frame()
            torch.cuda.synchronize()


@pytest.mark.parametrize("instances", [200, 300])  # the cascade cull fused with the fit, and by itself
def test_instance_overflow_of_a_cascade(instances):
    scene = HostScene.preset(abi.PRESET_SMALL, num_instances=instances)
    cam = make_camera((10, 5, 10), (14, 4, 12), 96, 64)
    orc = oracle_frame(scene, ViewConfig(96, 64, 64), make_uniforms(cam, scene.num_instances))
    counts = [orc[f"prefix{p}"][0] for p in range(abi.NUM_PASSES)]
    cap = counts[0] + 2
    assert max(counts[1:]) > cap
    r = _frame(scene, cam, ViewConfig(96, 64, 64, instance_capacity=cap))
    assert int(r.view.counters()[abi.CNT_OVERFLOW]) & OVERFLOW_INSTANCES
    for p in range(abi.NUM_PASSES):
        count, total, vals = r.view.prefix(p)
        assert (count, total) == orc[f"prefix{p}"][:2], p  # the counts go on, in every sector
        # what was kept are visible instances, each once
        kept = set(vals["index"].tolist())
        assert len(kept) == min(count, cap) and kept <= set(orc[f"prefix{p}"][2]["index"].tolist()), p
