"""Frames of small scenes, whose reset, culls and cascade fit share launches:
instance counts around a wave, the limits of the two fused launches (256 and
1,024 instances) and beyond them, against the oracle (visible sets, keys,
shadow depths and cascades exact), replayed on the same view, and with an
instance capacity that overflows."""
import numpy as np
import pytest

from lighthugger_amd import abi
from lighthugger_amd.frame import ViewConfig
from lighthugger_amd.scene import HostScene, make_camera, make_uniforms
from oracle.compare import compare_frames, oracle_frame, snapshot

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("instances", [1, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025])
def test_instance_counts(instances):
    import torch

    from lighthugger_amd.lib import Renderer

    print(f"case: {instances} instances", flush=True)
    scene = HostScene.preset(abi.PRESET_SMALL, num_instances=instances)
    cfg = ViewConfig(161, 97, 128)
    r = Renderer(scene, cfg)
    for pos, target in (((0, 20, 80), (0, 0, 0)), ((60, 10, 20), (0, 0, 0)), ((0, 0, 200), (0, 0, 400))):
        cam = make_camera(pos, target, cfg.width, cfg.height)  # the last one sees nothing
        r.set_camera(cam)
        orc = oracle_frame(scene, cfg, make_uniforms(cam, scene.num_instances))
        for _ in range(2):
            r.frame()
            torch.cuda.synchronize()
            gpu = snapshot(r.view)
            assert int(gpu["counters"][abi.CNT_FLAGS]) == int(orc["counters"][abi.CNT_FLAGS])
            if not orc["counters"][abi.CNT_FLAGS] & abi.FLAG_EMPTY_VIEW:
                compare_frames(gpu, orc, scene)
            else:
                assert np.array_equal(gpu["visbuffer"], orc["visbuffer"])


def test_instance_overflow_is_reported():
    import torch

    from lighthugger_amd.lib import Renderer

    scene = HostScene.preset(abi.PRESET_SMALL, num_instances=200)
    cam = make_camera((0, 20, 80), (0, 0, 0), 96, 64)
    r = Renderer(scene, ViewConfig(96, 64, 64, instance_capacity=3))
    r.set_camera(cam)
    r.frame()
    torch.cuda.synchronize()
    counters = r.view.counters()
    assert int(counters[abi.CNT_OVERFLOW]) & 0x1  # LH_OVERFLOW_INSTANCES
    assert r.view.prefix(0)[0] > 3  # the count goes on, the writes do not
