"""Large-triangle queues only as long as the triangles over 16 px (over 64 px in a
batch) need, whatever lower extents the tuning selects for longer queues, with
the least clip queue: narrow triangles between the extents may not take the
wide ones' places.  Opaque and alpha-clipped, single views and a batch, against
the oracle; nothing is reported lost."""
import numpy as np
import pytest

from lighthugger_amd import abi
from lighthugger_amd.frame import ViewConfig
from lighthugger_amd.scene import make_camera, make_uniforms
from oracle.compare import compare_frames, oracle_frame, snapshot

from .test_gpu_big_dealing import _mixed
from .test_gpu_raster_edges import H, _scene

pytestmark = pytest.mark.gpu


def _check(view, scene, orc, print_as):
    gpu = snapshot(view)
    print(f"case: {print_as}: big {gpu['counters'][8:10]} clip {gpu['counters'][16:18]}", flush=True)
    assert (orc["visbuffer"] != np.uint64(abi.LH_VISBUFFER_CLEAR)).any()
    assert int(gpu["counters"][abi.CNT_OVERFLOW]) == 0
    compare_frames(gpu, orc, scene)


@pytest.mark.parametrize("alpha", [False, True])
def test_view_queue_for_16_px(alpha):
    import torch

    from lighthugger_amd.lib import Renderer

    w, h = 1000, 700  # the class whose extent is lowest
    scene = _scene(_mixed([((9.0 if alpha else 13.6) * H / h, 700), (150.0 * H / h, 40)]), alpha)
    cam = make_camera((0.02, 0.01, 4.0), (0, 0, 0), w, h, sun_dir=(0.2, 0.3, 0.9))
    orc = oracle_frame(scene, ViewConfig(w, h, 193), make_uniforms(cam, scene.num_instances))
    r = Renderer(scene, ViewConfig(w, h, 193, big_capacity=41 if not alpha else 41 * abi.NUM_CASCADES, clip_capacity=1))
    r.set_camera(cam)
    r.frame()
    torch.cuda.synchronize()
    _check(r.view, scene, orc, f"alpha {alpha}")


@pytest.mark.parametrize("alpha", [False, True])
def test_batch_queue_for_64_px(alpha):
    import torch

    from lighthugger_amd.lib import BATCH_BATCHED, BatchRenderer

    w, h = 500, 350
    scene = _scene(_mixed([(45.0 * H / h, 300), (150.0 * H / h, 40)]), alpha)
    cams = [make_camera((0.02 + 0.1 * i, 0.01, 4.0), (0, 0, 0), w, h, sun_dir=(0.2, 0.3, 0.9)) for i in range(3)]
    b = BatchRenderer(scene, cams, shadow_sizes=[193] * 3, big_capacity=41 if not alpha else 41 * abi.NUM_CASCADES,
                      clip_capacity=1)
    b.run(BATCH_BATCHED)
    torch.cuda.synchronize()
    for i, cam in enumerate(cams):
        orc = oracle_frame(scene, ViewConfig(w, h, 193), make_uniforms(cam, scene.num_instances))
        _check(b.views[i], scene, orc, f"batch view {i} alpha {alpha}")
    b.close()
