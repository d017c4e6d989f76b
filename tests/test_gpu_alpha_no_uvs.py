"""Alpha-clip meshes without a base-colour texture need no uvs: a raster of
their depths alone (a mesh info whose uv address is null, which no texture
asks for) gives the keys and shadow depths of the same mesh with uvs."""
import numpy as np
import pytest

from lighthugger_amd import abi
from lighthugger_amd.frame import ViewConfig
from lighthugger_amd.scene import HostScene, Material, make_camera

from .test_gpu_raster_edges import H, W, _soup

pytestmark = pytest.mark.gpu


def _depths(scene, texture_index, uvs):
    import torch

    from lighthugger_amd.lib import Renderer

    r = Renderer(scene, ViewConfig(W, H, 193))
    mi = r.scene.mesh_infos.copy()
    mi["base_color_texture_index"] = texture_index
    if not uvs:
        mi["uvs"] = 0
    r.scene.set_mesh_infos(mi)
    r.set_camera(make_camera((0.02, 0.01, 4.0), (0, 0, 0), W, H, sun_dir=(0.2, 0.3, 0.9)))
    r.call("lh_view_reset")
    r.call("lh_cull_instances")
    r.call("lh_cull_meshlets", 0)
    for name in ("lh_raster_view", "lh_depth_bounds", "lh_fit_cascades", "lh_cull_instances_shadow"):
        r.call(name)
    for c in range(abi.NUM_CASCADES):
        r.call("lh_cull_meshlets", 1 + c)
        r.call("lh_raster_shadow", c)
    torch.cuda.synchronize()
    return r.view.visbuffer(), r.view.shadow_maps()


@pytest.mark.parametrize("texture_index", [abi.UNUSED_TEXTURE_INDEX, 3])  # 3: past the scene's textures
@pytest.mark.parametrize("extent", [4.4, 20.0, 150.0, 1200.0])
def test_untextured_alpha_clip_reads_no_uvs(extent, texture_index):
    print(f"case: extent {extent} texture {texture_index}", flush=True)
    scene = HostScene.build([_soup(extent, 60, 7)], [Material((0.7, 0.6, 0.5), 0.6, 0.2, alpha_clip=True)],
                            [(0, 0, np.eye(4, dtype=np.float32))])
    want = _depths(scene, texture_index, True)
    got = _depths(scene, texture_index, False)
    assert (want[0] != np.uint64(abi.LH_VISBUFFER_CLEAR)).any()
    for a, b in zip(want, got):
        assert np.array_equal(a, b)
