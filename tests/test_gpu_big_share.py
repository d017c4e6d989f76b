"""Large triangles whose rows several waves share: every ratio of queued
triangles to waves (the limits of the split, waves left over, more triangles
than lanes), narrow, wide and clip-crossing ones, against the oracle; keys,
shadow depth bits and covered samples are integers and must be equal."""
import pytest

from .test_gpu_raster_edges import _check, _scene, _soup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alpha", [False, True])
@pytest.mark.parametrize("blocks", [1, 2, 3, 5, 33])
def test_waves_per_triangle(blocks, alpha):
    for extent, count in ((20.0, 12), (20.0, 300), (66.0, 70), (150.0, 9), (150.0, 40), (1200.0, 12)):
        print(f"case: {blocks} blocks, {count} triangles of {extent} px, alpha {alpha}", flush=True)
        _check(_scene(_soup(extent, count, 11), alpha),
               {"tile_raster": 0, "medium_extent_px": 8, "small_extent_px": 8, "big_blocks": blocks})
