"""Large triangles in queues shorter and longer than half the grid, which deals
them out to blocks or to waves: a few triangles to a few hundred, narrow and
wide ones mixed, against the oracle; keys, shadow depth bits and covered
samples are integers and must be equal."""
import numpy as np
import pytest

from .test_gpu_raster_edges import _check, _scene, _soup

pytestmark = pytest.mark.gpu


def _mixed(parts):
    """Triangles of several extents in one mesh."""
    soups = [_soup(extent, count, 11 + i) for i, (extent, count) in enumerate(parts)]
    pos, uv = np.concatenate([p[0] for p in soups]), np.concatenate([p[2] for p in soups])
    return pos, None, uv, np.arange(len(pos), dtype=np.uint32).reshape(-1, 3)


@pytest.mark.parametrize("blocks", [1, 2, 7, 64, 350, 2048])
def test_dealt_to_blocks_or_waves(blocks):
    for parts in ([(150.0, 5)], [(1200.0, 3), (20.0, 30)], [(150.0, 40), (66.0, 40), (1200.0, 6)],
                  [(1200.0, 20), (20.0, 300), (150.0, 20)]):
        print(f"case: {blocks} blocks, triangles {parts}", flush=True)
        _check(_scene(_mixed(parts), False),
               {"tile_raster": 0, "medium_extent_px": 8, "small_extent_px": 8, "big_blocks": blocks})
