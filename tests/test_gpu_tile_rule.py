"""The tile shapes a domain starts with, on both sides of every size in the rule, and the names the shapes go by."""
import numpy as np
import pytest

from mithra_amd import abi
from test_gpu_flat_fields import coeffs
from test_gpu_fields import grid

pytestmark = pytest.mark.gpu

FP64, FP32 = abi.PRECISION_FP64, abi.PRECISION_FP32_BULK


# N1 = 128 fills the 64-node rows, 147 wastes a quarter of their lanes
@pytest.mark.parametrize("nodes,precision,tiles", [
    ((131, 147, 259), FP64, (0, 0, 0)), ((131, 147, 260), FP64, (7, 0, 0)),      # 5.0 million nodes
    ((131, 147, 415), FP64, (7, 0, 0)), ((131, 147, 416), FP64, (7, 7, 0)),      # 8.0
    ((128, 128, 488), FP64, (7, 0, 0)), ((128, 128, 489), FP64, (7, 8, 0)),
    ((128, 128, 976), FP64, (7, 8, 0)), ((128, 128, 977), FP64, (7, 8, 1)),      # 16.0
    ((128, 147, 851), FP64, (7, 7, 0)),
    ((131, 147, 260), FP32, (0, 0, 0)), ((128, 128, 976), FP32, (0, 0, 0)),
    ((128, 128, 977), FP32, (0, 8, 1)), ((128, 147, 851), FP32, (0, 0, 0)),
])
def test_starting_shapes(nodes, precision, tiles):
    dom = abi.Domain(grid(*nodes, 0), coeffs(np.random.default_rng(1)), precision=precision)
    assert dom.tiles() == tiles
    dom.set_tiles(3, 4)
    dom.set_fused_tile(2)
    assert dom.tiles() == (3, 4, 2)
    dom.close()


def test_shape_names():
    """The flat form has no rows of its own, and every shape is told apart from the others but for the
    LDS-staged forms, which share the rows and planes of tiled ones."""
    shapes = [abi.tile_shape(v) for v in range(abi.TILE_VARIANTS)]
    assert shapes[0] == (0, 8)
    assert all(r > 0 and k > 0 for r, k in shapes[1:])
    assert len(set(shapes[:7])) == 7
