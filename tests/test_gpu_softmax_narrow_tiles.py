"""Channel softmax in tiles of 16 and of 32 pixels, whose lanes share the channels of a wave: at the edges of the tiles,
of the channels that each holds, and of the sizes for which they are taken, against float64."""
import pytest

import test_gpu_softmax_split as split

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("c", [65, 67, 97, 98, 99, 127, 130, 194, 386, 514, 767, 770, 1023])
@pytest.mark.parametrize("n,spatial", [(1, 2), (1, 129), (3, 143), (2, 145), (17, 15), (1, 16 * 40)])
def test_sixteen_pixels(c, n, spatial, dtype):
    split._check(n, c, spatial, dtype)


# 256 and 257 tiles of 64 pixels, 512 and 513; the most elements for sixteen pixels a tile, and more
@pytest.mark.parametrize("n,c,spatial,dtype", [
    (1, 97, 256 * 64, "float32"), (1, 97, 256 * 64 + 1, "float32"), (1, 256, 256 * 64, "float32"), (1, 257, 256 * 64, "float32"),
    (1, 65, 257 * 64 - 31, "float32"), (1, 384, 257 * 64 - 33, "float32"), (128, 385, 65 * 2, "float32"),
    (1, 96, 300 * 64, "float32"), (1, 97, 300 * 64 - 47, "float32"), (1, 129, 383 * 64 + 1, "float32"), (1, 161, 385 * 64 - 1, "float32"),
    (1, 193, 576 * 64 - 15, "float32"), (1, 256, 577 * 64, "float32"), (1, 225, 600 * 64 - 1, "float32"), (11, 135, 45 * 61, "float32"),
    (1, 448, 600 * 64 - 1, "float32"), (1, 449, 600 * 64 - 1, "float32"), (1, 66, 512 * 64 - 1, "float32"), (1, 66, 512 * 64 + 1, "float32"), (300, 70, 107, "float32"), (1, 130, 300 * 64, "float32"),
    (1, 160, 256 * 64, "float64"), (1, 161, 256 * 64, "float64"), (1, 193, 256 * 64, "float64"), (1, 65, 257 * 64 - 31, "float64"),
    (1, 256, 400 * 64 - 33, "float64"), (1, 257, 600 * 64 - 33, "float64"), (2, 386, 300 * 64 + 2, "float64"),
    (1, 512, 513 * 64 + 31, "float64"), (1, 513, 257 * 64 + 1, "float64"), (1, 256, 513 * 64, "float64"),
])
def test_sizes_between_the_ways(n, c, spatial, dtype):
    split._check(n, c, spatial, dtype)
