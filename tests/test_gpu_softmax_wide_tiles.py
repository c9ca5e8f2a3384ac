"""Channel softmax in tiles of 64 pixels, one or two pixels a lane, where tiles are many or tensors large: at the edges of
the channels that each tile holds, of rows that are whole vectors (streamed from 24 MiB on) and that are not, against float64."""
import pytest

import test_gpu_softmax_split as split

pytestmark = pytest.mark.gpu

EDGES = [65, 96, 97, 128, 129, 160, 161, 192, 193, 224, 225, 256]


# beyond the sizes for tiles of 16 and of 32 pixels; the second streams from 164 channels on, of doubles from 82
@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("spatial", [577 * 64 + 1, 600 * 64])
@pytest.mark.parametrize("c", EDGES + [257, 384, 385, 448, 449, 512])
def test_many_tiles(c, spatial, dtype):
    split._check(1, c, spatial, dtype)


# rows of two and of four elements a vector
@pytest.mark.parametrize("spatial", [600 * 128 + 2, 600 * 128])
@pytest.mark.parametrize("c", [33, 64] + EDGES)
def test_two_pixels_a_lane(c, spatial):
    split._check(1, c, spatial, "float32")


# streamed, and one pixel a lane: fewer tiles of 128 pixels than 512 forward, than 256 backward
@pytest.mark.parametrize("c,spatial", [(97, 508 * 128), (128, 508 * 128), (160, 400 * 128), (161, 400 * 128), (192, 400 * 128),
                                       (193, 255 * 128), (224, 255 * 128), (225, 255 * 128), (256, 255 * 128)])
def test_streamed_one_pixel_a_lane(c, spatial):
    split._check(1, c, spatial, "float32")


# at most 256 tiles and more than 16 MiB (20 of doubles): sixteen waves
@pytest.mark.parametrize("n,c,spatial,dtype", [
    (1, 300, 16382, "float32"), (1, 384, 16384, "float32"), (1, 385, 16382, "float32"), (2, 400, 8192, "float32"),
    (1, 512, 16382, "float32"), (1, 512, 16384, "float32"), (1, 513, 16382, "float32"), (1, 768, 16384, "float32"),
    (1, 769, 16383, "float32"), (1, 1024, 16384, "float32"), (3, 1024, 64 * 80 + 1, "float32"), (1, 1025, 16384, "float32"),
    (1, 192, 16383, "float64"), (1, 256, 16382, "float64"), (1, 256, 16383, "float64")])
def test_few_tiles_of_large_tensors(n, c, spatial, dtype):
    split._check(n, c, spatial, dtype)
