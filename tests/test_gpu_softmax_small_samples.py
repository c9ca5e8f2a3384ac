"""Channel softmax of samples of a few tiles of 64 lanes, counted through all samples: the pixels around the
edges of samples and tiles, against softmax in float64 (the bounds are those of the streamed tensors)."""
import pytest

import test_gpu_softmax_streamed as streamed

pytestmark = pytest.mark.gpu

# N, C, H, W: samples of 128 pixels (fewer are counted pixel by pixel) to 1090, in 1 to 18 tiles
CASES = [(1, 40, 8, 16), (3, 40, 8, 16), (65, 33, 3, 43), (2, 100, 12, 16), (9, 100, 11, 35), (5, 64, 24, 24), (32, 300, 14, 14),
         (7, 400, 29, 31), (3, 384, 14, 13), (3, 385, 14, 13), (13, 260, 27, 40), (2, 1100, 13, 13), (6, 700, 10, 109), (4, 50, 2, 224)]


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("shape", CASES)
def test_samples_of_a_few_tiles(shape, dtype):
    streamed.test_streamed_softmax(shape, dtype)
