"""Channel softmax up to 32 channels around the numbers of pixels and bytes where the pixels a lane serves change:
against softmax in float64 (the bounds are those of the streamed tensors)."""
import pytest

import test_gpu_softmax_streamed as streamed

pytestmark = pytest.mark.gpu

# N, C, H, W
CASES = [(1, 17, 192, 256), (1, 17, 193, 256), (1, 16, 64, 64), (1, 32, 3, 43), (1, 12, 256, 256), (1, 12, 257, 256), (1, 11, 64, 64),
         (2, 32, 71, 72), (300, 20, 7, 7), (1, 9, 511, 512), (1, 9, 512, 512), (15, 5, 256, 256), (16, 5, 256, 256), (17, 16, 256, 256)]


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("shape", CASES)
def test_numbers_of_pixels(shape, dtype):
    streamed.test_streamed_softmax(shape, dtype)
