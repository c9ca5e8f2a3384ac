"""Softmax of samples that a wave or a workgroup holds, by their number: at the edges of the rule that chooses between the two, against float64."""
import pytest

import test_gpu_softmax_rows as rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("kind", ["instance", "channel"])
@pytest.mark.parametrize("n", [512, 768, 769, 2048, 2049])
def test_numbers_of_samples(n, kind, dtype):
    for size in (256, 257, 512, 513, 1025, 2048):
        rows._check(kind, n, size, dtype)
