"""Direct shuffles whose boxes share lines of memory - one side holds whole rows, the other parts of them - on
both sides of the rules that group them: every element moves (on the CPU, through the launch audit), and what
arrives equals the packed shuffle's bit for bit."""
import pytest

import test_gpu_direct as direct
import test_gpu_shuffle as cases
import test_host_direct_launch_audit as audits

_SAMPLES4, _SAMPLES8, _SAMPLES16 = ([1, 1, 1, n] for n in (4, 8, 16))

# (shape, source, destination): locale grid, split, overlap; innermost dimension first
LINES = {
    "parts of 6 and 7": ((26, 20, 9, 19), (_SAMPLES16, None, None), ([4, 4, 1, 1], None, None)),
    "halos": ((35, 30, 5, 9), (_SAMPLES8, None, None), ([2, 4, 1, 1], None, [1, 1, 0, 0])),
    "split source": ((26, 37, 3, 8), ([4, 2, 1, 1], None, [1, 1, 0, 0]), (_SAMPLES8, None, None)),
    "both split": ((29, 11, 6, 8), ([2, 1, 1, 4], None, None), ([8, 1, 1, 1], None, None)),
    "less than a vector": ((7, 70, 3, 4), (_SAMPLES4, None, None), ([4, 1, 1, 1], None, None)),
    "sixteen parts": ((67, 5, 4, 16), (_SAMPLES16, None, None), ([16, 1, 1, 1], None, None)),
    "too many parts": ((67, 5, 4, 20), ([1, 1, 1, 20], None, None), ([20, 1, 1, 1], None, None)),
    "empty ranks": ((21, 9, 5, 3), (_SAMPLES4, None, None), ([4, 1, 1, 1], None, None)),
    "parts of rows together": ((13, 9, 40, 4), (_SAMPLES4, None, None), ([1, 4, 1, 1], None, None)),
    "longest grouped": ((509, 3, 5, 4), (_SAMPLES4, None, None), ([2, 2, 1, 1], None, None)),
    "too long": ((2060, 3, 2, 4), (_SAMPLES4, None, None), ([2, 2, 1, 1], None, None)),
    "whole lines of memory": ((256, 6, 2, 4), (_SAMPLES4, None, None), ([2, 2, 1, 1], None, None)),
    "3-D": ((22, 9, 7, 3, 8), ([1, 1, 1, 1, 8], None, None), ([2, 2, 2, 1, 1], None, [1, 1, 1, 0, 0])),
    "channels too": ((18, 10, 8, 4), ([1, 1, 2, 2], None, None), ([2, 1, 2, 1], None, None)),
}


@pytest.mark.parametrize("name", LINES)
def test_every_element_moves(name, monkeypatch):
    from dihydrogen_amd import layers
    monkeypatch.setattr(layers, "_share_a_gpu", lambda tensors: True)
    monkeypatch.setattr(cases, "CASES", {name: LINES[name]})
    for dtype in ("float32", "int16"):
        audits.test_a_direct_shuffle_moves_every_element(dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float32", "int16", "float64"])
def test_equal_to_the_packed_shuffle(dtype, monkeypatch):
    streamed = ((130, 128, 33, 33), (_SAMPLES4, None, None), ([2, 2, 1, 1], None, None))
    monkeypatch.setattr(cases, "CASES", {**LINES, **({"streamed": streamed} if dtype == "float32" else {})})
    direct.test_direct_shuffles_equal_the_packed_ones(dtype, monkeypatch)
