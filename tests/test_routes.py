"""Which calls the routing hands to which kernels, and which it refuses, on the
CPU: the checks run, nothing is launched."""

import pytest
import torch

from sunshape_mlx_amd import _hip


@pytest.fixture
def no_launch(monkeypatch):
    """CPU tensors pass for GPU ones, and a codebook launch fails the test."""
    class Lib:
        def __getattr__(self, name):
            return getattr(real, name)

        def ss_codebook_f16x2(self, *args):
            pytest.fail("a refused codebook shape was launched")

    real = _hip.load_library()
    monkeypatch.setattr(_hip, "require_gpu", lambda *t: None)
    monkeypatch.setattr(_hip, "load_library", lambda: Lib())
    monkeypatch.setattr(_hip, "stream_handle", lambda device=None: 0)


@pytest.mark.parametrize("shape", [(32, 256, 4), (8, 256, 16), (16, 256, 1)])
def test_codebooks_of_other_block_dims_are_refused_before_a_launch(no_launch, shape):
    """codebook_f16x2_kernel reads 8 floats a centroid: past the end of the
    tensor for smaller blocks."""
    with pytest.raises(_hip.SunShapeUnsupported):
        _hip.codebook_f16x2(torch.zeros(shape))


@pytest.mark.parametrize("shape", [(10, 256, 8), (14, 256, 8), (9, 256, 8), (68, 256, 8),
                                   (16, 257, 8), (2, 256, 8)])
def test_codebooks_of_other_sizes_are_unsupported(no_launch, shape):
    """A block count that is not a multiple of 4 (head dims 80, 112, 72) or
    too many centroids: the error after which a call takes its other route."""
    with pytest.raises(_hip.SunShapeUnsupported):
        _hip.codebook_f16x2(torch.zeros(shape))
