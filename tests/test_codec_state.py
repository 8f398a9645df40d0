"""State that a codec keeps from call to call follows its tensors."""

import numpy as np
import pytest
import torch

import sunshape_mlx_amd as S


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("how", ["replaced", "in_place", "memory", "inference"])
def test_scoring_centroids_follow_the_heavy_mask(how, device):
    rng = np.random.default_rng(3)
    codec = S.SunShapeBlockCodec(32, n_centroids=4, device=device,
                                 mode="profileperm_mixed_precision", heavy_fp16=True)
    codec.load_state_dict({"centroids": rng.standard_normal((4, 4, 8)).astype(np.float32),
                           "permutation": np.arange(32, dtype=np.int32),
                           "mixed_high_precision_blocks": np.zeros(4, bool)})
    if how == "inference":
        with torch.inference_mode():
            codec.mixed_high_precision_blocks = torch.zeros(4, dtype=torch.bool, device=device)
            assert codec.scoring_centroids() is codec.centroids and codec.heavy_dims() is None
        return
    for heavy in ([], [1], [1, 3], []):
        mask = torch.zeros(4, dtype=torch.bool, device=device)
        mask[heavy] = True
        if how == "replaced":
            codec.mixed_high_precision_blocks = mask
        elif how == "memory":
            codec.mixed_high_precision_blocks.data = mask
        else:
            codec.mixed_high_precision_blocks.copy_(mask)
        for _ in range(2):
            got = codec.scoring_centroids()
            assert [b for b in range(4) if not got[b].any()] == heavy
            assert (got is codec.centroids) == (codec.heavy_dims() is None) == (not heavy)


def test_scoring_centroids_follow_an_array_shared_with_the_heavy_mask():
    rng = np.random.default_rng(3)
    codec = S.SunShapeBlockCodec(32, n_centroids=4, device="cpu",
                                 mode="profileperm_mixed_precision", heavy_fp16=True)
    codec.load_state_dict({"centroids": rng.standard_normal((4, 4, 8)).astype(np.float32),
                           "permutation": np.arange(32, dtype=np.int32)})
    shared = np.zeros(4, bool)
    codec.mixed_high_precision_blocks = torch.from_numpy(shared)
    assert codec.scoring_centroids() is codec.centroids
    shared[2] = True
    assert not codec.scoring_centroids()[2].any() and codec.heavy_dims() is not None
