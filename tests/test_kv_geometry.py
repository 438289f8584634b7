"""kv_geometry (the fused quantizers' strides) addresses the same elements as
canonicalize for every K/V layout the adapters accept."""
import numpy as np
import pytest
import torch

from origami_amd.quantization.cachegen_adapter import canonicalize, kv_geometry

SHAPES = [(2, 3, 4, 2, 8), (3, 2, 4, 2, 8), (3, 4, 2, 2, 8), (2, 12, 2, 8), (12, 2, 2, 8),
          (2, 2, 130, 8), (2, 2, 4, 2, 8), (2, 1, 1, 1, 8), (1, 2, 5, 3, 16), (2, 130, 131, 8)]


@pytest.mark.parametrize("shape", SHAPES)
def test_geometry_matches_canonicalize(shape):
    kv = torch.arange(int(np.prod(shape)), dtype=torch.int64).reshape(shape)
    want, name = canonicalize(kv)
    got_name, (T, H, D), (half, block, token, head, bs) = kv_geometry(kv)
    assert got_name == name and (T, H, D) == tuple(want.shape[1:])
    t = torch.arange(T)
    at = (torch.arange(2)[:, None, None, None] * half
          + ((t // bs) * block + (t % bs) * token)[None, :, None, None]
          + torch.arange(H)[None, None, :, None] * head + torch.arange(D))
    assert torch.equal(kv.reshape(-1)[at], want)


def test_geometry_rejects_what_canonicalize_rejects():
    for shape in [(3, 3, 4), (3, 3, 3, 8), (3, 3, 3, 3, 8)]:
        with pytest.raises(ValueError):
            kv_geometry(torch.zeros(shape))
