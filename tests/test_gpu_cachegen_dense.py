"""The dense CacheGen restore at the edges of its tiles (16 tokens x all heads), with
head rows of a power of two of groups and not, every symbol width, streams at any byte,
a short segment, and more segments than one launch takes, against the oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle
from origami_amd.lossless import native_gpu
from tests import bitref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("max_dtype", [np.float16, np.float32])
@pytest.mark.parametrize("layers,tokens,heads,head_dim", [
    (1, 1, 1, 8), (17, 33, 2, 24), (2, 16, 8, 128), (1, 47, 3, 80), (3, 300, 1, 64),
    (16, 15, 5, 16)])
def test_dense_matches_oracle(cuda_device, layers, tokens, heads, head_dim, max_dtype):
    rng = np.random.default_rng(tokens)
    count = tokens * heads * head_dim
    bits = [1 + (3 * j) % 8 for j in range(2 * layers)]
    bins = rng.integers(4, 200, (2, layers)).tolist()
    segs = [bitref.bits_pack(rng.integers(0, 1 << b, count, dtype=np.uint8), b) for b in bits]
    segs[-1] = segs[-1][:-1]  # the last symbols read 0
    offs = np.concatenate([[3], 3 + np.cumsum([s.size for s in segs])]).astype(np.int64)
    stream = np.concatenate([np.zeros(3, np.uint8)] + segs)
    mk, mv = ((rng.random(layers * tokens) * 2 + 0.1).astype(max_dtype) for _ in range(2))
    want = oracle.cachegen_unpack_dequantize(stream, offs, bits, *bins, mk, mv, tokens, heads,
                                             head_dim)
    dev = cuda_device
    got = native_gpu.cachegen_unpack_dequantize(
        torch.from_numpy(stream).to(dev), offs, bits, *bins, torch.from_numpy(mk).to(dev),
        torch.from_numpy(mv).to(dev), tokens=tokens, heads=heads, head_dim=head_dim)
    assert np.array_equal(got.cpu().view(torch.int16).numpy().view(np.uint16),
                          want.view(np.uint16))
