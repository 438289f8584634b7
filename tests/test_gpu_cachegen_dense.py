"""The dense CacheGen restore at the edges of its tiles (16 or, in short launches, fewer
tokens x all heads), with head rows of a power of two of groups and not, every symbol
width, streams at any byte, a short segment, and more segments than one launch takes,
against the oracle; and more tiles than a launch has workgroups."""
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
    (16, 15, 5, 16), (1, 101, 8, 128), (2, 3100, 4, 64), (1, 12300, 1, 128)])
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


def test_more_tiles_than_one_launch_takes(cuda_device):
    """2^28 + 33 tokens of one 8-channel head at 1 bit: a launch holds fewer than 2^32
    threads.  Symbols follow a period of 3 tokens, maxima one of 5."""
    dev, T = cuda_device, (1 << 28) + 33
    if torch.cuda.get_device_properties(dev).total_memory < 40 << 30:
        pytest.skip("needs 40 GiB")
    pattern = torch.tensor([0x35, 0xFF, 0x00], dtype=torch.uint8, device=dev)
    stream = pattern.repeat(T // 3 + 1)[:T].repeat(2)
    peaks = torch.tensor([1, 2, 3, 4, 5], dtype=torch.float16, device=dev).repeat(T // 5 + 1)[:T]
    got = native_gpu.cachegen_unpack_dequantize(
        stream, [0, T, 2 * T], [1, 1], [4], [4], peaks, peaks, tokens=T, heads=1, head_dim=8)
    small = native_gpu.cachegen_unpack_dequantize(
        stream[:15].repeat(2), [0, 15, 30], [1, 1], [4], [4], peaks[:15].contiguous(),
        peaks[:15].contiguous(), tokens=15, heads=1, head_dim=8)
    for half in range(2):
        rows = got.reshape(2, T, 8)[half]
        period = small.reshape(2, 15, 8)[half]
        assert bool((rows[:T // 15 * 15].view(-1, 15, 8) == period).all())
        assert torch.equal(rows[T // 15 * 15:], period[:T % 15])
