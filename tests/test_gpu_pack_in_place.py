"""The 8-bit pack off 128-byte lines: runs written in place (short layers, tiles that
would leave the staged pack's rounds part empty, runs on dwords beyond two rounds) and
the staged tiles on the other side of each rule, at every remainder of a 16-token run and
with streams at any byte, against the planes transposed by torch.  Bytes around the
stream keep their value."""
import pytest
import torch

from origami_amd.layout import kv_symbol_layout
from origami_amd.lossless import native_gpu
from origami_amd.lossless.chunking import plan_head_channel_chunks

pytestmark = pytest.mark.gpu


def _layout(T, H, C):
    plan = plan_head_channel_chunks(layer_index=0, num_heads=H, head_dim=C, token_count=2 * T,
                                    bytes_per_symbol=1, min_bytes=1 << 16, target_bytes=1 << 16,
                                    max_bytes=1 << 16)
    return kv_symbol_layout(T, H, C, 8, [
        [c.layout.head_start, c.layout.head_end, c.layout.channel_start, c.layout.channel_end, 0,
         2 * T] for c in plan])


def _check(dev, T, H, D, shift, bs=16, blocks_first=False, seed=0):
    C, nblk = 2 * D, -(-T // bs)
    NB = nblk + 5
    g = torch.Generator(device=dev).manual_seed(seed + T)
    shape = (NB, 2, bs, H, C) if blocks_first else (2, NB, bs, H, C)
    cache = torch.randint(0, 256, shape, generator=g, device=dev, dtype=torch.uint8)
    ids = torch.randperm(NB, generator=g, device=dev)[:nblk].contiguous()
    layout = _layout(T, H, C)
    whole = torch.full((layout.stream_bytes + shift + 160,), 0x5A, dtype=torch.uint8, device=dev)
    out = whole[shift:shift + layout.stream_bytes]
    native_gpu.pack_from_kv_cache(cache.view(torch.bfloat16), ids, T, layout, out)
    blocks = cache[ids].transpose(0, 1) if blocks_first else cache[:, ids]
    tokens = blocks.reshape(2, nblk * bs, H * C)[:, :T].reshape(2 * T, H * C)
    assert torch.equal(out, tokens.t().contiguous().reshape(-1))
    assert bool((whole[:shift] == 0x5A).all())
    assert bool((whole[shift + layout.stream_bytes:] == 0x5A).all())


@pytest.mark.parametrize("rest", range(16))
@pytest.mark.parametrize("tokens,heads,head_dim,shift", [
    (0, 1, 8, 0), (0, 1, 64, 1), (16, 1, 128, 16), (112, 2, 64, 3), (256, 1, 128, 0),
    (768, 2, 128, 5), (2048, 4, 128, 0)])
def test_every_remainder(cuda_device, tokens, heads, head_dim, shift, rest):
    _check(cuda_device, tokens + rest or 48, heads, head_dim, shift, blocks_first=rest % 2 == 1)


@pytest.mark.parametrize("tokens,shift", [
    (4104, 0), (8201, 0), (11008, 0), (11500, 0), (12001, 7), (18000, 0), (18001, 2), (24016, 0),
    (32784, 0), (32784, 2), (32770, 0), (49216, 0), (49217, 0)])
def test_rules(cuda_device, tokens, shift):
    _check(cuda_device, tokens, 8, 128, shift)


def test_block_sizes(cuda_device):
    for bs in (8, 24, 32):
        _check(cuda_device, 1001, 2, 64, 0, bs=bs)
