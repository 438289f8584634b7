"""The staged 8-bit pack (16-wave tiles, with and without single ownership of the stream's
lines) for the forms it takes: plans in another order (plane tables), channel counts that
leave lanes of a tile without a channel, block sizes off 16, symbol tensors (one half),
token counts on every alignment and outputs at any byte.  Each case states which tiles the
library's rule gives it on the device's CUs, and fails if a changed rule would send it
elsewhere.  Streams are compared with the planes transposed by torch; bytes around the
stream keep their value."""
import pytest
import torch

from origami_amd.layout import CanonicalLayout, kv_symbol_layout
from origami_amd.lossless import native_gpu
from origami_amd.lossless.chunking import plan_head_channel_chunks

pytestmark = pytest.mark.gpu

STAGED, OWNED = "staged", "single owner"


def tiles_of(T, H, C, halves, dwords, cus):
    """The pack that set_pack_grid picks for 8-bit planes off 128-byte lines."""
    cols = halves * -(-H * C // 128)
    tiles = cols * -(-T // 2048)
    rounds = -(-tiles // cus)
    if tiles < max(1, cus // 2) or cols * T / 2048 / (rounds * cus) <= 0.69 or (
            dwords and rounds > 2):
        return "in place"
    return OWNED if halves == 2 and cols * -(-T // 1920) <= rounds * cus else STAGED


def _specs(tokens, H, C, reverse, chunk=1 << 17):
    plan = plan_head_channel_chunks(layer_index=0, num_heads=H, head_dim=C, token_count=tokens,
                                    bytes_per_symbol=1, min_bytes=chunk, target_bytes=chunk,
                                    max_bytes=chunk)
    specs = [[c.layout.head_start, c.layout.head_end, c.layout.channel_start,
              c.layout.channel_end, 0, tokens] for c in plan]
    return specs[::-1] if reverse else specs


def _stream(rows, specs, H, C):
    """The 8-bit stream of [tokens, H * C] symbols under `specs`."""
    planes = rows.t().reshape(H, C, -1)
    return torch.cat([planes[s[0]:s[1], s[2]:s[3]].reshape(-1) for s in specs])


def _compare(pack, size, want, shift, dev):
    whole = torch.full((size + shift + 160,), 0x5A, dtype=torch.uint8, device=dev)
    out = whole[shift:shift + size]
    pack(out)
    assert torch.equal(out, want)
    assert bool((whole[:shift] == 0x5A).all()) and bool((whole[shift + size:] == 0x5A).all())


@pytest.mark.parametrize("T,H,C,bs,reverse,shift,want", [
    (16383, 8, 256, 16, True, 0, STAGED), (24001, 8, 256, 16, True, 3, OWNED),
    (16383, 5, 400, 16, False, 0, STAGED), (24001, 5, 400, 16, False, 0, OWNED),
    (16383, 5, 400, 16, True, 5, STAGED), (24001, 5, 400, 24, True, 64, OWNED),
    (16002, 8, 256, 8, False, 0, STAGED), (16002, 8, 256, 24, False, 2, STAGED),
    (24002, 8, 256, 8, False, 0, OWNED), (49218, 8, 256, 24, False, 1, OWNED),
    (16004, 8, 256, 16, False, 0, STAGED), (16016, 8, 256, 16, False, 0, STAGED),
    (16000, 8, 256, 16, False, 16, STAGED), (32753, 8, 256, 32, False, 1, STAGED)])
@pytest.mark.parametrize("blocks_first", [False, True])
def test_paged_cache(cuda_device, T, H, C, bs, reverse, shift, want, blocks_first):
    cus = torch.cuda.get_device_properties(cuda_device).multi_processor_count
    assert tiles_of(T, H, C, 2, T % 4 == 0 and shift % 4 == 0, cus) == want
    nblk = -(-T // bs)
    NB = nblk + 3
    g = torch.Generator(device=cuda_device).manual_seed(T + bs)
    shape = (NB, 2, bs, H, C) if blocks_first else (2, NB, bs, H, C)
    cache = torch.randint(0, 256, shape, generator=g, device=cuda_device, dtype=torch.uint8)
    ids = torch.randperm(NB, generator=g, device=cuda_device)[:nblk].contiguous()
    blocks = cache[ids].transpose(0, 1) if blocks_first else cache[:, ids]
    rows = blocks.reshape(2, nblk * bs, H * C)[:, :T].reshape(2 * T, H * C)
    specs = _specs(2 * T, H, C, reverse)
    layout = kv_symbol_layout(T, H, C, 8, specs)
    _compare(lambda out: native_gpu.pack_from_kv_cache(cache.view(torch.bfloat16), ids, T, layout,
                                                       out),
             layout.stream_bytes, _stream(rows, specs, H, C), shift, cuda_device)


@pytest.mark.parametrize("T,H,C,reverse,shift", [
    (32753, 8, 256, False, 0), (32753, 8, 256, True, 1), (32001, 5, 400, False, 7),
    (32750, 16, 128, False, 0)])
def test_symbol_tensor(cuda_device, T, H, C, reverse, shift):
    cus = torch.cuda.get_device_properties(cuda_device).multi_processor_count
    assert tiles_of(T, H, C, 1, False, cus) == STAGED
    g = torch.Generator(device=cuda_device).manual_seed(T)
    rows = torch.randint(0, 256, (T, H * C), generator=g, device=cuda_device, dtype=torch.uint8)
    specs = _specs(T, H, C, reverse)
    layout = CanonicalLayout.make([T, H, C], ["token", "head", "head_dim"], 8, specs)
    _compare(lambda out: native_gpu.pack_layout(rows, layout, out), layout.stream_bytes,
             _stream(rows, specs, H, C), shift, cuda_device)
