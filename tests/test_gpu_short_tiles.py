"""Restores and packs of short layers, where the tile is 1, 2 or 4 waves and may hold only
part of its token runs: every width at token counts on both sides of the rules' lines,
dense and reordered plans, against planes packed by torch."""
import pytest
import torch

from origami_amd.layout import kv_symbol_layout
from origami_amd.lossless import native_gpu
from origami_amd.lossless.chunking import plan_head_channel_chunks

pytestmark = pytest.mark.gpu


def _pack_rows(planes, bits):
    """[planes, tokens] symbols -> one LSB-first stream."""
    flat = planes.reshape(-1)
    pad = -flat.numel() % 8
    s = torch.cat([flat, flat.new_zeros(pad)]).reshape(-1, 8).to(torch.int64)
    word = (s << (bits * torch.arange(8, device=s.device))).sum(1)
    out = (word[:, None] >> (8 * torch.arange(bits, device=s.device))) & 255
    return out.to(torch.uint8).reshape(-1)[:(flat.numel() * bits + 7) // 8]


@pytest.mark.parametrize("bits", range(1, 9))
@pytest.mark.parametrize("tokens,heads,reverse", [
    (16, 1, False), (33, 2, False), (64, 8, False), (192, 1, True), (256, 4, False),
    (512, 1, False), (640, 2, False), (1536, 4, False), (2053, 2, True), (3000, 4, False),
    (4104, 8, False)])
def test_short_layers(cuda_device, tokens, heads, bits, reverse):
    T, H, C, bs = tokens, heads, 128, 16
    plan = plan_head_channel_chunks(layer_index=0, num_heads=H, head_dim=C, token_count=2 * T,
                                    bytes_per_symbol=1, min_bytes=1 << 14,
                                    target_bytes=1 << 14, max_bytes=1 << 14)
    specs = [[c.layout.head_start, c.layout.head_end, c.layout.channel_start,
              c.layout.channel_end, 0, 2 * T] for c in plan]
    specs = specs[::-1] if reverse else specs
    layout = kv_symbol_layout(T, H, C, bits, specs)
    nblk = -(-T // bs)
    NB = nblk + 3
    g = torch.Generator(device=cuda_device).manual_seed(T + bits)
    cache = torch.randint(0, 1 << bits, (2, NB, bs, H, C), generator=g, device=cuda_device,
                          dtype=torch.uint8)
    ids = torch.randperm(NB, generator=g, device=cuda_device)[:nblk].contiguous()
    rows = cache[:, ids].reshape(2, nblk * bs, H, C)[:, :T].reshape(2 * T, H, C)
    planes = rows.permute(1, 2, 0)
    want = torch.cat([_pack_rows(planes[s[0]:s[1], s[2]:s[3]].contiguous(), bits)
                      for s in specs])
    got = native_gpu.pack_from_kv_cache(cache.view(torch.bfloat16), ids, T, layout)
    assert torch.equal(got, want)

    restored = torch.full_like(cache, 0xC3)
    native_gpu.unpack_to_kv_cache(want, layout, T, restored.view(torch.bfloat16), ids)
    back = restored[:, ids].reshape(2, nblk * bs, H, C)
    assert torch.equal(back[:, :T].reshape(2 * T, H, C), rows)
    assert bool((back[:, T:] == 0).all())
    free = torch.ones(NB, dtype=torch.bool, device=cuda_device)
    free[ids] = False
    assert bool((restored[:, free] == 0xC3).all())
