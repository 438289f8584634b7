"""The fused quantizers against the adapters' tensor operations on the same GPU
tensors, byte for byte: every K/V layout and dtype, rows shorter and longer than a
wave, symbol runs and planes that do and do not start on words, group sizes the
kernel does and does not take, ragged token counts, and rows of zeros of one sign,
infinities and NaN of either sign and any payload.  The zero point of a KIVI group
whose least values are zeros of both signs is compared as a value."""
import pytest
import torch

from origami_amd.quantization import create_quantizer_adapter
from origami_amd.lossless import native_gpu

pytestmark = pytest.mark.gpu

DTYPES = [torch.bfloat16, torch.float16, torch.float32]


def _kv(dev, shape, dtype, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed)
    return (torch.randn(shape, generator=g, device=dev) * 2).to(dtype)


def _served(monkeypatch, name):
    """Counts the calls that the fused kernel served."""
    served, real = [], getattr(native_gpu, name)
    monkeypatch.setattr(native_gpu, name,
                        lambda *a, **k: served.append(real(*a, **k)) or served[-1])
    return served


def _check_cachegen(kv, config, layer, monkeypatch, fused=True):
    served = _served(monkeypatch, "cachegen_quantize")
    a = create_quantizer_adapter("cachegen", config)
    q = a.quantize(kv, layer_group=f"model.layers.{layer}.attn")
    m = q.metadata
    want = a._payload(kv, m["key_bins"], m["value_bins"], m["key_bits"], m["value_bits"])
    assert torch.equal(q.symbols, want)
    assert served == [fused]


def _check_kivi(kv, config, monkeypatch, fused=True):
    served = _served(monkeypatch, "kivi_quantize")
    a = create_quantizer_adapter("kivi", config)
    q = a.quantize(kv)
    assert torch.equal(q.symbols, a._payload(kv, q.metadata["sink_tokens"]))
    assert served == ([fused] if q.metadata["body_tokens"] else [])


SHAPES = [(2, 9, 16, 2, 64), (9, 2, 16, 2, 64), (9, 16, 2, 2, 64), (2, 150, 2, 64),
          (150, 2, 2, 64), (2, 2, 150, 64)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", SHAPES)
def test_layouts(cuda_device, shape, dtype, monkeypatch):
    kv = _kv(cuda_device, shape, dtype)
    _check_cachegen(kv, {}, 4, monkeypatch)
    _check_kivi(kv, {"sink_tokens": 16}, monkeypatch)


@pytest.mark.parametrize("tokens,heads,head_dim", [
    (1, 1, 8), (3, 1, 8), (257, 1, 24), (65, 3, 64), (33, 1, 128), (301, 8, 64), (70, 8, 128),
    (35, 10, 128), (21, 16, 256), (9, 33, 128), (4096, 8, 128), (2050, 1, 128), (5, 2, 20)])
@pytest.mark.parametrize("level,layer", [("2", 4), ("1", 25), ("3", 0)])
def test_cachegen_rows(cuda_device, tokens, heads, head_dim, level, layer, monkeypatch):
    kv = _kv(cuda_device, (2, 1, tokens, heads, head_dim), torch.bfloat16, tokens)
    fused = head_dim % 8 == 0 and heads * head_dim <= 4096
    _check_cachegen(kv, {"quant_level": level}, layer, monkeypatch, fused)
    _check_cachegen(kv, {"quant_level": level, "bitpacked": False}, layer, monkeypatch, fused)


@pytest.mark.parametrize("bits", [2, 3, 4, 8])
@pytest.mark.parametrize("tokens,heads,head_dim,group,sink", [
    (192, 2, 64, 64, 128), (1, 1, 8, 16, 0), (17, 1, 8, 16, 0), (16, 1, 72, 32, 0),
    (300, 3, 40, 32, 37), (2048, 8, 128, 64, 128), (515, 2, 128, 128, 3), (1040, 1, 128, 128, 16),
    (640, 4, 64, 16, 0), (64, 1, 64, 64, 64), (200, 1, 64, 48, 8), (100, 1, 20, 32, 4)])
def test_kivi_shapes(cuda_device, bits, tokens, heads, head_dim, group, sink, monkeypatch):
    kv = _kv(cuda_device, (2, 1, tokens, heads, head_dim), torch.bfloat16, tokens)
    fused = head_dim % 8 == 0 and group in (16, 32, 64, 128)
    if fused and (tokens - sink) % 16:  # streams off dwords are packed by tensor operations
        fused = heads * head_dim * (tokens - sink) * (4 if bits == 3 else bits) % 32 == 0
    _check_kivi(kv, {"bits": bits, "group_size": group, "sink_tokens": sink}, monkeypatch, fused)


@pytest.mark.parametrize("dtype", DTYPES)
def test_unusual_values(cuda_device, dtype, monkeypatch):
    kv = _kv(cuda_device, (2, 10, 16, 2, 64), dtype)
    flat = kv.view(2, 160, 128)
    flat[:, 3] = 0
    flat[:, 20, 5] = float("inf")
    flat[:, 40, 6] = -float("inf")
    flat[:, 60, 7] = float("nan")
    flat[:, 61] = float("nan")
    flat[:, 62:64] = float("inf")
    flat[:, 64:128, 9] = 1.25  # one value in a whole key group
    flat[:, 80] = torch.finfo(torch.float16).tiny / 2
    flat[:, 81] = 1e-7
    flat[:, 82, 3] = 6e4
    flat[:, 96:112] *= 1e-6  # float16 subnormals
    _check_cachegen(kv, {}, 4, monkeypatch)
    for bits in (2, 8):
        _check_kivi(kv, {"bits": bits, "group_size": 64, "sink_tokens": 0}, monkeypatch)


def _nan(dtype, sign, payload, dev):
    """One quiet NaN of the given sign and payload bits (of those float16 keeps)."""
    bits, width = {torch.bfloat16: (0x7fc0, 16), torch.float16: (0x7e00, 16),
                   torch.float32: (0x7fc00000, 32)}[dtype]
    place = {torch.bfloat16: 3, torch.float16: 6, torch.float32: 19}[dtype]
    v = bits | (payload << place) | (sign << (width - 1))
    v -= (1 << width) if sign else 0
    return torch.tensor([v], dtype=torch.int64).to(
        torch.int16 if width == 16 else torch.int32).view(dtype).to(dev)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("where", ["value", "row", "keys"])
@pytest.mark.parametrize("sign,payload", [(0, 0), (1, 0), (0, 1), (1, 5)])
def test_nan_bytes(cuda_device, dtype, where, sign, payload, monkeypatch):
    kv = _kv(cuda_device, (2, 10, 16, 2, 64), dtype)
    flat = kv.view(2, 160, 128)
    nan = _nan(dtype, sign, payload, cuda_device)
    at = {"value": (slice(None), 60, 7), "row": (slice(None), 61),
          "keys": (slice(None), slice(64, 128), 9)}[where]
    flat[at] = nan
    _check_cachegen(kv, {}, 4, monkeypatch)
    for bits in (2, 8):
        _check_kivi(kv, {"bits": bits, "group_size": 64, "sink_tokens": 0}, monkeypatch)


@pytest.mark.parametrize("dtype", DTYPES)
def test_least_zeros(cuda_device, dtype, monkeypatch):
    kv = _kv(cuda_device, (2, 10, 16, 2, 64), dtype)
    flat = kv.view(2, 160, 128)
    flat[:, :64] = flat[:, :64].abs() + 0.5
    flat[:, 5, :64] = -0.0  # zeros of one sign in a group
    flat[:, 6, 64:] = 0.0
    config = {"bits": 2, "group_size": 64, "sink_tokens": 0}
    _check_cachegen(kv, {}, 4, monkeypatch)
    _check_kivi(kv, config, monkeypatch)
    flat[:, 64:128] = 0.0  # of both signs
    flat[:, 64:128:2, ::3] = -0.0
    _check_cachegen(kv, {}, 4, monkeypatch)
    a = create_quantizer_adapter("kivi", config)
    q = a.quantize(kv)
    m, want = q.metadata, a._payload(kv, 0)
    same = q.symbols == want
    for name in ("key_zero", "value_zero"):
        part = slice(m[f"{name}_offset"], m[f"{name}_offset"] + 2 * m[f"{name}_numel"])
        got, ref = (x[part].view(torch.float16) for x in (q.symbols, want))
        assert torch.equal(got, ref)  # -0 == 0
        same[part] = True
    assert bool(same.all())
