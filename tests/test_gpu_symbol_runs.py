"""Chunk plans whose chunks are memory runs of the symbol tensor: plain bit
streams ([1, 1, n]), token-fastest tensors, and plans that merge into one run,
stay several runs, leave gaps or mix both kinds.  Unpacks and packs at the
edges of a lane's group (16 or 32 symbols), of an unrolled launch, and with
streams and outputs off their alignment, byte for byte against the oracle;
bytes around an output inside a larger buffer keep their value."""
import os

import numpy as np
import pytest
import torch

from oracle import oracle
from origami_amd.layout import CanonicalLayout
from origami_amd.lossless import native_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _oracle_threads():
    oracle.set_threads(min(16, os.cpu_count() or 1))


def _check(dev, shape, names, specs, bits, stream_shift=0, symbol_shift=0):
    layout = CanonicalLayout.make(shape, names, bits, specs)
    rng = np.random.default_rng(bits * 1000 + layout.symbol_count % 997)
    symbols = rng.integers(0, 256, layout.symbol_count, dtype=np.uint8)  # bits past b ignored
    axes = [int(a) for a in layout.axes]
    stream, offsets = oracle.pack_canonical(symbols, bits, specs, shape, axes)
    want = oracle.unpack_canonical(stream, offsets, bits, specs, shape, axes)

    def buffer(n, shift):
        whole = torch.full((n + shift + 64,), 0xA5, dtype=torch.uint8, device=dev)
        return whole, whole[shift:shift + n]

    whole, out = buffer(stream.size, stream_shift)
    src = buffer(symbols.size, symbol_shift)[1]
    src.copy_(torch.from_numpy(symbols))
    native_gpu.pack_layout(src, layout, out)
    got = whole.cpu().numpy()
    assert np.array_equal(got[stream_shift:stream_shift + stream.size], stream)
    assert (got[:stream_shift] == 0xA5).all() and (got[stream_shift + stream.size:] == 0xA5).all()

    whole, flat = buffer(stream.size, stream_shift)
    flat.copy_(torch.from_numpy(stream))
    whole_out, out = buffer(symbols.size, symbol_shift)
    native_gpu.unpack_layout(flat, layout, out)
    got = whole_out.cpu().numpy()
    assert np.array_equal(got[symbol_shift:symbol_shift + symbols.size], want)
    assert (got[:symbol_shift] == 0xA5).all()
    assert (got[symbol_shift + symbols.size:] == 0xA5).all()


TOKEN = ["token", "head", "head_dim"]


@pytest.mark.parametrize("bits", range(1, 9))
@pytest.mark.parametrize("n,stream_shift,symbol_shift", [
    (1, 0, 0), (15, 1, 2), (16, 0, 0), (17, 0, 13), (33, 3, 5), (8191, 2, 4), (8192, 4, 16),
    (8224, 0, 4), ((1 << 23) + 21, 0, 0)])  # the last: several groups per lane
def test_plain_streams(cuda_device, bits, n, stream_shift, symbol_shift):
    _check(cuda_device, [1, 1, n], TOKEN, [[0, 1, 0, n, 0, 1]], bits, stream_shift, symbol_shift)


@pytest.mark.parametrize("bits", [3, 4, 8])
@pytest.mark.parametrize("case", ["merged", "off_bytes", "gap", "reordered", "many_runs",
                                  "token_fastest", "token_fastest_part", "heads_split"])
def test_plans_of_runs(cuda_device, bits, case):
    shape, names = [1, 1, 4000], TOKEN
    cuts = {"merged": range(0, 4001, 1000), "off_bytes": [0, 1001, 2003, 4000],
            "reordered": [0, 1024, 2048, 4000], "gap": [0, 1024, 2048, 4000],
            "many_runs": range(0, 4001, 125)}.get(case)
    if cuts is not None:
        cuts = list(cuts)
        specs = [[0, 1, a, b, 0, 1] for a, b in zip(cuts, cuts[1:])]
        if case == "gap":
            specs = [specs[0], specs[2]]
        if case == "reordered":
            specs = specs[::-1]
    elif case == "token_fastest":
        shape, names = [1, 3, 20, 77], ["layer", "head", "head_dim", "token"]
        specs = [[0, 1, 0, 20, 0, 77], [1, 3, 0, 20, 0, 77]]
    elif case == "token_fastest_part":  # token ranges: runs of one plane each at most
        shape, names = [1, 2, 77], ["head", "head_dim", "token"]
        specs = [[0, 1, 0, 1, 0, 40], [0, 1, 0, 1, 40, 77], [0, 1, 1, 2, 0, 77]]
    else:  # T = 1 and a channel range of each head: a run per head, not one run
        shape, names = [1, 4, 48], TOKEN
        specs = [[0, 4, 0, 16, 0, 1], [0, 2, 16, 48, 0, 1], [2, 3, 16, 48, 0, 1],
                 [3, 4, 16, 48, 0, 1]]
    _check(cuda_device, shape, names, specs, bits)
    _check(cuda_device, shape, names, specs, bits, 4, 8)
