"""A chunk of a kept layer whose queries' keys are taken in parts (``bf_prefix_attention``), against the oracle.

The part counts follow the launch's slots per XCD and the key blocks of an item; the cases cover a few slots in many parts,
one query row past a 128-query item, the shortest history that is split, and a last round more than half full. Tolerance: q, k, v
and the probabilities are bf16 (2^-9 each) with fp32 sums, as in the unsplit kernel.
"""
import ctypes

import pytest
import torch

from oracle import teacher as ot

TOL16 = 8e-3


def _parts(B, G, R, D, T, cap, start):
    from heimdall_amd import _lib
    n = ctypes.c_size_t(0)
    assert _lib.load().bf_prefix_attention_workspace_size(B, G, R, D, T, cap, start, 1, ctypes.byref(n)) == 0
    return n.value


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,G,D,n,t", [
    (1, 4, 2, 256, 4200, 17),          # one item row, the most parts
    (2, 8, 2, 128, 3000, 129),         # a second item of one query
    (1, 24, 4, 64, 1600, 100),         # few key blocks: fewer parts
    (1, 8, 1, 64, 9000, 2100),         # 17 query blocks of 8 heads: 24 slots per XCD, some past an XCD's items
])
def test_prefix_parts(dev, B, H, G, D, n, t):
    from heimdall_amd.teacher import teacher
    assert _parts(B, G, H // G, D, t, n + 256, n - t) > 0
    gen = torch.Generator().manual_seed(n)
    qr, kr, v = (torch.randn(B, h, n, D, generator=gen).to(torch.bfloat16) for h in (H, G, G))
    cache = {"k": kr[:, :, :n - t].to(dev), "v": v[:, :, :n - t].to(dev)}
    m = type("M", (), {"retrieval": None})()
    o = teacher(m, qr[:, :, n - t:].to(dev), kr[:, :, n - t:].to(dev), v[:, :, n - t:].transpose(1, 2).to(dev), cache)
    ocache = {"k": kr[:, :, :n - t].float(), "v": v[:, :, :n - t].float()}
    ref = ot.teacher(qr[:, :, n - t:].float(), kr[:, :, n - t:].float(), v[:, :, n - t:].transpose(1, 2).float(), ocache, None)
    err = ((o.double().cpu() - ref.double()).norm() / ref.double().norm()).item()
    assert err < TOL16, err


def test_prefix_workspace_arguments():
    from heimdall_amd import _lib
    n, lib = ctypes.c_size_t(0), _lib.load()
    size = lib.bf_prefix_attention_workspace_size
    assert size(1, 4, 6, 256, 2048, 24576, 14336, 0, ctypes.byref(n)) == 0 and n.value == 0       # fp32: never in parts
    assert size(1, 4, 6, 256, 2048, 24576, 64, 1, ctypes.byref(n)) == 0                           # a short history
    assert size(1, 4, 6, 96, 2048, 24576, 64, 1, ctypes.byref(n)) == -2
    assert size(1, 4, 6, 256, 2048, 2048, 1, 1, ctypes.byref(n)) == -1                            # start + T > cap
    assert lib.bf_prefix_attention(1, 4, 6, 256, 2048, 24576, 14336, 1, 256, 0, 0, 0, 256, 256, 256, 256, 1, None, 0, None) == -3
    # partial rows are written with 16-byte stores
    assert size(1, 4, 6, 256, 2048, 24576, 14336, 1, ctypes.byref(n)) == 0 and n.value > 0
    assert lib.bf_prefix_attention(1, 4, 6, 256, 2048, 24576, 14336, 1, 256, 0, 0, 0, 256, 256, 256, 256, 1, 264, n.value, None) == -3


def test_short_histories_stay_whole():
    """After an odd number of full rounds, a last round of 12 or 16 slots is split only where the items' shortest keys pay for
    the parts' rows; a launch of one round, one after an even number, a last round of few slots, and D = 64 are split as before."""
    for H, G, D, T, start, parts in ((24, 4, 256, 2048, 1, False), (24, 4, 256, 2048, 300, False), (24, 4, 256, 2048, 1000, True),
                                     (24, 4, 256, 4600, 1, False), (24, 4, 256, 4600, 1150, True), (16, 4, 256, 3000, 1, False),
                                     (16, 4, 256, 7000, 1, False), (16, 4, 256, 2816, 1, False), (16, 4, 256, 2816, 704, True),
                                     (32, 8, 128, 1500, 300, False), (32, 8, 128, 1500, 1000, True), (32, 8, 128, 1400, 350, True),
                                     (32, 8, 128, 2330, 1, True), (16, 4, 256, 5000, 1, True), (8, 2, 256, 6000, 1, True),
                                     (8, 2, 256, 2048, 1, True), (16, 4, 256, 2304, 1, True), (24, 4, 256, 2800, 1, True),
                                     (8, 2, 64, 6000, 1, True)):
        assert (_parts(1, G, H // G, D, T, start + T + 256, start) > 0) == parts, (H, G, D, T, start)
