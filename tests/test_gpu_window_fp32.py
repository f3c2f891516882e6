"""fp32 window attention at the edges of its tiles, against the same attention in 64 bits: 64- and 128-query workgroups (few
and many items), a last item of one query, windows shorter than a block, rings with missing rows, sinks past and before them.

Tolerance: every product carries its 24 bits and the sums are fp32, D + W of them in order, so the error stays within a
few 2^-24 per row: 2e-6 of the norm, and 1e-5 in the log-sum-exp.
"""
import math

import pytest
import torch

from test_gpu_window import make_case, run

pytestmark = pytest.mark.gpu


def reference(c):
    """(o, lse) in 64 bits from the definition: a loop over sequences and heads."""
    B, H, G, T, W, start = (c[k] for k in ("B", "H", "G", "T", "W", "start"))
    old = torch.arange(max(0, start - W), start)
    old = old[c["ring_pos"][old % W] == old]
    ns = c["sink_k"].shape[2]
    pos = torch.cat((torch.arange(ns), old, torch.arange(start, start + T)))
    sink = torch.arange(len(pos)) < ns
    p = torch.arange(start, start + T)[:, None]
    see = torch.where(sink, pos <= p, (pos >= c["S"]) & (pos <= p) & (p - pos < W))
    o, lse = torch.empty(B, T, H, c["D"], dtype=torch.float64), torch.empty(B, H, T, dtype=torch.float64)
    for b in range(B):
        for h in range(H):
            g = h // (H // G)
            k = torch.cat((c["sink_k"][b, g], c["ring_k"][b, g, old % W], c["kr"][b, g])).double()
            v = torch.cat((c["sink_v"][b, g], c["ring_v"][b, g, old % W], c["v"][b, :, g])).double()
            s = (c["qr"][b, h].double() @ k.t() / math.sqrt(c["D"])).masked_fill(~see, -math.inf)
            lse[b, h] = s.logsumexp(-1)
            o[b, :, h] = s.softmax(-1) @ v
    return o, lse


@pytest.mark.parametrize("B,H,G,D,T,W,S,start,miss", [
    (1, 2, 1, 256, 65, 40, 3, 0, 0.0),          # 64-query items, the second of one query
    (1, 4, 2, 256, 33, 64, 2, 777, 0.2),        # a wrapped ring with missing rows
    (1, 66, 22, 256, 257, 96, 4, 500, 0.1),     # 128-query items, the third of one query
    (3, 24, 4, 128, 300, 33, 1, 0, 0.0),
    (1, 96, 8, 64, 191, 200, 4, 150, 0.0),      # a ring that is not full
    (1, 8, 8, 64, 1, 16, 0, 40, 0.0),           # one query, no sinks
    (1, 4, 2, 64, 33, 400, 3, 900, 0.1),        # D = 64: unsplit rows from 33 queries on, or up to 128 keys
    (1, 4, 2, 64, 32, 400, 3, 900, 0.1),
    (2, 4, 1, 64, 20, 128, 3, 900, 0.0),
    (2, 4, 1, 64, 20, 129, 3, 900, 0.0),
    (3, 4, 2, 64, 130, 70, 2, 0, 0.0),
    (40, 8, 2, 128, 64, 300, 2, 500, 0.1),      # many items of half a 128-query workgroup, and of one query more
    (20, 8, 2, 128, 65, 300, 2, 500, 0.0),
    (9, 16, 4, 128, 140, 256, 3, 700, 0.0),     # the last window of 64-query items, the first of 128, at either dim
    (9, 16, 4, 128, 140, 257, 3, 700, 0.0),
    (9, 16, 4, 64, 140, 1024, 3, 2000, 0.1),
    (9, 16, 4, 64, 140, 1025, 3, 2000, 0.0),
])
def test_window_fp32_tiles(dev, B, H, G, D, T, W, S, start, miss):
    c = make_case(B, H, G, D, T, W, S, start, seed=T + W, invalid_frac=miss, dtype=torch.float32)
    print(f"window fp32 B={B} H={H} G={G} D={D} T={T} W={W} S={S} start={start}", flush=True)
    o, lse = run(c, dev)[:2]
    ref, ref_lse = reference(c)
    err = ((o.cpu().double() - ref).norm() / ref.norm()).item()
    assert err < 2e-6, err
    assert (lse.cpu().double() - ref_lse).abs().max().item() < 1e-5


def classes(x):
    """0 finite, 1 +inf, 2 -inf, 3 nan."""
    return torch.where(x.isnan(), 3, torch.where(x == math.inf, 1, torch.where(x == -math.inf, 2, 0)))


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("T", [40, 200])
def test_window_fp32_infinities(dev, D, T):
    """Infinite elements give what they give in 64 bits: in a value row that every query sees, that column; in a key, a score
    of -inf, which leaves the key out. The finite elements stay within the tolerance above."""
    c = make_case(1, 4, 2, D, T, 64, 4, 300, seed=T, dtype=torch.float32)
    print(f"window fp32 infinities D={D} T={T}", flush=True)
    c["sink_v"][0, 0, 1, 3] = math.inf
    c["sink_v"][0, 1, 2, D - 1] = -math.inf
    c["qr"][..., 2] = -1.0
    c["kr"][0, 0, 20, 2] = math.inf
    c["ring_k"][0, 1, :, 2] = 0.0
    c["ring_k"][0, 1, 290 % 64, 2] = math.inf
    o, lse = run(c, dev)[:2]
    ref, ref_lse = reference(c)
    assert torch.equal(classes(o.cpu()), classes(ref))
    fin = ref.isfinite()
    assert ((o.cpu().double() - ref)[fin].norm() / ref[fin].norm()).item() < 2e-6
    assert (lse.cpu().double() - ref_lse).abs().max().item() < 1e-5
