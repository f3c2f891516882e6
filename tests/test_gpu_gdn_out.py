"""fp32 outputs (the pass over all chunks after the scan), against the recurrence in 64 bits.

Chunk tails of 1 and 63 tokens, one chunk, several segments, packed sequences (one of them empty), every head dim, head counts
that are not a power of two, an initial state, and bf16 outputs. Tolerance: operands carry their 24 bits and sums are fp32 over
at most 2 D + 64 terms per chunk and a state carried in fp32, as in the scan: 2e-6 (bf16 outputs: their rounding, 2^-9, and a
margin of two).
"""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def recurrence(q, k, v, g, beta, s):
    """One sequence in 64 bits: q [T, G, R, D], k, v [T, G, D], g, beta [T, G], s [G, D, D]."""
    o = torch.empty(q.shape, dtype=torch.float64)
    for t in range(q.shape[0]):
        s = s * g[t].exp()[:, None, None]
        new = (v[t] - (k[t][:, None] @ s)[:, 0]) * beta[t][:, None]
        s = s + k[t][:, :, None] * new[:, None]
        o[t] = q[t] @ s
    return o, s


@pytest.mark.parametrize("lens,G,R,D,s0,out_dtype", [
    ([1], 1, 2, 64, False, torch.float32),
    ([64], 2, 3, 128, True, torch.float32),
    ([129], 2, 6, 256, False, torch.float32),
    ([63, 0, 200, 65], 3, 2, 64, True, torch.float32),
    ([300, 31], 1, 5, 256, True, torch.float32),
    ([100], 5, 4, 128, False, torch.bfloat16),
    ([130, 7], 2, 1, 256, True, torch.float32),
    ([77], 3, 1, 128, False, torch.float32),
])
def test_fp32_outputs(dev, lens, G, R, D, s0, out_dtype):
    from heimdall_amd._device import gdn_forward
    gen = torch.Generator().manual_seed(sum(lens) + D)
    N, B = sum(lens), len(lens)
    print(f"fp32 outputs lens={lens} G={G} R={R} D={D}", flush=True)
    q, k = torch.randn(N, G, R, D, generator=gen), F.normalize(torch.randn(N, G, D, generator=gen), dim=-1)
    v, g = torch.randn(N, G, D, generator=gen), -0.05 * torch.rand(N, G, generator=gen)
    beta, s = torch.sigmoid(torch.randn(N, G, generator=gen)), torch.randn(B, G, D, D, generator=gen) if s0 else None
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    to = lambda x: x.to(dev)
    for seg in (0, 1):                                    # 1: a segment per chunk, through the summary and combine passes
        o, sf = gdn_forward(to(q.reshape(N, G * R, D)), to(k), to(v), to(g), to(beta), num_seqs=B, cu_seqlens=to(cu),
                            initial_state=None if s is None else to(s), out_dtype=out_dtype, segment_chunks=seg)
        tol = 2e-6 if out_dtype == torch.float32 else 2 ** -8
        for i in range(B):
            a, e = int(cu[i]), int(cu[i + 1])
            zero = torch.zeros(G, D, D, dtype=torch.float64)
            ro, rs = recurrence(*(x[a:e].double() for x in (q, k, v, g, beta)), zero if s is None else s[i].double())
            if e > a:
                err = (o[a:e].cpu().double().reshape(ro.shape) - ro).norm() / ro.norm()
                assert err < tol, (seg, i, err)
            if rs.norm() > 0:
                assert (sf[i].cpu().double() - rs).norm() / rs.norm() < 2e-6, (seg, i)


@pytest.mark.parametrize("lens,G,R,D", [([1], 1, 2, 64), ([129, 0, 63], 2, 3, 128), ([300, 31], 1, 2, 256), ([200], 2, 1, 128)])
def test_fp32_outputs_in_the_scan(dev, lens, G, R, D):
    """A workspace without room for the planes keeps the outputs in the scan (fp32 MFMAs): the same values, same tolerance."""
    from heimdall_amd import _lib
    gen = torch.Generator().manual_seed(sum(lens) + D)
    N, B, H = sum(lens), len(lens), G * R
    print(f"fp32 outputs in the scan lens={lens} G={G} R={R} D={D}", flush=True)
    q, k = torch.randn(N, G, R, D, generator=gen), F.normalize(torch.randn(N, G, D, generator=gen), dim=-1)
    v, g = torch.randn(N, G, D, generator=gen), -0.05 * torch.rand(N, G, generator=gen)
    beta, s = torch.sigmoid(torch.randn(N, G, generator=gen)), torch.randn(B, G, D, D, generator=gen)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    lib, n = _lib.load(), _lib.ctypes.c_size_t(0)
    dq, dk, dv, dg, db, ds, dcu = (x.to(dev).contiguous() for x in (q, k, v, g, beta, s, cu))
    for seg in (0, 1):
        _lib.check(lib.bf_gdn_workspace_size(N, B, G, R, D, 0, seg, _lib.ctypes.byref(n)), "size")
        ws = torch.empty(n.value, dtype=torch.uint8, device=dev)
        outs = []
        for short in (0, 1):
            o, sf = torch.empty(N, H, D, device=dev), torch.empty(B, G, D, D, device=dev)
            _lib.check(lib.bf_gdn_fwd(dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), dg.data_ptr(), db.data_ptr(), dcu.data_ptr(),
                                      B, N, G, R, D, 0, 1.0, ds.data_ptr(), o.data_ptr(), 0, sf.data_ptr(), seg, ws.data_ptr(),
                                      n.value - short, 15, torch.cuda.current_stream().cuda_stream), "bf_gdn_fwd")
            outs.append(o)
            for i in range(B):
                a, e = int(cu[i]), int(cu[i + 1])
                ro, rs = recurrence(*(x[a:e].double() for x in (q, k, v, g, beta)), s[i].double())
                if e > a:
                    err = (o[a:e].cpu().double().reshape(ro.shape) - ro).norm() / ro.norm()
                    assert err < 2e-6, (seg, short, i, err)
                assert (sf[i].cpu().double() - rs).norm() / rs.norm() < 2e-6, (seg, short, i)
        assert N < 64 or not torch.equal(*outs)           # two routes


def test_planes_without_memory(dev, monkeypatch):
    """Where memory does not reach for the planes, the calls take the smallest workspace and its route; bf16 runs have no
    smaller one and raise."""
    from heimdall_amd import _device
    gen = torch.Generator().manual_seed(3)
    N, G, R, D = 150, 2, 2, 64
    q, k = torch.randn(N, G * R, D, generator=gen), F.normalize(torch.randn(N, G, D, generator=gen), dim=-1)
    v, g, beta = torch.randn(N, G, D, generator=gen), -0.05 * torch.rand(N, G, generator=gen), torch.rand(N, G, generator=gen)
    args = [x.to(dev) for x in (q, k, v, g, beta)]
    ref = _device.gdn_forward(*args, num_seqs=1)
    plain, asked = _device.workspace, []

    def full(nbytes, dev_):
        asked.append(nbytes)
        if len(asked) == 1:
            raise torch.OutOfMemoryError("no memory")
        return plain(nbytes, dev_)

    monkeypatch.setattr(_device, "workspace", full)
    got = _device.gdn_forward(*args, num_seqs=1)
    assert len(asked) == 2 and asked[0] - asked[1] == 2 * (N // 64 + 1) * G * (D // 16) * (D // 32 + 2) * 1536
    for x, y in zip(got, ref):
        assert ((x - y).norm() / y.norm()).item() < 4e-6
    asked.clear()
    with pytest.raises(torch.OutOfMemoryError):
        _device.gdn_forward(*(x.bfloat16() for x in args[:3]), *args[3:], num_seqs=1)
