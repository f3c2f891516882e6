"""Short chunks of the converted layer: bf_student_inputs against the separate entry points it stands for, and the
token-by-token memory branch of bf_layer_prefill_fwd (up to 12 tokens in fp32; in bf16 8 at 4 query heads per KV head or
fewer, else 5) and the scan after it against the oracle."""
import pytest
import torch

from oracle import layer as olayer
from test_gpu_decode import compare_caches, make_core, make_inputs, rel, split, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,t,h,g,d,dm", [(1, 2, 24, 4, 256, 5120), (2, 8, 4, 2, 64, 40), (1, 17, 32, 8, 128, 264),
                                          (1, 65, 6, 2, 256, 128), (4, 64, 48, 8, 64, 136)])
@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16])
def test_student_inputs_equal_separate_calls(dev, b, t, h, g, d, dm, out):
    """The same products and sums in the same order: bit for bit. Token tiles of 16, groups of 64 and the 256-token
    limit, one and two gate tiles (2G + H up to 64), q rows that are views of a wider tensor."""
    from heimdall_amd import hibrit
    print(f"student inputs B={b} t={t} H={h} G={g} D={d} d_model={dm} {out}", flush=True)
    m = make_core(h, g, d, dm, window=16, sinks=3).to(dev)
    x, q, k, _, _, _ = to_dev(make_inputs(m, b, t, seed=3, dtype=torch.bfloat16), dev)
    wide = torch.cat((q, q), 3)[..., :d]                   # head rows 2 d apart
    with torch.no_grad():
        got = hibrit._few_inputs(m, x, wide, k, 1, out)
        ab, z = hibrit._gate_logits(m, x)
        ref = hibrit._mem_inputs_bf16(m, ab, q, k, 1, out) + (z,)
    for name, a_, b_ in zip(("qm", "km", "g", "beta", "z"), got, ref):
        assert torch.equal(a_, b_), (name, rel(a_, b_))


# fp32: sums of D products and 16 state updates in fp32, ~1e-6; bf16: operands rounded to bf16 (2^-9 each)


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-4), (torch.bfloat16, 2e-2)])
@pytest.mark.parametrize("h,g,d,w", [(4, 2, 64, 8), (12, 2, 128, 16), (8, 1, 256, 24)])
def test_short_chunks_match_oracle(dev, dtype, tol, h, g, d, w):
    """Chunks of 2 .. 17 tokens from position 0 (the memory off, then on inside a chunk; with W = 8 rows of the chunk
    itself leave the window), on either side of the lines at 5, 8 and 12 tokens, two sequences, whole caches compared."""
    from heimdall_amd import hibrit
    print(f"short chunks {dtype} H={h} G={g} D={d} W={w}", flush=True)
    m = make_core(h, g, d, 32, window=w, sinks=2)
    mg = make_core(h, g, d, 32, window=w, sinks=2).to(dev)
    args = make_inputs(m, 2, 129, seed=31, dtype=dtype)
    ref = tuple(z.float() for z in args)
    c_ref, c_gpu, a = {}, {}, 0
    with torch.no_grad():
        for n in (16, 2, 7, 16, 17, 3, 1, 10, 4, 5, 6, 8, 9, 12, 13):
            o_ref = olayer.student(m, *split(ref, a, a + n), a, c_ref)
            o = hibrit.student(mg, *to_dev(split(args, a, a + n), dev), a, c_gpu)
            assert rel(o, o_ref) < tol, (a, n, rel(o, o_ref))
            a += n
    compare_caches(c_ref, c_gpu, tol)


@pytest.mark.parametrize("dtype,b,g,r,d,t", [(torch.float32, 1, 2, 2, 128, 300), (torch.float32, 2, 2, 3, 64, 5),
                                             (torch.bfloat16, 2, 2, 3, 64, 3)])
def test_workspace_of_the_plain_layout(dev, monkeypatch, dtype, b, g, r, d, t):
    """bf_layer_prefill_fwd with a workspace that has no room for the fp32 scan's planes, nor for anything of its own in a short
    chunk, against the full one: the same values (the scan's sums in another order, 1e-5; the short chunk's bits)."""
    from heimdall_amd import _lib, hibrit
    h, w = g * r, 16
    al = lambda n: (n + 255) // 256 * 256
    es = 2 if dtype == torch.bfloat16 else 4
    n = _lib.ctypes.c_size_t(0)
    _lib.check(_lib.load().bf_gdn_workspace_size(b * t, b, g, r, d, 1 if es == 2 else 0, 0, _lib.ctypes.byref(n)), "size")
    planes = 2 * (b * t // 64 + b) * g * (d // 16) * (d // 32 + 2) * 1536 if es == 4 else 0
    plain = sum(map(al, (b * t * h * d * es, b * t * g * d * es, b * t * g * d * es, b * t * g * 4, b * t * g * 4,
                         b * t * h * d * es, b * t * h * d * es, b * g * d * d * 4))) + al(n.value - planes)
    if es == 2:                                            # the window's key parts: 3 slots per XCD in 8 parts
        plain += 8 * 3 * 8 * 128 * (d + 4) * 4
    m = make_core(h, g, d, 32, window=w, sinks=2).to(dev)
    args = to_dev(make_inputs(m, b, 40 + t, seed=6, dtype=dtype), dev)
    c0, c1 = {}, {}
    with torch.no_grad():
        for c in (c0, c1):
            hibrit.student(m, *split(args, 0, 40), 0, c)
        ref = hibrit.student(m, *split(args, 40, 40 + t), 40, c0)
        got = []

        def small(nbytes, size_fn, size_args, dev_):
            got.append(nbytes)
            return hibrit.workspace(plain, dev_)

        monkeypatch.setattr(hibrit, "workspace_or_min", small)
        o = hibrit.student(m, *split(args, 40, 40 + t), 40, c1)
    assert any(x >= plain for x in got)
    assert rel(o, ref) < 1e-5 and rel(c1["S"], c0["S"]) < 1e-5


@pytest.mark.parametrize("h,g,b", [(4, 2, 65), (8, 1, 66)])
def test_memory_inputs_do_not_depend_on_the_batch(dev, h, g, b):
    """Short chunks whose memory inputs come from the separate calls (more than 256 tokens in all) keep them in fp32 for the
    ring, as the fused call does."""
    from heimdall_amd import hibrit
    t, d, w = 4, 64, 8
    m = make_core(h, g, d, 32, window=w, sinks=2).to(dev)
    x, q, k, v, qr, kr = to_dev(make_inputs(m, b, t, seed=5, dtype=torch.bfloat16), dev)
    c = {}
    with torch.no_grad():
        hibrit.student(m, x, q, k, v, qr, kr, 0, c)
        km = hibrit._project_bf16(k, m.fk, 1.0, torch.float32)
    slot = torch.arange(t, device=dev) % w
    assert torch.equal(c["ring_km"][:, slot], km)
