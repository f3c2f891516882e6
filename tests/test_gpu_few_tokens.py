"""Short chunks of the converted layer: bf_student_inputs against the separate entry points it stands for, and the
token-by-token memory branch of bf_layer_prefill_fwd (up to 16 tokens) against the oracle."""
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
    """Chunks of 2 .. 16 tokens from position 0 (the memory off, then on inside a chunk; with W = 8 rows of the chunk
    itself leave the window), one of 17 on the scan between them, two sequences, whole caches compared."""
    from heimdall_amd import hibrit
    print(f"short chunks {dtype} H={h} G={g} D={d} W={w}", flush=True)
    m = make_core(h, g, d, 32, window=w, sinks=2)
    mg = make_core(h, g, d, 32, window=w, sinks=2).to(dev)
    args = make_inputs(m, 2, 72, seed=31, dtype=dtype)
    ref = tuple(z.float() for z in args)
    c_ref, c_gpu, a = {}, {}, 0
    with torch.no_grad():
        for n in (16, 2, 7, 16, 17, 3, 1, 10):
            o_ref = olayer.student(m, *split(ref, a, a + n), a, c_ref)
            o = hibrit.student(mg, *to_dev(split(args, a, a + n), dev), a, c_gpu)
            assert rel(o, o_ref) < tol, (a, n, rel(o, o_ref))
            a += n
    compare_caches(c_ref, c_gpu, tol)
