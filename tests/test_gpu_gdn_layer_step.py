"""bf_gdn_layer_step (one token per sequence through the native layer in one launch) against the separate calls it
stands for, and the conv pass at the token counts where its block length changes."""
import pytest
import torch

from test_gpu_gdn_layer import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("b,hk,hv,d,K,prefixed", [(1, 1, 1, 64, 4, True), (3, 2, 6, 128, 4, True), (2, 2, 2, 256, 2, True),
                                                  (2, 1, 2, 128, 4, False), (5, 3, 3, 64, 7, True)])
def test_layer_step_equals_separate_calls(dev, dtype, b, hk, hv, d, K, prefixed):
    """out, the state and the conv cache. fp32: sums of D terms in another order, ~1e-6; bf16: q, k, v stay fp32 in both,
    so only values on a rounding edge of o or the norm differ by one bf16 step (2^-8) here and there."""
    from heimdall_amd import gdn_layer as gl
    from heimdall_amd.kernels import gdn_step
    print(f"gdn layer step B={b} HK={hk} HV={hv} D={d} K={K} {dtype}", flush=True)
    torch.manual_seed(1)
    m = gl.GatedDeltaNet(gl.GdnLayerConfig(d=32, lin_hk=hk, lin_hv=hv, lin_dk=d, lin_dv=d, conv_k=K))
    with torch.no_grad():
        m.conv1d.weight.normal_(0, 0.5)
        m.A_log.normal_(-2, 0.5)
        m.dt_bias.normal_()
        m.norm.weight.normal_(1, 0.2)
    m = m.to(device=dev, dtype=dtype)
    m.A_log.data = m.A_log.data.float()                    # each parameter in its own dtype
    C = (2 * hk + hv) * d
    wide = torch.randn(b, C + 8, device=dev).to(dtype)
    z, a, bb = wide[:, :C], torch.randn(b, hv, device=dev).to(dtype), torch.randn(b, hv, device=dev).to(dtype)
    zg = torch.randn(b, hv * d, device=dev).to(dtype)
    prefix = torch.randn(b, K - 1, C, device=dev).to(dtype) if prefixed else None
    s0 = torch.randn(b, hv, d, d, device=dev) * 0.3
    with torch.no_grad():
        out, conv, s = gl._layer_step(m, z, a, bb, zg, prefix, s0)
        q, k, v, g, beta = gl.conv_inputs(z, m.conv1d.weight[:, 0], prefix, a, bb, m.A_log, m.dt_bias, hk, hv, d,
                                          cu_seqlens=gl._seqlens(b, 1, dev), out_dtype=torch.float32)
        o, s_ref = gdn_step(q, k, v, g, beta, s0)
        ref = gl.gated_norm(o.to(dtype), zg.view(b, hv, d), m.norm.weight, m.norm.eps).reshape(b, -1)
    full = torch.cat((prefix if prefixed else torch.zeros(b, K - 1, C, device=dev, dtype=dtype), z[:, None]), 1)
    assert torch.equal(conv, full[:, 1:])
    assert rel(s, s_ref) < 1e-5, rel(s, s_ref)
    assert rel(out, ref) < (1e-5 if dtype == torch.float32 else 2e-3), rel(out, ref)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("b,hk,hv,d,x", [(1, 1, 2, 64, 8), (3, 2, 2, 128, 520), (2, 1, 1, 128, 2056), (5, 1, 3, 64, 1024)])
def test_step_with_gates_inside(dev, dtype, b, hk, hv, d, x):
    """The gate logits formed in the step kernel against the projections: rows shorter and longer than one pass of the
    workgroup. fp32: sums in another order; bf16: a logit on a rounding edge moves by one step (2^-8 of it) here and there."""
    from heimdall_amd import gdn_layer as gl
    print(f"gates inside B={b} HV={hv} D={d} d_model={x} {dtype}", flush=True)
    torch.manual_seed(2)
    m = gl.GatedDeltaNet(gl.GdnLayerConfig(d=x, lin_hk=hk, lin_hv=hv, lin_dk=d, lin_dv=d)).to(device=dev, dtype=dtype)
    u = torch.randn(b, 1, x, device=dev).to(dtype)
    cache = lambda: dict(conv=torch.ones(b, 3, (2 * hk + hv) * d, device=dev, dtype=dtype), S=torch.ones(b, hv, d, d, device=dev) * 0.1)
    assert gl._gates_inside(m, u)
    c0, c1 = cache(), cache()
    o = m(u, c0)
    handle = m.in_proj_a.register_forward_hook(lambda *a: None)          # a hooked projection is called
    assert not gl._gates_inside(m, u)
    ref = m(u, c1)
    handle.remove()
    tol = 1e-5 if dtype == torch.float32 else 4e-3
    assert rel(o, ref) < tol and rel(c0["S"], c1["S"]) < tol and torch.equal(c0["conv"], c1["conv"])
    assert not gl._gates_inside(m, u[..., :x - 1] if x % 8 == 0 else u)


def make_layer(dev, dtype, hk, hv, d, x, norm=None):
    from heimdall_amd import gdn_layer as gl
    torch.manual_seed(4)
    m = gl.GatedDeltaNet(gl.GdnLayerConfig(d=x, lin_hk=hk, lin_hv=hv, lin_dk=d, lin_dv=d))
    if norm is not None:
        m.norm = norm
    m = m.to(device=dev, dtype=dtype)
    with torch.no_grad():
        m.conv1d.weight.normal_(0, 0.5)
    return m


def step_cache(dev, dtype, b, hk, hv, d):
    gen = torch.Generator(device=dev).manual_seed(b)
    return dict(conv=torch.randn(b, 3, (2 * hk + hv) * d, device=dev, generator=gen).to(dtype),
                S=torch.randn(b, hv, d, d, device=dev, generator=gen) * 0.1)


@pytest.mark.parametrize("b,d,inside", [(64, 128, True), (65, 128, False), (64, 64, True), (3, 256, False)])
def test_where_the_gates_are_formed(dev, b, d, inside):
    """The last batch with the gate logits in the step kernel, the first without, and D = 256, which never has them; each equals
    the same step with its projections called (bf16, tolerance as above)."""
    from heimdall_amd import gdn_layer as gl
    print(f"gates B={b} D={d}", flush=True)
    m = make_layer(dev, torch.bfloat16, 1, 2, d, 264)
    u = torch.randn(b, 1, 264, device=dev).bfloat16()
    assert gl._gates_inside(m, u) == inside
    c0, c1 = (step_cache(dev, torch.bfloat16, b, 1, 2, d) for _ in range(2))
    o = m(u, c0)
    m.in_proj_b.register_forward_hook(lambda *a: None)
    ref = m(u, c1)
    assert rel(o, ref) < 4e-3 and rel(c0["S"], c1["S"]) < 4e-3 and torch.equal(c0["conv"], c1["conv"])


@pytest.mark.parametrize("how", ["hook", "pre-hook", "global hook", "instance"])
def test_step_calls_a_changed_norm(dev, how):
    """A norm with hooks or a forward of its own is called: its doubled output doubles the layer's (bf16, tolerance as above)."""
    from heimdall_amd import gdn_layer as gl
    m = make_layer(dev, torch.bfloat16, 1, 2, 64, 72)
    u = torch.randn(2, 1, 72, device=dev).bfloat16()
    handle = m.in_proj_a.register_forward_hook(lambda *a: None)          # the same projections in both calls
    ref = m(u, step_cache(dev, torch.bfloat16, 2, 1, 2, 64))
    if how == "hook":
        m.norm.register_forward_hook(lambda mod, args, out: 2 * out)
    elif how == "pre-hook":
        m.norm.register_forward_pre_hook(lambda mod, args: (args[0], args[1] * 0))
    elif how == "global hook":
        handle = torch.nn.modules.module.register_module_forward_hook(
            lambda mod, args, out: 2 * out if mod is m.norm else None)
    else:
        m.norm.forward = lambda x, z: 2 * gl.gated_norm(x, z, m.norm.weight, m.norm.eps)
    try:
        o = m(u, step_cache(dev, torch.bfloat16, 2, 1, 2, 64))
    finally:
        handle.remove()
    if how == "pre-hook":                                  # a gate of zero: SiLU(0) = 0
        assert ref.any() and not o.any()
    else:
        assert rel(o, 2 * ref) < 4e-3


def test_step_runs_each_projection_once(dev):
    """Where the step call does not apply (here: another norm), as where it does, every projection runs once."""
    from heimdall_amd import gdn_layer as gl

    class Norm(gl.GatedNorm):
        pass

    for norm in (None, Norm(64)):
        m = make_layer(dev, torch.bfloat16, 1, 2, 64, 72, norm)
        calls = {}
        for name in ("in_proj_qkv", "in_proj_z", "in_proj_a", "in_proj_b", "out_proj"):
            getattr(m, name).register_forward_hook(lambda mod, args, out, name=name: calls.__setitem__(name, calls.get(name, 0) + 1))
        m(torch.randn(2, 1, 72, device=dev).bfloat16(), step_cache(dev, torch.bfloat16, 2, 1, 2, 64))
        assert len(calls) == 5 and set(calls.values()) == {1}, calls


@pytest.mark.parametrize("n", [1, 5, 64, 700, 1400, 5000, 5440, 5441])
def test_conv_blocks(dev, n):
    """Token blocks of 4, 8, 16, 32 and 64 (H = 32, D = 128: from 681, 1361, 2721 and 5441 tokens on) over packed sequences give
    the same bits as one token at a time with the rows before it as its prefix."""
    from heimdall_amd import gdn_layer as gl
    hk = hv = 32
    d, K = 128, 4
    print(f"conv blocks n={n}", flush=True)
    C = 3 * hk * d
    gen = torch.Generator(device=dev).manual_seed(n)
    z = torch.randn(n, C, device=dev, generator=gen).bfloat16()
    w = torch.randn(C, K, device=dev, generator=gen)
    a, b = (torch.randn(n, hv, device=dev, generator=gen) for _ in range(2))
    al, dt = torch.randn(hv, device=dev, generator=gen), torch.randn(hv, device=dev, generator=gen)
    cut = sorted({0, n, n // 3, n // 2})
    cu = torch.tensor(cut, dtype=torch.int32, device=dev)
    run = lambda z_, pre, a_, b_, cu_: gl.conv_inputs(z_, w, pre, a_, b_, al, dt, hk, hv, d, cu_seqlens=cu_)
    with torch.no_grad():
        got = run(z, None, a, b, cu)
        for i in sorted({0, n // 3, n // 2, n - 1}):
            lo = max(c for c in cut if c <= i)
            rows = z[max(lo, i - 3):i]
            pre = torch.cat((torch.zeros(K - 1 - rows.shape[0], C, device=dev, dtype=z.dtype), rows))[None]
            one = run(z[i:i + 1], pre, a[i:i + 1], b[i:i + 1], torch.tensor([0, 1], dtype=torch.int32, device=dev))
            for x, y in zip(got, one):
                assert torch.equal(x[i:i + 1], y), i
