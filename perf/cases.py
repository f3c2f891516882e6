"""The work whose speed matters to a user of this package, as cases with seeded inputs, one pass each, and its 64-bit value.

A case is a dict of plain values. Its ``kind`` names the public entry point of one pass:

  layer    ``hibrit.student``: a converted layer over a chunk of tokens, from an empty cache (start 0) or over a full one
  batch    ``hibrit.student_batch``: one token for each of b sequences at their own positions
  delta    ``kernels.delta_rule``: the chunked gated delta rule alone
  train    ``motor.delta_rule_gqa`` forward and backward: one segment of the conversion's training, fp32
  packed   ``gdn_layer.gdn_layer_packed``: the native Gated DeltaNet core on packed sequences of different lengths
  module   ``gdn_layer.GatedDeltaNet.forward`` over its carried cache
  kept     ``teacher.teacher``: a kept full-attention layer over its KV cache, with or without retrieval
"""
import math

import torch
import torch.nn.functional as F

from heimdall_amd import gdn_layer, hibrit, kernels, motor, teacher

W, S = 2048, 4                                            # attention window and sinks of a converted layer
RET = dict(k=16, block=64, window=2048, sinks=4)          # the retrieval defaults of a kept layer
CONV_K = 4
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
RINGS = ("ring_k", "ring_v", "ring_km", "ring_g", "ring_beta", "ring_pos")


def listed():
    layer = dict(kind="layer", b=1, h=24, g=4, d=256, x=5120, dtype="bf16")
    return [
        # a long prompt through a converted layer in one call, the headline workload
        dict(layer, name="layer_prefill_32k", t=32768, start=0),
        # the same prompt as the generation loop feeds it, 2048 tokens at a time over the layer's cache
        dict(layer, name="layer_chunk_2048", t=2048, start=30720),
        # speculative decoding: the last token and one draft, verified in one call
        dict(layer, name="layer_verify_2", t=2, start=32768),
        # one user generating: the smallest call, launches and host time included
        dict(layer, name="layer_decode_1", t=1, start=32768),
        # a server's step: sequences at their own positions, bandwidth bound
        dict(kind="batch", name="layer_decode_batch_64", b=64, h=16, g=4, d=256, x=5120, last=131072, dtype="bf16"),
        # the layer in full precision, as a conversion is checked
        dict(layer, name="layer_prefill_fp32_4k", t=4096, start=0, h=16, dtype="fp32"),
        # the delta-rule operator on a long sequence
        dict(kind="delta", name="delta_rule_32k", b=1, t=32768, h=4, d=256, dtype="bf16"),
        # one time segment of the conversion's training, with every gradient
        dict(kind="train", name="train_segment_8k", b=1, t=8192, g=4, r=6, d=256),
        # prompts of different lengths packed through a native Gated DeltaNet layer
        dict(kind="packed", name="gdn_packed_64k", n=65536, seqs=4, hk=32, hv=32, d=128, dtype="bf16"),
        # a server's step through the whole native layer, its projections included
        dict(kind="module", name="gdn_decode_32", b=32, t=1, hk=32, hv=32, d=128, x=5120, dtype="bf16"),
        # a server's step through a kept attention layer that reads selected blocks of a long cache
        dict(kind="kept", name="kept_decode_retrieval_64", b=64, t=1, n=32768, h=16, g=4, d=256, retrieval=True, dtype="bf16"),
        # a prompt chunk through a kept attention layer, every earlier key visible
        dict(kind="kept", name="kept_chunk_2048", b=1, t=2048, n=14336, h=24, g=4, d=256, retrieval=False, dtype="bf16"),
    ]


def draw(rng):
    def size(lo, hi):                                     # spread over the logarithm, any integer
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    h, g, d = rng.choice([(24, 4, 256), (16, 4, 256), (32, 8, 128), (8, 2, 256)])
    kind = rng.choice(("prefill", "chunk", "few", "layer32", "batch", "delta", "train", "packed", "module", "kept1", "keptn"))
    layer = dict(kind="layer", b=1, h=h, g=g, d=d, x=rng.choice((2048, 4096, 5120)), dtype="bf16")
    if kind == "prefill":
        return dict(layer, b=rng.choice((1, 1, 2)), t=size(64, 12000), start=0)
    if kind == "chunk":
        return dict(layer, t=size(64, 4096), start=size(W + 64, 120000))
    if kind == "few":
        return dict(layer, b=rng.choice((1, 1, 2, 4)), t=rng.choice((1, 2, 3, 5, 8, 16)), start=size(64, 120000))
    if kind == "layer32":
        return dict(layer, h=min(h, 16), t=size(64, 4096), start=rng.choice((0, 3000)), dtype="fp32")
    if kind == "batch":
        return dict(layer, kind="batch", b=size(2, 64), h=min(h, 16), g=min(g, 4), last=size(3000, 120000))
    if kind == "delta":
        return dict(kind="delta", b=rng.choice((1, 1, 3)), t=size(64, 10000), h=rng.choice((2, 4, 16)), d=rng.choice((64, 128, 256)),
                    dtype=rng.choice(("bf16", "bf16", "fp32")))
    if kind == "train":
        return dict(kind="train", b=1, t=size(256, 8192), g=g, r=min(h // g, 6), d=d)
    if kind == "packed":
        hv = rng.choice((16, 32))
        return dict(kind="packed", n=size(1000, 60000), seqs=rng.randint(1, 12), hk=rng.choice((16, hv)), hv=hv, d=128, dtype="bf16")
    if kind == "module":
        return dict(kind="module", b=size(1, 64), t=rng.choice((1, 1, 1, 2, 64)), hk=16, hv=rng.choice((16, 32)), d=128, x=rng.choice((2048, 4096)),
                    dtype="bf16")
    if kind == "kept1":
        return dict(kind="kept", b=size(1, 32), t=1, n=size(4000, 32768), h=h, g=g, d=d, retrieval=rng.random() < 0.6, dtype="bf16")
    return dict(kind="kept", b=1, t=size(2, 2048), n=rng.choice((0, size(300, 14000))), h=h, g=g, d=d, retrieval=False, dtype="bf16")


# ------------------------------------------------------------------------------------------------------------- inputs
class _Rand:
    """Seeded random tensors on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, dtype=torch.float32, scale=1.0):
        y = torch.randn(*shape, device="cuda", generator=self.gen, dtype=dtype)
        return y if scale == 1.0 else y.mul_(scale)

    def uniform(self, *shape):
        return torch.rand(*shape, device="cuda", generator=self.gen)


def _rope(x, pos):
    """Rotary embedding (the first half of the head, base 1e7) of x [b, heads, t, d] at positions pos [b or 1, t]."""
    half = x.shape[-1] // 4
    f = 1e7 ** (-torch.arange(half, device=x.device, dtype=torch.float32) / half)
    a = pos.float()[:, None, :, None] * f
    y = x.float()
    u, v = y[..., :half], y[..., half:2 * half]
    return torch.cat((u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin(), y[..., 2 * half:]), -1).to(x.dtype)


def _core(c, r):
    """A converted layer with the parameters of a trained one: projections near the identity, learned gates."""
    m = hibrit.BifrostCore(hibrit.CoreConfig(c["h"], c["g"], c["d"], c["x"]))
    torch.manual_seed(0)
    m.convert(W, S, 1)
    m = m.cuda()
    with torch.no_grad():
        for p, scale in ((m.fq, 0.2 * c["d"] ** -0.5), (m.fk, 0.2 * c["d"] ** -0.5), (m.ab.weight, c["x"] ** -0.5),
                         (m.mix.weight, c["x"] ** -0.5), (m.mix_lse, 0.1), (m.ab.bias, 0.2)):
            p.add_(r.normal(*p.shape, scale=scale))
        m.mix.bias.fill_(-1.0)
    return m


def _tokens(c, r, b, t, pos):
    """x [b, t, x], q, k with rows of unit mean square (as the q / k norms leave them), v, and the rotated qr, kr."""
    dt, h, g, d = DTYPES[c["dtype"]], c["h"], c["g"], c["d"]
    unit = lambda y: (y * torch.rsqrt(y.square().mean(-1, keepdim=True))).to(dt)
    x, q, k, v = r.normal(b, t, c["x"]).to(dt), unit(r.normal(b, t, h, d)), unit(r.normal(b, t, g, d)), r.normal(b, t, g, d).to(dt)
    qr, kr = (_rope(y.transpose(1, 2), pos).contiguous() for y in (q, k))
    return dict(x=x, q=q, k=k, v=v, qr=qr, kr=kr)


def _ring(c, r, b, pos):
    """The cache of b sequences that are at positions pos [b]: the last W tokens in their slots, the sinks, the memory."""
    dt, g, d = DTYPES[c["dtype"]], c["g"], c["d"]
    slot = torch.arange(W, device="cuda")
    last = pos[:, None] - 1
    held = last - (last - slot) % W                       # the latest position in each slot, negative where there is none
    has = held >= 0
    out = dict(ring_k=r.normal(b, g, W, d).to(dt), ring_v=r.normal(b, g, W, d).to(dt), ring_km=F.normalize(r.normal(b, W, g, d), dim=-1),
               ring_g=-0.01 * r.uniform(b, W, g), ring_beta=torch.sigmoid(r.normal(b, W, g)), S=r.normal(b, g, d, d, scale=0.5),
               sink_k=r.normal(b, g, S, d).to(dt), sink_v=r.normal(b, g, S, d).to(dt))
    for key, where in (("ring_k", has[:, None, :, None]), ("ring_v", has[:, None, :, None]), ("ring_km", has[..., None, None]),
                       ("ring_g", has[..., None]), ("ring_beta", (held >= S)[..., None]), ("S", (pos > W)[:, None, None, None])):
        out[key] = out[key] * where
    out["ring_pos"] = torch.where(has, held, -1)
    return out


def _lengths(c, seed):
    """The lengths of the packed sequences, between half and twice the mean, from the seed."""
    gen = torch.Generator().manual_seed(seed)
    cut = (torch.rand(c["seqs"], generator=gen) + 0.5).cumsum(0)
    ends = (cut / cut[-1] * c["n"]).long()
    ends[-1] = c["n"]
    return torch.cat((torch.zeros(1, dtype=torch.long), ends))


def _gdn(c, r):
    with torch.device("cuda"):
        m = gdn_layer.GatedDeltaNet(gdn_layer.GdnLayerConfig(d=c.get("x", 64), lin_hk=c["hk"], lin_hv=c["hv"], lin_dk=c["d"], lin_dv=c["d"], conv_k=CONV_K))
    with torch.no_grad():
        for p in m.parameters():
            p.copy_(r.normal(*p.shape, scale=p.shape[-1] ** -0.5))
        m.norm.weight.add_(1.0)
        m.dt_bias.copy_(r.normal(*m.dt_bias.shape))
        m.A_log.copy_(-6.0 + 4.0 * r.uniform(*m.A_log.shape))
    return m.to(DTYPES[c["dtype"]])


def _inputs(c, seed):
    r, kind = _Rand(seed), c["kind"]
    if kind == "layer":
        pos = torch.arange(c["start"], c["start"] + c["t"], device="cuda")[None]
        st = dict(core=_core(c, r), pos=c["start"], cache={}, **_tokens(c, r, c["b"], c["t"], pos))
        if c["start"]:
            ring = _ring(c, r, c["b"], pos[:, 0].expand(c["b"]).contiguous())
            ring["ring_pos"] = ring["ring_pos"][0].contiguous()
            if c["start"] <= W:
                ring.pop("S")
            st["cache"] = ring
        return st
    if kind == "batch":
        pos = (c["last"] * r.uniform(c["b"])).long() + 16  # some in their first window, most past it
        return dict(core=_core(c, r), pos=pos, cache=_ring(c, r, c["b"], pos), **_tokens(c, r, c["b"], 1, pos[:, None]))
    if kind == "delta":
        dt, shape = DTYPES[c["dtype"]], (c["b"], c["t"], c["h"], c["d"])
        return dict(q=(F.normalize(r.normal(*shape), dim=-1) * c["d"] ** -0.5).to(dt), k=F.normalize(r.normal(*shape), dim=-1).to(dt),
                    v=r.normal(*shape).to(dt), g=-0.01 * r.uniform(*shape[:3]), beta=torch.sigmoid(r.normal(*shape[:3])))
    if kind == "train":
        b, t, g, n, d = c["b"], c["t"], c["g"], c["r"], c["d"]
        x = [F.normalize(r.normal(b, t, g, n, d), dim=-1) * d ** -0.5, F.normalize(r.normal(b, t, g, d), dim=-1), r.normal(b, t, g, d),
             -0.01 * r.uniform(b, t, g), torch.sigmoid(r.normal(b, t, g)), r.normal(b, g, d, d, scale=0.5)]
        return dict(x=[y.requires_grad_(True) for y in x], do=r.normal(b, t, g, n, d), ds=r.normal(b, g, d, d, scale=0.1))
    if kind == "packed":
        n, hv, dt = c["n"], c["hv"], DTYPES[c["dtype"]]
        return dict(m=_gdn(c, r), z=r.normal(n, (2 * c["hk"] + hv) * c["d"]).to(dt), a=r.normal(n, hv).to(dt), b=r.normal(n, hv).to(dt),
                    zg=r.normal(n, hv * c["d"]).to(dt), cu=_lengths(c, seed).to(device="cuda", dtype=torch.int32))
    if kind == "module":
        dt = DTYPES[c["dtype"]]
        return dict(m=_gdn(c, r), x=r.normal(c["b"], c["t"], c["x"]).to(dt), cache=dict(
            conv=r.normal(c["b"], CONV_K - 1, (2 * c["hk"] + c["hv"]) * c["d"]).to(dt), S=r.normal(c["b"], c["hv"], c["d"], c["d"], scale=0.3)))
    dt, b, t, n, h, g, d = DTYPES[c["dtype"]], c["b"], c["t"], c["n"], c["h"], c["g"], c["d"]
    return dict(qr=r.normal(b, h, t, d, dtype=dt), kr=r.normal(b, g, t, d, dtype=dt), v=r.normal(b, t, g, d, dtype=dt),
                k=r.normal(b, g, n, d, dtype=dt), vt=r.normal(b, g, n, d, dtype=dt))


def prepare(case, seed):
    st = _inputs(case, seed)
    st["kind"] = case["kind"]
    if case["kind"] == "kept":
        layer = hibrit.BifrostCore(hibrit.CoreConfig(case["h"], case["g"], case["d"], case["h"] * case["d"]))
        layer.set_retrieval(**RET) if case["retrieval"] else layer.set_retrieval(None)
        cache, n = {}, case["n"]
        if n:                                             # a cache filled elsewhere is taken over by the layer's first call
            cache = {"k": st.pop("k"), "v": st.pop("vt")}
            layer._teacher(st["qr"][:, :, :1], st["kr"][:, :, :1], st["v"][:, :1], cache)
        st.update(layer=layer, cache=cache, n=n)
    return st


# -------------------------------------------------------------------------------------------------------------- a pass
def run(st):
    kind = st["kind"]
    if kind == "train":
        o, s = motor.delta_rule_gqa(*st["x"][:5], 64, st["x"][5])
        return (o.detach(), s.detach()) + torch.autograd.grad((o, s), st["x"], (st["do"], st["ds"]))
    with torch.no_grad():
        if kind in ("layer", "batch"):
            m, args = st["core"], [st[key] for key in ("x", "q", "k", "v", "qr", "kr")]
            if kind == "batch":
                o, cache = hibrit.student_batch(m, *args, st["pos"], st["cache"]), st["cache"]
                st["pos"] = st["pos"] + 1
            else:
                cache = st["cache"] if st["pos"] else {}
                o = m._student(*args, st["pos"], cache)
                if st["pos"]:
                    st["pos"] += args[0].shape[1]
            return dict(o=o, **{key: cache[key] for key in RINGS + ("sink_k", "sink_v", "S") if cache.get(key) is not None})
        if kind == "delta":
            return kernels.delta_rule(*(st[key] for key in ("q", "k", "v", "g", "beta")))
        if kind == "packed":
            return gdn_layer.gdn_layer_packed(st["m"], st["z"], st["a"], st["b"], st["zg"], st["cu"])
        if kind == "module":
            return dict(o=st["m"](st["x"], st["cache"]), conv=st["cache"]["conv"], S=st["cache"]["S"])
        cache, n = st["cache"], st["n"]
        if n:                                             # back to n positions, as after a rejected draft
            cache["k"], cache["v"] = cache["k"][:, :, :n], cache["v"][:, :, :n]
        else:
            cache = {}
        o = st["layer"]._teacher(st["qr"], st["kr"], st["v"], cache)
        return dict(o=o, k=cache["k"], v=cache["v"])


# ----------------------------------------------------------------------------------------------- what a pass has to do
def _pairs(start, t, span):
    """Visible keys summed over t queries from position start, at most span each."""
    free = max(0, min(t, span - start))
    return free * start + free * (free + 1) // 2 + (t - free) * span


def _delta_flops(n, g, h, d):
    return n * (g * (6 * 64 * d + 4 * d * d) + h * (4 * 64 * d + 2 * d * d))


def work(case):
    c, kind, d = case, case["kind"], case["d"]
    e = 2 if case.get("dtype") == "bf16" else 4
    if kind in ("layer", "batch"):
        b, t, h, g = c["b"], c.get("t", 1), c["h"], c["g"]
        full = [c["start"]] * b if kind == "layer" else [max(16, int(c["last"] * (i + 0.5) / b)) for i in range(b)]
        past = sum(min(W, p) for p in full)                                     # ring rows read
        out = sum(max(0, min(t, p + t - W)) if p else 0 for p in full)          # rows that leave the window from the ring
        mem = sum(max(0, min(t, p + t - W)) for p in full)                      # tokens that write the memory
        par = (h + g) * d * d * 4 + (2 * g + h) * (c["x"] + 1) * 4
        tok = c["x"] * e + 2 * (h + g) * d * e + g * d * e + h * d * 4
        ring = g * (2 * d * e + d * 4 + 8)
        state = sum(g * d * d * 4 * (2 if p > W else 1) for p in full if p + t > W)
        flops = 4 * d * h * sum(_pairs(p, t, W + S) for p in full) + b * t * (2 * (h + g) * d * d + 2 * c["x"] * (2 * g + h))
        flops += _delta_flops(mem, g, h, d) if t > 1 else mem * (4 * g + 2 * h) * d * d
        return dict(bytes=par + b * t * tok + b * min(t, W) * ring + past * g * 2 * d * e + out * g * (d * 4 + 8) + state, flops=flops)
    if kind == "delta":
        n = c["b"] * c["t"] * c["h"]
        return dict(bytes=n * (3 * d * e + 8 + 4 * d) + c["b"] * c["h"] * d * d * 4, flops=_delta_flops(c["b"] * c["t"], c["h"], c["h"], d))
    if kind == "train":
        n, g, r = c["b"] * c["t"], c["g"], c["r"]
        rows = n * (g * r * d * 4 + g * (2 * d + 2) * 4)
        return dict(bytes=2 * rows + 2 * n * g * r * d * 4 + 4 * c["b"] * g * d * d * 4, flops=3 * _delta_flops(n, g, g * r, d))
    if kind in ("packed", "module"):
        hk, hv, b = c["hk"], c["hv"], c.get("b", c.get("seqs"))
        n, wide = c.get("n", c.get("t", 1) * b), (2 * hk + hv) * d
        flops, state = _delta_flops(n, hv, hv, d) + 2 * n * wide * CONV_K, b * hv * d * d * 4
        if kind == "packed":
            return dict(bytes=n * (wide * e + 2 * hv * e + 2 * hv * d * e) + state, flops=flops)
        if c["t"] == 1:
            flops = n * hv * 6 * d * d
        mats = c["x"] * (wide + 2 * hv * d + 2 * hv)
        return dict(bytes=mats * e + n * 2 * c["x"] * e + 2 * b * (CONV_K - 1) * wide * e + 2 * state, flops=flops + 2 * n * mats)
    b, t, n, h, g = c["b"], c["t"], c["n"], c["h"], c["g"]
    new = b * t * ((h + 2 * g) * d * e + 2 * g * d * e + h * d * e)
    if c["retrieval"] and t == 1 and n + 1 - RET["sinks"] - RET["window"] >= RET["k"] * RET["block"]:
        keys, blocks = RET["sinks"] + RET["k"] * RET["block"] + RET["window"], max(0, n - RET["window"] - RET["sinks"]) // RET["block"]
        return dict(bytes=new + b * g * (keys + blocks) * 2 * d * e, flops=b * h * d * 4 * (keys + blocks))
    return dict(bytes=new + b * g * n * 2 * d * e, flops=b * h * 4 * d * _pairs(n, t, n + t))


def tolerance(case):
    # Distances from the 64-bit value, measured: operands rounded to bf16 with sums in fp32 2e-3 to 6e-3, fp32 throughout
    # 3e-7 to 9e-7. Two correct implementations are at most the sum of theirs apart; fp32 has four times the largest.
    return {"rel": 1.2e-2 if case.get("dtype") == "bf16" else 4e-6}


# ------------------------------------------------------------------------------------------------- the value in 64 bits
def _delta64(q, k, v, g, beta, s):
    """The gated delta rule in chunks of 64: q [b, t, g, r, d], k, v [b, t, g, d], g, beta [b, t, g], s [b, g, d, d] or None."""
    b, t, G, R, d = q.shape
    n, pad = -(-t // 64), -t % 64
    rows = lambda y: F.pad(y.double(), (0, 0) * (y.dim() - 2) + (0, pad)).reshape(b, n, 64, *y.shape[2:])
    q, k, v = rows(q).permute(1, 0, 3, 4, 2, 5), rows(k).permute(1, 0, 3, 2, 4), rows(v).permute(1, 0, 3, 2, 4)
    g, beta = rows(g).permute(1, 0, 3, 2).cumsum(-1), rows(beta).permute(1, 0, 3, 2)[..., None]
    low = torch.ones(64, 64, dtype=torch.bool, device=q.device).tril()
    decay = (g[..., :, None] - g[..., None, :]).masked_fill(~low, float("-inf")).exp()
    kt = k.transpose(-1, -2).contiguous()
    a = -((k * beta) @ kt * decay).tril(-1)
    inv = torch.eye(64, dtype=a.dtype, device=a.device) + a
    for _ in range(5):                                    # (I - a)^-1 of a strictly lower a, by doubling
        a = a @ a
        inv = inv + inv @ a
    e = g.exp()[..., None]
    u, w = inv @ (v * beta), inv @ (k * beta * e)
    tail = k * (g[..., -1:] - g).exp()[..., None]
    s = torch.zeros(b, G, d, d, dtype=torch.float64, device=q.device) if s is None else s.double()
    out = []
    for i in range(n):
        new = u[i] - w[i] @ s
        out.append((q[i] * e[i][:, :, None]) @ s[:, :, None] + (q[i] @ kt[i][:, :, None] * decay[i][:, :, None]) @ new[:, :, None])
        s = s * e[i][:, :, -1:] + tail[i].transpose(-1, -2) @ new
    return torch.stack(out, 1).permute(0, 1, 4, 2, 3, 5).reshape(b, n * 64, G, R, d)[:, :t], s


def _attend64(q, k, v, see):
    """q [R, t, d] over k, v [n, d] where see [t, n]: the rows [R, t, d] and their log-sum-exp [R, t]."""
    x = (q.double() @ k.double().t().contiguous() * q.shape[-1] ** -0.5).masked_fill_(~see, float("-inf"))
    lse = x.logsumexp(-1)
    return x.sub_(lse[..., None]).exp_() @ v.double(), lse


def _student64(m, st, start, cache):
    """A converted layer's chunk at positions start .. in 64 bits. Returns o [b, t, h, d] and the new cache."""
    x, q, k, v, qr, kr = (st[key] for key in ("x", "q", "k", "v", "qr", "kr"))
    b, t, H, d = q.shape
    G = k.shape[2]
    R, dev = H // G, q.device
    D = lambda y: y.detach().double()
    heads = lambda y, f: F.normalize((D(y).transpose(1, 2) @ D(f)), dim=-1).transpose(1, 2)
    qm, km = heads(q, m.fq) * d ** -0.5, heads(k, m.fk)
    pos = torch.arange(start, start + t, device=dev)
    a, bb = F.linear(D(x), D(m.ab.weight), D(m.ab.bias)).chunk(2, -1)
    g = -D(m.A_log).exp() * F.softplus(a + D(m.dt_bias)) * D(m.decay_mask)
    beta = torch.sigmoid(bb) * (pos >= S)[None, :, None]
    if not cache:
        cache = dict(ring_k=kr.new_zeros(b, G, W, d), ring_v=v.new_zeros(b, G, W, d), ring_km=km.new_zeros(b, W, G, d), ring_g=g.new_zeros(b, W, G),
                     ring_beta=g.new_zeros(b, W, G), ring_pos=torch.full((W,), -1, device=dev), sink_k=kr[:, :, :S], sink_v=v.transpose(1, 2)[:, :, :S])
    old = torch.arange(start - W, start, device=dev)
    at = old % W
    ok = cache["ring_pos"][at] == old
    where = torch.cat((torch.arange(S, device=dev), torch.where(ok, old, -1), pos))
    sink = torch.arange(len(where), device=dev) < S
    o, lse = torch.empty(b, t, H, d, dtype=torch.float64, device=dev), torch.empty(b, t, H, dtype=torch.float64, device=dev)
    for i in range(b):
        for j in range(G):
            keys = torch.cat((cache["sink_k"][i, j], cache["ring_k"][i, j, at], kr[i, j]))
            vals = torch.cat((cache["sink_v"][i, j], cache["ring_v"][i, j, at], v[i, :, j]))
            for p in range(0, t, 1024):
                n = min(1024, t - p)
                near = torch.cat((torch.arange(S, device=dev), torch.arange(S + p, S + W + p + n, device=dev)))
                kp, qp = where[near], pos[p:p + n, None]
                see = (kp >= 0) & (kp <= qp) & (sink[near] | ((qp - kp < W) & (kp >= S)))
                y, z = _attend64(qr[i, j * R:(j + 1) * R, p:p + n], keys[near], vals[near], see)
                o[i, p:p + n, j * R:(j + 1) * R], lse[i, p:p + n, j * R:(j + 1) * R] = y.transpose(0, 1), z.t()
    new = dict(cache)
    if start + t > W:
        live = ok[None, :, None]
        past = lambda key, y: torch.cat((D(cache[key][:, at]) * (live if y.dim() == 3 else 1.0), y), 1)[:, :t]
        wv = torch.cat((D(cache["ring_v"][:, :, at]).transpose(1, 2), D(v)), 1)[:, :t]
        om, new["S"] = _delta64(qm.reshape(b, t, G, R, d), past("ring_km", km), wv, past("ring_g", g), past("ring_beta", beta), cache.get("S"))
        z = F.linear(D(x), D(m.mix.weight), D(m.mix.bias)) + D(m.mix_lse) * (lse - math.log(W))
        gate = (torch.sigmoid(z) * (pos >= W)[None, :, None])[..., None]
        o = o + gate * (D(m.mem_scale)[:, None] * om.reshape(b, t, H, d) - o)
    n = min(t, W)
    slot = pos[-n:] % W
    for key, y in (("ring_k", kr), ("ring_v", v.transpose(1, 2)), ("ring_km", km), ("ring_g", g), ("ring_beta", beta)):
        new[key] = D(cache[key]).clone()
        if y.dim() == 4 and key != "ring_km":
            new[key][:, :, slot] = D(y[:, :, -n:])
        else:
            new[key][:, slot] = D(y[:, -n:])
    new["ring_pos"] = cache["ring_pos"].clone()
    new["ring_pos"][slot] = pos[-n:]
    return dict(o=o, **{key: new[key] for key in RINGS + ("sink_k", "sink_v", "S") if new.get(key) is not None})


def _native64(m, z, a, b, zg, prefix, s):
    """The native layer's core on one sequence batch: z [B, T, C], a, b [B, T, hv], zg [B, T, hv, d]. Returns the rows and the state."""
    c, D = m.c, lambda y: y.detach().double()
    B, T, _ = z.shape
    full = F.pad(D(z), (0, 0, CONV_K - 1, 0)) if prefix is None else torch.cat((D(prefix), D(z)), 1)
    y = F.silu(sum(full[:, j:j + T] * D(m.conv1d.weight)[:, 0, j] for j in range(CONV_K)))
    q, k, v = (u.reshape(B, T, -1, c.lin_dk) for u in y.split((m.kd, m.kd, m.vd), -1))
    norm = lambda u: (u * torch.rsqrt(u.square().sum(-1, keepdim=True) + 1e-6)).repeat_interleave(c.lin_hv // c.lin_hk, 2)
    g = -D(m.A_log).exp() * F.softplus(D(a) + D(m.dt_bias))
    o, s = _delta64(norm(q)[:, :, :, None] * c.lin_dk ** -0.5, norm(k), v, g, torch.sigmoid(D(b)), s)
    o = o.reshape(B, T, c.lin_hv, c.lin_dv)
    return D(m.norm.weight) * o * torch.rsqrt(o.square().mean(-1, keepdim=True) + m.norm.eps) * F.silu(D(zg)), s, full[:, 1 - CONV_K:]


def _see(c, q, keys, n, t):
    """The keys [t, n] that the queries q [R, t, d] of one KV head attend to."""
    at, p = torch.arange(n, device=q.device), torch.arange(n - t, n, device=q.device)
    s, w, size, k = (RET[key] for key in ("sinks", "window", "block", "k"))
    if not (c["retrieval"] and t == 1 and n - s - w >= k * size):
        return at <= p[:, None]
    nb, nc = (n - s) // size, max(n - w - s, 0) // size
    blocks = keys[s:s + nb * size].double().reshape(nb, size, -1)[:nc]
    bound = torch.maximum(q.double() * blocks.amin(1)[:, None, None], q.double() * blocks.amax(1)[:, None, None]).sum(-1).amax((1, 2))
    best = torch.sort(-bound, stable=True).indices[:k]
    see = (at < s) | (at >= s + nc * size)
    return (see | torch.isin((at - s).div(size, rounding_mode="floor"), best))[None]


@torch.no_grad()
def exact(case, seed):
    c, st, kind = case, _inputs(case, seed), case["kind"]
    if kind == "layer":
        return _student64(st["core"], st, c["start"], st["cache"])
    if kind == "batch":
        got = []
        for i in range(c["b"]):
            p = int(st["pos"][i])
            cache = {key: y[i:i + 1] if key != "ring_pos" else y[i] for key, y in st["cache"].items()}
            got.append(_student64(st["core"], {key: st[key][i:i + 1] for key in ("x", "q", "k", "v", "qr", "kr")}, p, cache))
        return {key: torch.stack([y[key] for y in got]) if key == "ring_pos" else torch.cat([y[key] for y in got]) for key in got[0]}
    if kind == "delta":
        o, s = _delta64(st["q"][:, :, :, None], st["k"], st["v"], st["g"], st["beta"], None)
        return o[:, :, :, 0], s
    if kind == "train":
        x = [y.detach().double().requires_grad_(True) for y in st["x"]]
        with torch.enable_grad():
            o, s = _delta64(*x)
            grads = torch.autograd.grad((o, s), x, (st["do"].double(), st["ds"].double()))
        return (o.detach(), s.detach()) + grads
    if kind == "packed":
        out, cu = [], st["cu"].tolist()
        for a, e in zip(cu, cu[1:]):
            rows = [st[key][None, a:e] for key in ("z", "a", "b", "zg")]
            rows[3] = rows[3].reshape(1, e - a, c["hv"], c["d"])
            out.append(_native64(st["m"], *rows, None, None)[:2])
        return torch.cat([y[0] for y, _ in out]).reshape(c["n"], -1), torch.cat([s for _, s in out])
    if kind == "module":
        m, x = st["m"], st["x"].double()
        lin = lambda p: x @ p.weight.double().t().contiguous()
        zg = lin(m.in_proj_z).reshape(c["b"], c["t"], c["hv"], c["d"])
        o, s, conv = _native64(m, lin(m.in_proj_qkv), lin(m.in_proj_a), lin(m.in_proj_b), zg, st["cache"]["conv"], st["cache"]["S"])
        return dict(o=o.reshape(c["b"], c["t"], -1) @ m.out_proj.weight.double().t().contiguous(), conv=conv, S=s)
    k, v = torch.cat((st["k"], st["kr"]), 2), torch.cat((st["vt"], st["v"].transpose(1, 2)), 2)
    b, t, R, n = c["b"], c["t"], c["h"] // c["g"], k.shape[2]
    o = torch.empty(b, t, c["h"], c["d"], dtype=torch.float64, device="cuda")
    for i in range(b):
        for j in range(c["g"]):
            q, kj = st["qr"][i, j * R:(j + 1) * R], k[i, j]
            see = _see(c, q, kj, n, t)
            for p in range(0, t, 1024):
                o[i, p:p + 1024, j * R:(j + 1) * R] = _attend64(q[:, p:p + 1024], kj, v[i, j], see[p:p + 1024])[0].transpose(0, 1)
    return dict(o=o, k=None, v=None)
