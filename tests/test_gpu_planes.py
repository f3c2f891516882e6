"""The products of the fp32 kernels (bf16 MFMAs over three planes per operand), one term at a time, against 64 bits.

A token that writes nothing (beta = 0) reads o = q S with one nonzero element in q and one in each column of S: a single
product. An operand is the sum of its planes; of a product, the parts left out are at most 2 * 2^-8 * 2^-17 = 2^-24 of it (the
second plane is within 2^-8, the third within 2^-17 of the operand). The others are added by the matrix instruction, whose
additions are not all rounded to nearest: up to a last place, 2^-23, once at the product's size and before that at 2^-7 of it
or less. In all 3 * 2^-24, with a margin of 2 % (a first plane cut off instead of rounded gave 3.7 to 5.7 * 2^-24).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

N, R, D = 128, 2, 128


def values(kind, shape, gen):
    u = torch.rand(shape, generator=gen, dtype=torch.float64)
    sign = torch.where(torch.rand(shape, generator=gen) < 0.5, -1.0, 1.0)
    if kind == "long":                                    # just below 1 + 2^-7: the longest rests after 8 bits cut off
        x = 1 + 2.0 ** -7 - u * 2.0 ** -13
    elif kind == "half":                                  # around 1 + 2^-8: after 8 bits rounded
        x = 1 + 2.0 ** -8 + (u - 0.5) * 2.0 ** -12
    else:                                                 # any significand over 60 binades
        x = (1 + u) * 2.0 ** torch.randint(-30, 30, shape, generator=gen)
    return (sign * x).float()


@pytest.mark.parametrize("kind", ["long", "half", "any"])
def test_single_products(dev, kind):
    from heimdall_amd._device import gdn_forward
    gen = torch.Generator().manual_seed(1)
    a, b = values(kind, (N, R), gen), values(kind, (N, D), gen)
    q, s = torch.zeros(N, R, D), torch.zeros(N, 1, D, D)
    q[:, :, 3], s[:, 0, 3] = a, b
    k = torch.nn.functional.normalize(torch.randn(N, 1, D, generator=gen), dim=-1)
    zero = torch.zeros(N, 1, device=dev)
    print(f"single products {kind}", flush=True)
    o, _ = gdn_forward(q.to(dev), k.to(dev), torch.zeros(N, 1, D, device=dev), zero, zero, num_seqs=N, initial_state=s.to(dev))
    ref = a.double()[:, :, None] * b.double()[:, None]
    err = ((o.cpu().double() - ref).abs() / ref.abs()).max().item()
    print(f"  largest relative error 2^{torch.tensor(err).log2().item():.2f}", flush=True)
    assert err < 1.02 * 3 * 2 ** -24, err
