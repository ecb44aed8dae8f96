"""The Q/K pass with one to eight tokens per wave, bit for bit.

How many tokens a wave walks follows from the sequence length; a token's own result does not depend on
it. The pass over the first S rows must return the first S rows of the pass over all of them (eight
tokens per wave), in place and to another layout, with the queries' 1/rms; the key-norm maximum is the
one of those rows. The long pass itself is held to the oracle elsewhere (test_gpu_rope, test_gpu_block).
S covers a single token, a last wave without any, and both sides of each step in tokens per wave."""

import pytest
import torch

pytestmark = pytest.mark.gpu

LONG, N = 28700, 40


@pytest.fixture(scope="module")
def operands(pkg, dev):
    g = torch.Generator(device=dev).manual_seed(71)
    x = torch.randn(LONG, N * 128, device=dev, generator=g).to(torch.bfloat16)
    gamma = 1.0 + 0.1 * torch.randn(N * 128, device=dev, generator=g)
    ang = torch.randn(LONG, 64, device=dev, generator=g)
    return x, gamma, ang.cos(), ang.sin(), torch.rand(LONG, 2 * N, device=dev, generator=g) * 256


@pytest.mark.parametrize("pairs", ["interleaved", "halves"])
@pytest.mark.parametrize("S", [1, 3, 511, 4095, 4096, 4097, 8193, 16385, 24577])
def test_tokens_per_wave_give_the_same_bits(pkg, dev, operands, S, pairs):
    ops, (x, gamma, cos, sin, ss) = pkg.attention_ops, operands
    outs = []
    for n in (LONG, S):
        y, rr = x[:n].clone(), torch.empty(n, device=dev)
        kmax = ops.qk_rmsnorm_rope_(y, gamma, cos=cos[:n], sin=sin[:n], want_max=True, rope_pairs=pairs,
                                    q_sumsq=ss[:n], q_rr=rr)
        to = torch.empty(N, n, 128, dtype=torch.bfloat16, device=dev)
        ops.qk_rmsnorm_rope_to(x[:n], to.permute(1, 0, 2), gamma, cos=cos[:n], sin=sin[:n], rope_pairs=pairs)
        assert torch.equal(to.permute(1, 0, 2).reshape(n, -1), y)
        outs.append((y[:S], rr[:S]))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    ref = outs[1][0].double().view(S, N, 128).norm(dim=-1).amax(0)
    # fp32 sums of 128 squares, every partial sum rounded up or down by at most 2^-24 of itself
    assert bool(((kmax.double() - ref).abs() <= 128 * 2.0**-24 * ref).all())


@pytest.mark.parametrize("pairs", ["interleaved", "halves"])
@pytest.mark.parametrize("heads", [4, 16, 20, 40])
@pytest.mark.parametrize("S", [1, 65, 4097, 28673])
def test_key_norm_maximum_of_every_workgroup_size(pkg, dev, S, heads, pairs):
    """The pass with the key-norm maximum against the pass without it, bit for bit, and the maximum against
    the norms of its rows (the last of them the longest in every other head)."""
    g = torch.Generator(device=dev).manual_seed(S + heads)
    x = torch.randn(S, heads * 128, device=dev, generator=g).to(torch.bfloat16)
    gamma = 1.0 + 0.1 * torch.randn(heads * 128, device=dev, generator=g)
    ang = torch.randn(S, 64, device=dev, generator=g)
    x.view(S, heads, 128)[-1, ::2] *= 4
    kw = dict(cos=ang.cos(), sin=ang.sin(), rope_pairs=pairs)
    y = x.clone()
    kmax = pkg.attention_ops.qk_rmsnorm_rope_(y, gamma, want_max=True, **kw)
    pkg.attention_ops.qk_rmsnorm_rope_(x, gamma, **kw)
    assert torch.equal(x, y)
    ref = y.double().view(S, heads, 128).norm(dim=-1).amax(0)
    # fp32 sums of 128 squares, every partial sum rounded up or down by at most 2^-24 of itself
    assert bool(((kmax.double() - ref).abs() <= 128 * 2.0**-24 * ref).all())


@pytest.mark.parametrize("S,heads", [(1, 4), (640, 40), (641, 40), (25000, 40), (25008, 40)])
def test_key_norm_maximum_alone_of_every_workgroup_size(pkg, dev, S, heads):
    g = torch.Generator(device=dev).manual_seed(S)
    k = torch.randn(S, heads, 128, device=dev, generator=g).to(torch.bfloat16)
    k[-1, ::2] *= 4
    k[0, 1::2] *= 4
    ref = k.double().norm(dim=-1).amax(0)
    # fp32 sums of 128 squares, every partial sum rounded up or down by at most 2^-24 of itself
    assert bool(((pkg.attention_ops.head_max_norm(k).double() - ref).abs() <= 128 * 2.0**-24 * ref).all())
