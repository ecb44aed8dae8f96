"""Q and K normalized and rotated in one launch against the two passes, bit for bit: in place and to the
head-major layout, tables contiguous, as the first halves of rotate-half caches, or on a base and stride
that the kernel cannot read in place, one to eight tokens per wave."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,N", [(1, 4), (130, 8), (2049, 40), (5000, 40), (70, 44)])
@pytest.mark.parametrize("tables", ["none", "pairs", "halves", "odd"])
@pytest.mark.parametrize("pairs", ["interleaved", "halves"])
def test_pair_gives_the_bits_of_two_passes(pkg, dev, S, N, tables, pairs):
    ops, W = pkg.attention_ops, N * 128
    g = torch.Generator(device=dev).manual_seed(S + N)
    x = torch.randn(S, 3 * W, device=dev, generator=g).to(torch.bfloat16)
    gq, gk = (1 + 0.1 * torch.randn(W, device=dev, generator=g) for _ in range(2))
    wide = torch.randn(S, 129 if tables == "odd" else 128, device=dev, generator=g)
    cos, sin = {"none": (None, None), "pairs": (wide[:, :64].cos(), wide[:, :64].sin()),
                "halves": (wide.cos()[:, :64], wide.sin()[:, :64]), "odd": (wide.cos()[:, 1:65], wide.sin()[:, 1:65])}[tables]
    copy = lambda t: None if t is None else t.clone(memory_format=torch.contiguous_format)  # noqa: E731
    kw = dict(cos=copy(cos), sin=copy(sin), eps=1e-6, rope_pairs=pairs)
    ref = x.clone()
    ops.qk_rmsnorm_rope_(ref[:, :W], gq, **kw)
    ops.qk_rmsnorm_rope_(ref[:, W : 2 * W], gk, **kw)
    y = x.clone()
    ops._qk_rmsnorm_rope_pair(y, N, (gq, gk), cos, sin, 1e-6, pairs, None)
    assert torch.equal(y, ref)
    if N <= 40:
        out = torch.empty(3 * N, S, 128, dtype=torch.bfloat16, device=dev)
        ops._qk_rmsnorm_rope_pair(x, N, (gq, gk), cos, sin, 1e-6, pairs, out[: 2 * N])
        assert torch.equal(out[: 2 * N].permute(1, 0, 2).reshape(S, 2 * W), ref[:, : 2 * W])
