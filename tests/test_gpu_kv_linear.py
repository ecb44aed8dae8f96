"""K and V of one activation from two weights against a plain product and the transposing pass, bit for
bit, whichever tile and number of launches the token count takes (one launch of 128 x 256 or 128 x 128
tiles, two launches, the unpipelined kernel for K = 384), with and without the row recipe's scales."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1, 512, 512), (64, 5120, 512), (129, 5120, 1024), (512, 5120, 1024), (700, 1024, 512),
                                   (2049, 5120, 512), (300, 512, 384)])
@pytest.mark.parametrize("recipe", ["mx", "row"])
def test_kv_linear(pkg, dev, M, N, K, recipe):
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    rnd = lambda *s: torch.randn(*s, device=dev, generator=g)  # noqa: E731
    x = pkg.adaln_modulate(rnd(M, K).to(torch.bfloat16), eps=0.0, norm_type="none", quant=recipe)
    w = [pkg.quantize_weight_mx((rnd(K, N) * 0.02).to(torch.bfloat16), rnd(N) * 0.1) for _ in range(2)]
    if recipe == "row":
        w = [p._replace(col_scale=torch.rand(N, device=dev, generator=g) + 0.5) for p in w]
    k, vt = pkg.mxfp8_kv_linear(x, *w)
    assert torch.equal(k, pkg.mxfp8_linear(x, w[0]))
    ref, _ = pkg.attention_ops.transpose_heads(pkg.mxfp8_linear(x, w[1]).view(M, N // 128, 128))
    assert torch.equal(vt, ref)


def test_kv_linear_without_tokens(pkg, dev):
    w = pkg.quantize_weight_mx(torch.ones(512, 256, dtype=torch.bfloat16, device=dev))
    x = pkg.adaln_modulate(torch.empty(0, 512, dtype=torch.bfloat16, device=dev), eps=0.0, norm_type="none", quant="mx")
    k, vt = pkg.mxfp8_kv_linear(x, w, w)
    assert k.shape == (0, 256) and vt.shape == (2, 128, 64) and not bool(vt.any())
    with pytest.raises(ValueError):
        pkg.mxfp8_kv_linear(x, w, pkg.quantize_weight_mx(torch.ones(512, 512, dtype=torch.bfloat16, device=dev)))
