"""How a launch covers its queries -- blocks of 256, wave jobs behind them, several heads per workgroup --
must not show in the result.

Which one runs follows from the numbers of queries, keys and heads (and the 256 CUs). Rows in whole blocks
are the same operations either way, so they must equal, bit for bit, a call that takes those rows
alone. Rows in wave jobs add the same bf16 products in another order: the fp32 sums of both orders differ
by at most 2 Sk 2^-24 of the sum of magnitudes, i.e. of max|v| after normalization, and their bf16 roundings
by one unit (2^-8). The calls on few rows are held to exact softmax in test_gpu_attention.

Jobs: 24 queries behind 240 blocks over 1, 5 (short-key kernel) and 18 tiles (the first with a wave that has
no keys); 5 queries and 100 (four jobs a head, the last partial) where the heads are no multiple of 8, two
and four waves per job. Head groups over few keys: (10000, 129, 10). Blocks: (300, 512, 40)."""

import numpy as np
import pytest
import torch

from oracle import mx as omx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Sq,Sk,N", [(1560, 20, 40), (1560, 300, 40), (1560, 1100, 40), (1797, 1100, 34), (1797, 1900, 34),
                                     (1124, 1090, 62), (10000, 129, 10), (300, 512, 40)])
@pytest.mark.parametrize("prep", [False, True])
def test_routes_agree(pkg, dev, Sq, Sk, N, prep):
    ops, s = pkg.attention_ops, 128**-0.5
    g = torch.Generator(device=dev).manual_seed(Sq + Sk)
    rnd = lambda *shape: torch.randn(*shape, device=dev, generator=g)  # noqa: E731
    q, k, v = (rnd(n, N, 128).to(torch.bfloat16) for n in (Sq, Sk, Sk))
    vt, _ = ops.transpose_heads(v)
    kmax = ops.head_max_norm(k)
    gamma, ang, rr = 1 + 0.1 * rnd(N * 128), rnd(Sq, 64), 1 + 0.1 * rnd(Sq)
    rope = Sk > 1024  # without a rotation over few keys, as the cross-attention

    def call(lo, hi, mode=ops.OUT_TOKEN):
        qp = None
        if prep:
            cs = (ang[lo:hi].cos(), ang[lo:hi].sin()) if rope else (None, None)
            qp = ops.QPrep(None, gamma, *cs, rr=rr[lo:hi].contiguous())
        return ops.attention_core(q[lo:hi], k, vt, kmax, s, mode, q_prep=qp)

    full, whole = call(0, Sq), Sq // 256 * 256
    assert torch.equal(full[:256], call(0, 256))
    assert torch.equal(full[:whole], call(0, whole))
    tail, ref = full[whole:].double(), call(whole, Sq).double()
    bound = 2.0**-8 * ref.abs() + 2 * Sk * 2.0**-24 * float(v.abs().max())
    assert bool(((tail - ref).abs() <= bound).all())
    # the same rows in the other layouts
    dm = call(0, Sq, ops.OUT_DMAJOR)
    assert torch.equal(dm.permute(2, 0, 1).reshape(Sq, -1), full)
    mx = call(0, Sq, ops.OUT_MX)
    codes, scales = omx.mx_quantize(full[-300:].float().cpu().numpy())
    np.testing.assert_array_equal(mx.codes[-300:].view(torch.uint8).cpu().numpy(), codes)
    np.testing.assert_array_equal(mx.scales[-300:].cpu().numpy(), scales)
    if not prep:  # the row sums are those of the rows' own exps: no row is recomputed
        assert torch.equal(ops.attention_core(q, k, vt, kmax, s, exact=True), full)
