"""The MXFP8 GEMM's tile sizes against each other, bit for bit.

The tile (256, 192 or 128 tokens by 256 features, or 128 by 128) follows from the number of tokens;
every output element is the same sequence of MFMAs on the same operands with any of them. A call on
the first M rows of a long activation must therefore return the first M rows of the call on all of it
(the 256 x 256 tile: 16380 tokens fill whole rounds of it), whatever tile M takes. The long call itself
is held to the fp64 product elsewhere (test_gpu_gemm, test_gpu_gemm_full). M covers a few rows, tile edges
and remainders of every tile, waves without any token, and both sides of the QKV launch's split."""

import pytest
import torch

pytestmark = pytest.mark.gpu

LONG, D, K = 16380, 5120, 512
ROWS = [2, 31, 128, 129, 385, 768, 1000, 1024, 1025, 1560, 2113, 3120, 3137, 4100, 5500]


@pytest.fixture(scope="module", params=["mx", "row"])
def operands(request, pkg, dev):
    """Codes of N(0, 1) rows, as MX blocks or with one scale per row and per output channel."""
    g = torch.Generator(device=dev).manual_seed(41)
    x = torch.randn(LONG, K, device=dev, generator=g).to(torch.bfloat16)
    a = pkg.adaln_modulate(x, eps=0.0, norm_type="none", quant=request.param)
    w = pkg.quantize_weight_mx((torch.randn(K, 3 * D, device=dev, generator=g) * 0.02).to(torch.bfloat16),
                               torch.randn(3 * D, device=dev, generator=g) * 0.1)
    if request.param == "row":
        w = w._replace(col_scale=torch.rand(3 * D, device=dev, generator=g) + 0.5)
    res = torch.randn(LONG, D, device=dev, generator=g).to(torch.bfloat16)
    return a, w, res, torch.randn(D, device=dev, generator=g)


def _first(a, rows):
    return a[:rows] if isinstance(a, torch.Tensor) else type(a)(a.codes[:rows], a.scales[:rows])


def _cols(w, n):
    part = lambda t: None if t is None else t[:n]  # noqa: E731
    return w._replace(codes=w.codes[:n], scales=w.scales[:n], col_scale=part(w.col_scale), bias=part(w.bias))


def _bits(t):
    return t.view(torch.int16) if t.dtype == torch.bfloat16 else t.view(torch.uint8)


@pytest.mark.parametrize("epilogue", ["bf16", "gelu_mx", "gelu_bf16", "gated_residual"])
def test_tiles_give_the_same_bits(pkg, dev, operands, epilogue):
    a, w, res, gate = operands
    w = _cols(w, D)

    def call(m):
        kw, ss = {}, None
        if epilogue == "gated_residual":
            kw = {"residual": res[:m], "gate": gate}
        elif epilogue == "bf16":
            ss = torch.full((m, D // 128), -1.0, device=dev)
            kw = {"row_sumsq": ss, "sumsq_cols": D // 2}
        y = pkg.mxfp8_linear(_first(a, m), w, epilogue=epilogue, **kw)
        return (*y,) if isinstance(y, tuple) else (y,) if ss is None else (y, ss)

    ref = call(LONG)
    for m in ROWS:
        for got, want in zip(call(m), ref):
            assert torch.equal(_bits(got), _bits(want[:m])), (epilogue, m)


def test_qkv_tiles_give_the_same_bits(pkg, dev, operands):
    a, w, _, _ = operands

    def call(m):
        ss = torch.full((m, 2 * D // 128), -1.0, device=dev)
        return (*pkg.mxfp8_qkv_linear(_first(a, m), w, vt_col0=2 * D, row_sumsq=ss, sumsq_cols=D), ss)

    qk_ref, vt_ref, ss_ref = call(LONG)
    for m in ROWS:
        qk, vt, ss = call(m)
        assert torch.equal(_bits(qk), _bits(qk_ref[:m])) and torch.equal(ss, ss_ref[:m]), m
        pad = vt.shape[-1]
        slot = torch.arange(pad, device=dev)
        key = (slot & ~15) | (slot & 3) | ((slot & 4) << 1) | ((slot & 8) >> 1)
        want = torch.where((key < m), vt_ref[:, :, :pad], torch.zeros((), dtype=vt.dtype, device=dev))
        assert torch.equal(_bits(vt), _bits(want)), m


# V narrower than Q|K / 2 (grouped K/V heads) and wider: the split of the CUs between the parts follows the widths
@pytest.mark.parametrize("M,qk,v", [(2561, 6144, 1024), (2880, 6144, 1024), (3840, 6144, 1024), (2048, 10240, 2560),
                                    (3073, 5120, 256), (4416, 5120, 256), (3000, 1024, 10240)])
def test_qkv_of_any_widths_writes_its_own_outputs_only(pkg, dev, M, qk, v):
    """Q|K, V^T and the partial sums inside larger buffers, against one product per part and the transposing
    pass; what lies around them must stay as it was."""
    K, guard = 512, 1 << 20
    g = torch.Generator(device=dev).manual_seed(M + qk)
    x = torch.randn(M, K, device=dev, generator=g).to(torch.bfloat16)
    a = pkg.adaln_modulate(x, eps=0.0, norm_type="none", quant="mx")
    w = pkg.quantize_weight_mx((torch.randn(K, qk + v, device=dev, generator=g) * 0.02).to(torch.bfloat16),
                               torch.randn(qk + v, device=dev, generator=g) * 0.1)
    ld = (M + 63) // 64 * 64
    sizes = {"qk": M * qk, "vt": v * ld, "ss": M * (qk // 128)}
    bufs = {n: torch.full((k + 2 * guard,), -7.0, dtype=torch.float32 if n == "ss" else torch.bfloat16, device=dev)
            for n, k in sizes.items()}
    own = {n: bufs[n][guard : guard + k] for n, k in sizes.items()}
    ptr, lib = pkg._lib.ptr, pkg._lib.load()
    st = lib.wanmi_mxfp8_gemm_qkv(ptr(a.codes), ptr(a.scales), ptr(w.codes), ptr(w.scales), None, None, ptr(w.bias), M,
                                  qk + v, K, K, ptr(own["qk"]), qk, ptr(own["ss"]), qk, ptr(own["vt"]), qk, ld,
                                  pkg._lib.stream_of(a.codes))
    pkg._lib.check(st, "wanmi_mxfp8_gemm_qkv")
    for n, k in sizes.items():
        assert bool((bufs[n][:guard] == -7.0).all()) and bool((bufs[n][guard + k :] == -7.0).all()), n
    ss = torch.empty(M, qk // 128, device=dev)
    y = pkg.mxfp8_linear(a, _cols(w, qk), row_sumsq=ss, sumsq_cols=qk)
    rest = w._replace(codes=w.codes[qk:], scales=w.scales[qk:], bias=w.bias[qk:])
    vt, _ = pkg.attention_ops.transpose_heads(pkg.mxfp8_linear(a, rest).view(M, v // 128, 128))
    assert torch.equal(own["qk"].view(M, qk), y) and torch.equal(own["ss"].view(M, -1), ss)
    assert torch.equal(own["vt"].view(vt.shape), vt)


@pytest.mark.parametrize("M,N,K", [(3, 256, 512), (100, 512, 1024), (129, 256, 512), (1400, 1024, 512), (3900, 256, 512),
                                   (1000, 5120, 1024), (1560, 5120, 1024)])
def test_fetching_ahead_keeps_the_bits(pkg, dev, M, N, K):
    """Products of fewer tiles than CUs, where idle workgroups fetch the operand panels ahead of the tiles: one or
    several groups of m tiles per XCD, XCDs without a tile, a last tile of one row. The first half of the
    tokens and the rest, each on its own, must give the same rows."""
    g = torch.Generator(device=dev).manual_seed(M + N)
    x = torch.randn(M, K, device=dev, generator=g).to(torch.bfloat16)
    a = pkg.adaln_modulate(x, eps=0.0, norm_type="none", quant="mx")
    w = pkg.quantize_weight_mx((torch.randn(K, N, device=dev, generator=g) * 0.02).to(torch.bfloat16))
    y, h = pkg.mxfp8_linear(a, w), M // 2
    ref = torch.cat([pkg.mxfp8_linear(type(a)(a.codes[i:j], a.scales[i:j]), w) for i, j in ((0, h), (h, M))])
    assert torch.equal(y, ref)
    # and each element within the bound of bf16 rounding and fp32 accumulation of the fp64 product
    v = [t.codes.float().double().reshape(t.codes.shape[0], -1, 32) * torch.exp2(t.scales.double() - 127)[..., None]
         for t in (a, w)]
    p, q = (t.reshape(t.shape[0], K) for t in v)
    bound = 2.0**-8 * (p @ q.T).abs() + 2.0**-14 * (p.abs() @ q.T.abs())
    assert bool(((y.double() - p @ q.T).abs() <= bound).all())
