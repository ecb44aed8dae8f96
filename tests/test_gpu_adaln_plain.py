"""Quantization alone (no norm, no vectors), bit for bit against the oracle: partial chunks and workgroups, every
register width of the kernel, rows of zeros and of huge values."""

import numpy as np
import pytest
import torch

from oracle import adaln as oracle_adaln

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H", [(1, 32), (7, 96), (33, 544), (5, 2048), (9, 4096), (514, 5120), (6, 8192), (3, 12288),
                                 (64, 13824), (5, 16384)])
@pytest.mark.parametrize("quant", ["mx", "row"])
def test_plain_quantization_bit_exact(pkg, dev, T, H, quant):
    g = torch.Generator().manual_seed(T + H)
    x = torch.randn(T, H, generator=g)
    x[0] *= 1e30
    x[T // 2] = 0.0
    x = x.to(torch.bfloat16)
    out = pkg.adaln_modulate(x.to(dev), eps=0.0, norm_type="none", quant=quant)
    ref = oracle_adaln.adaln_quant(x.float().numpy(), None, None, eps=0.0, norm_type="none", quant=quant)
    if quant == "mx":
        np.testing.assert_array_equal(out.scales.cpu().numpy(), ref["scales"])
        np.testing.assert_array_equal(out.codes.view(torch.uint8).cpu().numpy(), ref["codes"])
    else:
        np.testing.assert_array_equal(out.view(torch.uint8).cpu().numpy(), ref["packed"])
