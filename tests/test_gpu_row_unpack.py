"""Packed rows taken apart in one pass: every byte where the GEMM reads it, whatever the rows' base and stride."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# widths: one block of 32, an odd number of blocks, more than one pass of 4 KiB, the model's; rows: a
# partial workgroup, one row, none
@pytest.mark.parametrize("T,K", [(5, 32), (1, 96), (7, 4128), (130, 5120), (9, 13824), (0, 64)])
# (first byte, bytes between rows): whole rows, rows of a wider buffer, off the 4-byte boundary
@pytest.mark.parametrize("first,extra", [(0, 0), (16, 28), (1, 0), (0, 3)])
def test_row_unpack_bytes(pkg, dev, T, K, first, extra):
    from vllm_omni_neuron_amd import row_mx_kernels as rm

    g = torch.Generator(device=dev).manual_seed(K + T)
    buf = torch.randint(0, 256, (T * (K + 4 + extra) + first + 64,), dtype=torch.uint8, device=dev, generator=g)
    packed = torch.as_strided(buf, (T, K + 4), (K + 4 + extra, 1), first).view(torch.float8_e4m3fn)
    codes, scales, row_scale = rm._split_row_packed(packed)
    raw = packed.view(torch.uint8)
    assert torch.equal(codes, raw[:, :K]) and codes.is_contiguous()
    assert torch.equal(row_scale.view(torch.uint8).view(T, 4), raw[:, K:])
    assert scales.shape == (T, K // 32) and bool((scales == 127).all())
