"""fp8_linear of up to 16 rows deeper than 2048: the wide kernel's four- and
eight-slot forms, fused and on prequantized codes, at depths that do not fill
their slots, every column width, and codes off 16-byte alignment.  Bit for
bit: quantizing apart or inside the kernel gives the same result, and the
oracle's float64 equation (src/akas/ops/linear/validation.py:206-230) bounds
it."""

import numpy as np
import pytest

from oracle import fp8 as ofp8

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n", [
    (1, 2176, 512), (2, 2560, 6144), (3, 8192, 2048), (16, 2304, 6144), (15, 2560, 4096),
    (9, 4096, 1040), (8, 4224, 2048), (7, 8064, 272), (16, 8192, 528), (5, 8192, 6144),
    (16, 8832, 256), (16, 9216, 256), (4, 4096, 24 * 16),
    # 32 columns, fused: eight slots filled in part, full and over
    (1, 2176, 8192), (9, 2304, 7680), (5, 9728, 8192),
    # 8 columns, more workgroups than CUs: four slots and two, and on codes quantized apart
    (1, 2176, 3072), (3, 4224, 2320), (12, 2176, 3072), (16, 2304, 3072)])
@pytest.mark.parametrize("scale_dtype", ["float32", "bfloat16"])
def test_deep_rows(dev, m, k, n, scale_dtype):
    import torch
    from akas_amd import ops

    rng = np.random.default_rng(m + k + n)
    x = torch.from_numpy(rng.normal(0, 1, (m, k)).astype(np.float32)).to(dev)
    w = torch.from_numpy(rng.normal(0, 0.02, (n, k)).astype(np.float32)).to(dev)
    wc, ws = ops.quantize_weight_blocks(w, scale_dtype=getattr(torch, scale_dtype))
    got = ops.fp8_linear(x, wc, ws)
    codes, scales = ops.quantize(x)
    pre = ops.fp8_linear(codes, wc, ws, activation_scales=scales)
    # the codes 8 bytes off alignment: staged through registers, the same bits
    shifted = torch.empty(m * k + 8, dtype=torch.uint8, device=dev)[8:].view(m, k)
    shifted.copy_(codes)
    off = ops.fp8_linear(shifted, wc, ws, activation_scales=scales)
    want = ofp8.fp8_linear(x.cpu().numpy(), wc.cpu().numpy(), ws.float().cpu().numpy())
    assert torch.equal(pre, off)
    assert torch.equal(got, pre)
    err = np.linalg.norm(got.cpu().numpy() - want) / np.linalg.norm(want)
    assert err <= 1e-4  # the FP8 matrix instruction's own sums of 128 products
