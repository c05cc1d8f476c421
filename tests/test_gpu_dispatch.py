"""Which kernel a call launches, where two of them give the same bits or
nearly so and only time tells them apart."""

import pytest

pytestmark = pytest.mark.gpu


def _linear(dev, m, k, n, *, quantized=False, offset=0):
    """fp8_linear as a call without arguments; prequantized codes start
    ``offset`` bytes off 16-byte alignment."""
    import torch
    from akas_amd import ops

    w = torch.ones((n, k), dtype=torch.uint8, device=dev)
    s = torch.ones(((n + 127) // 128, k // 128), dtype=torch.float32, device=dev)
    if not quantized:
        x = torch.ones((m, k), dtype=torch.bfloat16, device=dev)
        return lambda: ops.fp8_linear(x, w, s)
    x = torch.ones(m * k + offset, dtype=torch.uint8, device=dev)[offset:].view(m, k)
    a = torch.ones((m, k // 128), dtype=torch.float32, device=dev)
    return lambda: ops.fp8_linear(x, w, s, activation_scales=a)


# Products past 128 k-blocks, and codes off alignment, on register-staged tiles.
@pytest.mark.parametrize("m,k,n,offset,kernel", [
    (65, 16512, 64, 0, "dense_tiled_kernel<64, 64,"),
    (256, 16512, 192, 0, "dense_tiled_kernel<64, 64,"),
    (257, 16512, 128, 0, "dense_tiled_kernel<128, 128,"),
    (20, 16512, 272, 0, "dense_small_kernel<2,"),
    (64, 16512, 272, 0, "dense_small_kernel<4,"),
    (20, 2176, 512, 8, "dense_wide_kernel<2,"),
    (50, 1152, 512, 8, "dense_wide_kernel<4,"),
    (20, 640, 512, 8, "dense_small_kernel<2,"),
    (20, 640, 6144, 8, "dense_small_kernel<2,"),
    (20, 1536, 6144, 8, "dense_wide_kernel<2,"),
    (100, 640, 512, 8, "dense_tiled_kernel<64, 64,"),
    (300, 640, 512, 8, "dense_tiled_kernel<128, 128,"),
    (8192, 256, 2048, 8, "dense_tiled_kernel<256, 128,"),
    (300, 640, 528, 8, "dense_small_kernel<4,"),
    # the same sizes on aligned codes
    (100, 640, 512, 0, "dense_pipe_kernel<"),
    (8192, 256, 2048, 0, "dense_dma_kernel<"),
])
def test_staged_kernels(dev, launched, m, k, n, offset, kernel):
    names = launched(_linear(dev, m, k, n, quantized=True, offset=offset))
    assert names and all(name.startswith(kernel) for name in names), names
