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


# Prefill tiles past one round of 256x256 ones: those, unless their last round
# is nearly empty.
@pytest.mark.parametrize("m,k,n,kernel", [
    (8192, 1024, 8192, "dense_dma_kernel<"),
    (4100, 768, 6144, "dense_dma_kernel<"),
    (7000, 2048, 3072, "dense_dma_kernel<"),
    (4096, 512, 4096, "dense_dma_kernel<"),  # one full round
    (4100, 512, 4096, "dense_pipe_kernel<"),  # 16 tiles over
    (3000, 1024, 6144, "dense_pipe_kernel<"),  # 32 over
    (5571, 768, 6144, "dense_pipe_kernel<"),  # two rounds and 16
    (5571, 1536, 6144, "dense_dma_kernel<"),
    # below a round, ragged
    (2000, 512, 7808, "dense_dma_kernel<"), (1537, 384, 9088, "dense_dma_kernel<"),
    (4097, 256, 3840, "dense_dma_kernel<"), (2304, 1024, 6784, "dense_dma_kernel<"),
])
def test_prefill_tiles(dev, launched, m, k, n, kernel):
    names = launched(_linear(dev, m, k, n, quantized=True))
    assert len(names) == 1 and names[0].startswith(kernel), names


# Between decode and prefill: the tiles of the pipelined engine, and what comes
# before it.
@pytest.mark.parametrize("m,k,n,kernel", [
    (17, 128, 512, "dense_small_kernel<2,"),
    (33, 256, 528, "dense_small_kernel<4,"),
    (17, 1152, 4128, "dense_wide_kernel<2,"),
    (32, 1920, 6144, "dense_wide_kernel<2,"),
    (20, 1920, 1536, "dense_wide_kernel<2,"),
    (20, 1536, 1536, "dense_small_kernel<2,"),
    (32, 4864, 3072, "dense_wide_kernel<2,"),
    (32, 4992, 3072, "dense_pipe_kernel<"),  # past its slab
    (65, 128, 512, "dense_pipe_kernel<pipe::Engine<64, 64,"),
    (127, 384, 1040, "dense_pipe_kernel<pipe::Engine<64, 64,"),
    (300, 2048, 6144, "dense_pipe_kernel<pipe::Engine<64, 128,"),
    (513, 1408, 6000, "dense_pipe_kernel<pipe::Engine<128, 128, 2, 2, 2,"),
    (1290, 2048, 2000, "dense_pipe_kernel<pipe::Engine<128, 128, 2, 2, 2,"),
    (1100, 768, 5008, "dense_pipe_kernel<pipe::Engine<128, 128, 2, 2, 1,"),
])
def test_mid_size_tiles(dev, launched, m, k, n, kernel):
    names = launched(_linear(dev, m, k, n, quantized=True))
    assert len(names) == 1 and names[0].startswith(kernel), names


# fp8_linear past 2048 deep: 2048-deep partitions on the split kernel or the
# pipelined engine, then the merge; up to 16 rows the fused kernel, or the
# quantizer and the product.
@pytest.mark.parametrize("m,k,n,kernels", [
    (64, 8192, 2048, ("quantize", "dense_split", "merge")),
    (100, 18432, 2048, ("quantize", "dense_split", "merge")),
    (200, 8192, 2048, ("quantize", "dense_pipe", "merge")),
    (64, 8192, 4096, ("quantize", "dense_pipe", "merge")),
    (256, 4096, 8192, ("quantize", "dense_pipe", "merge")),
    (1, 8192, 2048, ("dense_wide",)),
    (8, 2688, 2048, ("dense_wide",)),
    (16, 2560, 6144, ("dense_wide",)),
    (8, 8192, 2048, ("quantize", "dense_wide")),
    (16, 4096, 6144, ("quantize", "dense_wide")),
])
def test_deep_linear_kernels(dev, launched, m, k, n, kernels):
    names = launched(_linear(dev, m, k, n))
    assert len(names) == len(kernels), names
    assert all(name.startswith(kernel + "_kernel") for name, kernel in zip(names, kernels)), names


def _experts(dev, t, h, f, experts, top, *, offset=0):
    """The gate/up and down products of a routed batch, as calls without
    arguments; codes start ``offset`` bytes off 16-byte alignment."""
    import torch
    from akas_amd import ops

    def codes(*shape):
        n = int(torch.Size(shape).numel())
        return torch.ones(n + offset, dtype=torch.uint8, device=dev)[offset:].view(shape)

    def scales(*shape):
        return torch.ones(shape, dtype=torch.float32, device=dev)

    ids = (torch.arange(t * top, device=dev, dtype=torch.int32) % experts).view(t, top)
    counts, routes = ops.quantized_routes(ids, torch.ones(t, dtype=torch.int32, device=dev),
                                          experts=experts)
    up, us = codes(experts, f, h), scales(experts, f // 128, h // 128)
    down, ds = codes(experts, h, f), scales(experts, h // 128, f // 128)
    x, xs = codes(t, h), scales(t, h // 128)
    act, acs = codes(t, top, f), scales(t, top, f // 128)
    kw = dict(r=t, top=top)
    return (lambda: ops.fp8_expert_swiglu(x, xs, up, us, up, us, counts, routes, **kw),
            lambda **kv: ops.expert_partial(act, acs, down, ds, counts, routes, routed_input=True,
                                            **kw, **kv))


# Decode kernels that may take the non-temporal hint end in "true": only where
# the launch's weights can pass the last-level cache.
@pytest.mark.parametrize("t,h,f,experts,top,up,down", [
    (256, 2048, 1536, 64, 4, True, False),  # 403 and 201 MB
    (16, 2048, 1536, 64, 4, True, False),
    (10, 2048, 1536, 64, 4, False, False),  # 40 routes reach at most 252 MB
    (256, 1536, 768, 48, 2, False, False),  # 113 and 57 MB
    (400, 2048, 512, 129, 4, False, False),  # 258 MB
])
def test_hint_needs_more_than_the_cache(dev, launched, t, h, f, experts, top, up, down):
    for call, hint in zip(_experts(dev, t, h, f, experts, top), (up, down)):
        names = launched(call)
        assert len(names) == 1 and names[0].startswith("expert_tiled_kernel<"), names
        assert names[0].endswith("true>" if hint else "false>"), names


# Row tiles of the expert products at the means where the choice turns.
@pytest.mark.parametrize("mean,h,f,experts,up,down,down_f32", [
    (104, 512, 2048, 64, "dma", "pipe", "pipe"),
    (114, 2048, 1536, 64, "dma", "dma", "pipe"),
    (128, 2048, 512, 64, "dma", "dma", "dma"),
    (120, 1024, 512, 32, "pipe", "pipe", "pipe"),  # few 256-row tiles
    (128, 1024, 512, 32, "pipe", "dma", "dma"),  # one round however they fall
    (187, 1024, 512, 32, "dma", "dma", "dma"),
    (240, 1024, 512, 8, "pipe", "dma", "dma"),
    (242, 1024, 512, 8, "dma", "dma", "dma"),
    (40, 1536, 768, 64, "tiled", "pipe", "pipe"),
    (47, 1536, 768, 64, "tiled", "tiled", "tiled"),  # 768 tiles of 64 rows fill the CUs
    (49, 1536, 768, 64, "pipe", "pipe", "pipe"),
])
def test_expert_row_tiles(dev, launched, mean, h, f, experts, up, down, down_f32):
    import torch

    gate_up, product = _experts(dev, mean * experts // 4, h, f, experts, 4)
    half = lambda: product(output_dtype=torch.bfloat16)  # noqa: E731
    for call, kernel in ((gate_up, up), (half, down), (product, down_f32)):
        names = launched(call)
        assert len(names) == 1 and names[0].startswith(f"expert_{kernel}_kernel<"), names


@pytest.mark.parametrize("mean,f,experts,kernel", [
    (104, 1536, 64, "tiled"), (119, 768, 64, "tiled"), (120, 768, 64, "dma"),
    (127, 512, 32, "tiled"), (128, 512, 32, "dma")])
def test_pair_partial_row_tiles(dev, launched, mean, f, experts, kernel):
    import torch
    from akas_amd import ops

    t, h, top = mean * experts // 4, 1024, 4
    ids = (torch.arange(t * top, device=dev, dtype=torch.int32) % experts).view(t, top)
    counts, routes = ops.quantized_routes(ids, torch.ones(t, dtype=torch.int32, device=dev),
                                          experts=experts)
    w = torch.ones((experts, f, h), dtype=torch.uint8, device=dev)
    s = torch.ones((experts, f // 128, h // 128), dtype=torch.float32, device=dev)
    x = torch.ones((t, h), dtype=torch.uint8, device=dev)
    xs = torch.ones((t, h // 128), dtype=torch.float32, device=dev)
    names = launched(lambda: ops.expert_pair_partial(x, xs, w, s, w, s, counts, routes, r=t, top=top))
    assert len(names) == 1 and names[0].startswith(f"expert_{kernel}_kernel<"), names


@pytest.mark.parametrize("t,kernel", [(1599, "pipe"), (1600, "dma")])
def test_shared_block_row_tiles(dev, launched, t, kernel):
    """The mean that chooses the gate/up tiles is that of the routed experts
    (100 at 1600 rows x 4 over 64), without the shared one's rows."""
    import torch
    from akas_amd import moe

    experts, h, f = 64, 1024, 512

    def weights(*lead):
        def one(n, k):
            return (torch.ones((*lead, n, k), dtype=torch.uint8, device=dev),
                    torch.ones((*lead, n // 128, k // 128), dtype=torch.float32, device=dev))
        return *one(f, h), *one(f, h), *one(h, f)

    x = torch.ones((t, h), dtype=torch.bfloat16, device=dev)
    logits = torch.randn((t, experts), device=dev)
    gate = torch.ones(t, dtype=torch.bfloat16, device=dev)
    bank, shared = moe.ExpertWeights(*weights(experts)), moe.SharedExpert(*weights())
    names = launched(lambda: moe.shared_expert_moe(x, logits, gate, bank, shared, top=4))
    products = [name for name in names if name.startswith("expert_")]
    assert len(products) == 2, names
    assert products[0].startswith(f"expert_{kernel}_kernel<"), names


@pytest.mark.parametrize("offset", [0, 8])
@pytest.mark.parametrize("mean", [56, 110, 300])
def test_expert_codes_off_alignment(dev, launched, mean, offset):
    """Neither DMA engine takes codes off 16-byte alignment."""
    for call in _experts(dev, mean * 16 // 4, 256, 256, 16, 4, offset=offset):
        names = launched(call)
        assert len(names) == 1, names
        assert names[0].startswith("expert_tiled_kernel<") == (offset != 0), names
