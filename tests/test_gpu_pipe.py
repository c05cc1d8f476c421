"""GPU parity of the dense product between decode and prefill sizes, where
the pipelined tile engine runs, at the sizes where its tiling can go wrong:
row and column remainders of every tile, k-block counts below, at and past
its stages and groups, partitions, its k-block limit, and operands off the
alignment its copies and stores take.  Checked against the oracle's float64
equation (src/akas/ops/linear/validation.py:206-230)."""

import numpy as np
import pytest

from oracle import fp8 as ofp8

pytestmark = pytest.mark.gpu

# float32 out: the FP8 matrix instruction's own sum of 128 products is the
# error that remains, 3e-5 of the result in norm over every kernel here.
F32_TOL = 1e-4


def _rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)


def _problem(dev, m, k, n, seed, scale_dtype="float32"):
    import torch
    from akas_amd import ops

    rng = np.random.default_rng(seed)
    x = rng.normal(0, 1, (m, k)).astype(np.float32)
    w = rng.normal(0, 0.02, (n, k)).astype(np.float32)
    wc, ws = ops.quantize_weight_blocks(torch.from_numpy(w).to(dev),
                                        scale_dtype=getattr(torch, scale_dtype))
    xt = torch.from_numpy(x).to(dev)
    want = ofp8.fp8_linear(x, wc.cpu().numpy(), ws.float().cpu().numpy())
    return xt, wc, ws, want


@pytest.mark.parametrize("m,k,n", [
    # few rows and k-blocks: the direct small kernel
    (17, 128, 512), (33, 256, 528), (63, 384, 1040),
    # 64x64 tiles in two k-block groups: one row past a tile, one short of
    # it, ragged columns, 1 to 5 and 17 k-blocks (four stages of two)
    (65, 128, 512), (65, 256, 528), (127, 384, 1040), (65, 512, 2000), (127, 640, 2048),
    (257, 2176, 80), (300, 1152, 1008),
    # 64x128 tiles (three stages of two)
    (300, 2048, 6144), (641, 1280, 2064), (999, 896, 2048), (770, 384, 1936),
    # 128x128 tiles, one workgroup per CU in two groups, and two per CU
    (513, 1408, 6000), (1290, 2048, 2000), (1100, 768, 5008), (2049, 1024, 2048),
    # 256x256 tiles below a full round, one and three quarters of the last
    (2049, 512, 6144), (2177, 384, 6144),
    # the largest depth, and the register-staged kernels past it
    (40, 16384, 272), (40, 16512, 272), (100, 16512, 256), (130, 16512, 192),
    (300, 16512, 272),
])
@pytest.mark.parametrize("scale_dtype", ["float32", "bfloat16"])
def test_mid_size_linear(dev, m, k, n, scale_dtype):
    import torch
    from akas_amd import ops

    xt, wc, ws, want = _problem(dev, m, k, n, m + k + n, scale_dtype)
    got = ops.fp8_linear(xt, wc, ws)
    codes, scales = ops.quantize(xt)
    pre = ops.fp8_linear(codes, wc, ws, activation_scales=scales)
    half = ops.fp8_linear(codes, wc, ws, activation_scales=scales, out_dtype=torch.bfloat16)
    assert _rel(got.cpu().numpy(), want) <= F32_TOL
    assert _rel(pre.cpu().numpy(), want) <= F32_TOL
    # one rounding to bf16 (2^-9 of each value at most)
    assert _rel(half.float().cpu().numpy(), want) <= 2.0 ** -8


@pytest.mark.parametrize("m,k,n,parts", [(300, 1536, 1040, 4), (70, 640, 512, 5),
                                         (520, 4096, 2048, 2), (200, 6144, 2048, 3)])
def test_mid_size_partitions(dev, m, k, n, parts):
    from akas_amd import ops

    xt, wc, ws, want = _problem(dev, m, k, n, 7 * m + k)
    codes, scales = ops.quantize(xt)
    partial = ops.projection_partial(codes, scales, wc, ws, partitions=parts)
    assert tuple(partial.shape) == (m, parts, n)
    merged = ops.projection_merge(partial)
    assert _rel(merged.cpu().numpy(), want) <= F32_TOL
    # every partition is its own slice of k
    step = k // parts
    for p in (0, parts - 1):
        cut = slice(p * step, (p + 1) * step)
        part = ofp8.fp8_linear(xt[:, cut].cpu().numpy(), wc[:, cut].cpu().numpy(),
                               ws[:, p * step // 128:(p + 1) * step // 128].cpu().numpy())
        assert _rel(partial[:, p].cpu().numpy(), part) <= F32_TOL


@pytest.mark.parametrize("out_dtype", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("m,n", [(300, 1040), (130, 512), (17, 512), (50, 544), (65, 576),
                                 (300, 384), (4097, 4096)])
def test_mid_size_unaligned_operands(dev, m, n, out_dtype):
    """An output off 16-byte alignment takes element stores, codes off it the
    register-staged kernels; neither writes outside its rows."""
    import torch
    from akas_amd import ops

    k = 640
    xt, wc, ws, want = _problem(dev, m, k, n, 11 * m)
    codes, scales = ops.quantize(xt)
    dt = getattr(torch, out_dtype)
    tol = {"float32": F32_TOL, "bfloat16": 2.0 ** -8, "float16": 2.0 ** -11 + F32_TOL}[out_dtype]
    buf = torch.full((m * n + 16,), 7.0, dtype=dt, device=dev)
    out = buf[1:1 + m * n].view(m, n)
    ops.fp8_linear(codes, wc, ws, activation_scales=scales, out=out)
    assert _rel(out.float().cpu().numpy(), want) <= tol
    assert float(buf[0]) == 7.0 and bool((buf[1 + m * n:] == 7.0).all())
    raw = torch.empty(m * k + 8, dtype=torch.uint8, device=dev)
    shifted = raw[8:].view(m, k)
    shifted.copy_(codes)
    got = ops.fp8_linear(shifted, wc, ws, activation_scales=scales, out_dtype=dt)
    assert _rel(got.float().cpu().numpy(), want) <= tol


@pytest.mark.parametrize("m,k,n", [(17, 1152, 4128), (24, 1536, 6144), (25, 1920, 4128),
                                   (32, 1152, 6144), (20, 1920, 544), (32, 4864, 96)])
@pytest.mark.parametrize("scale_dtype", ["float32", "bfloat16"])
def test_wide_rows_exact_products(dev, m, k, n, scale_dtype):
    """17 to 32 rows of 9 to 38 k-blocks on the wide kernel, codes on and off
    16-byte alignment: exact products with binary scales, so the output equals
    the float64 oracle bit for bit."""
    import torch
    from akas_amd import ops
    from golden_inputs import exact_codes

    rng = np.random.default_rng(m + k + n)
    x, w = exact_codes(rng, (m, k)), exact_codes(rng, (n, k))
    xs = (2.0 ** rng.integers(-4, 2, (m, k // 128))).astype(np.float32)
    ws = (2.0 ** rng.integers(-4, 2, ((n + 127) // 128, k // 128))).astype(np.float32)
    want = ofp8.fp8_linear(x, w, ws, activation_scales=xs)
    wt, xst = torch.from_numpy(w).to(dev), torch.from_numpy(xs).to(dev)
    wst = torch.from_numpy(ws).to(dev).to(getattr(torch, scale_dtype))
    for offset in (0, 8):
        raw = torch.empty(m * k + offset, dtype=torch.uint8, device=dev)
        xt = raw[offset:].view(m, k)
        xt.copy_(torch.from_numpy(x))
        got = ops.fp8_linear(xt, wt, wst, activation_scales=xst)
        np.testing.assert_array_equal(got.cpu().numpy(), want)
