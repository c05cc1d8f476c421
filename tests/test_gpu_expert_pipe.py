"""Grouped expert products on the pipelined tiles (32 to 111 mean rows per
expert) and the 256-row ones: row tiles full, one over and one short, empty
and one-row experts, k-block counts below and past the stages, packed rows,
both scale dtypes, stores off alignment.  Bit for bit against the same call on a few rows at a
time, which runs on the decode tiles: every (row, column) is one float32
chain in ascending k-block order on any tile, and so is the fused activation
(src/akas/ops/moe/cuda.py:541-1354, :823-946)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bank(torch, g, experts, n, k, dtype, dev):
    codes = torch.randint(0, 256, (experts, n, k), generator=g, device=dev, dtype=torch.uint8)
    codes[(codes & 127) == 127] = 1  # no NaN codes
    scales = torch.rand((experts, n // 128, k // 128), generator=g, device=dev) * 1e-3 + 1e-4
    return codes, scales.to(dtype)


def _routing(torch, sizes, top, dev):
    """ids [r, top] in which expert e takes sizes[e] of the entries: rank by
    rank, so that no row names an expert twice."""
    flat = np.concatenate([np.full(n, e, np.int32) for e, n in enumerate(sizes)])
    r = len(flat) // top
    assert max(sizes) <= r and r * top == len(flat)
    return torch.from_numpy(flat.reshape(top, r).T.copy()).to(dev)


@pytest.mark.parametrize("sizes,h,f", [
    ([64, 65, 63, 1, 0, 128, 71, 8], 384, 256),        # 50 mean rows
    ([127, 128, 129, 2, 40, 60, 61, 93], 1024, 384),   # 80
    ([100, 101, 102, 103, 104, 105, 0, 121], 256, 128),  # 92
    ([192, 64, 1, 63, 66, 62, 32, 32], 1152, 640),     # 64
    # 256-row tiles whose last one holds one to four quarters of rows
    ([320, 321, 384, 385, 448, 449, 512, 513], 256, 384),  # 416
])
@pytest.mark.parametrize("scale_dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("packed", [False, True])
def test_expert_tiles_match_single_experts(dev, sizes, h, f, scale_dtype, packed):
    import torch
    from akas_amd import ops

    experts, top = len(sizes), 2
    g = torch.Generator(device=dev)
    g.manual_seed(sum(sizes) + h)
    sd = getattr(torch, scale_dtype)
    w1, s1 = _bank(torch, g, experts, f, h, sd, dev)
    w3, s3 = _bank(torch, g, experts, f, h, sd, dev)
    w2, s2 = _bank(torch, g, experts, h, f, sd, dev)
    ids = _routing(torch, sizes, top, dev)
    r = ids.shape[0]
    x = torch.randn((r, h), generator=g, device=dev).to(torch.bfloat16)
    codes, scales = ops.quantize(x)
    active = torch.ones(r, dtype=torch.int32, device=dev)
    counts, routes = ops.quantized_routes(ids, active, experts=experts)
    assert counts.tolist() == sizes
    kw = dict(r=r, top=top, product_dtype=torch.bfloat16, activation_dtype=torch.bfloat16)
    xin, sin, offsets = codes, scales, None
    if packed:  # packed input, routed output: the same codes
        xin, sin, offsets = ops.expert_pack(codes, scales, counts, routes, None, None, top=top)
    act, act_scales = ops.fp8_expert_swiglu(xin, sin, w1, s1, w3, s3, counts, routes,
                                            expert_offsets=offsets, packed_input=packed, **kw)
    down = {dt: ops.expert_partial(act, act_scales, w2, s2, counts, routes, r=r, top=top,
                                   routed_input=True, output_dtype=dt)
            for dt in (torch.float32, torch.bfloat16)}
    half = ops.expert_partial(act, act_scales, w2, s2, counts, routes, r=r, top=top,
                              routed_input=True,
                              out=torch.zeros(r * top * h + 1, dtype=torch.bfloat16,
                                              device=dev)[1:].view(r, top, h),
                              output_dtype=torch.bfloat16)
    assert torch.equal(half, down[torch.bfloat16])  # element stores, off alignment
    for part in torch.arange(r, device=dev).split(39):
        # at most 39 rows: the decode tiles
        rows = len(part)
        c, rt = ops.quantized_routes(ids[part], active[part], experts=experts)
        few = dict(kw, r=rows)
        wa, wsc = ops.fp8_expert_swiglu(codes[part], scales[part], w1, s1, w3, s3, c, rt, **few)
        assert torch.equal(act[part], wa) and torch.equal(act_scales[part], wsc)
        for dt, got in down.items():
            want = ops.expert_partial(act[part], act_scales[part], w2, s2, c, rt, r=rows, top=top,
                                      routed_input=True, output_dtype=dt)
            assert torch.equal(got[part], want)
    # against the product itself, whole output
    for e, n in enumerate(sizes):
        if n == 0:
            continue
        mask = ids == e
        a = act[mask].view(torch.float8_e4m3fn).float().double().view(n, f // 128, 128)
        a = (a * act_scales[mask].double()[..., None]).view(n, f)
        w = w2[e].view(torch.float8_e4m3fn).float().double()
        w = w * s2[e].double().repeat_interleave(128, 0).repeat_interleave(128, 1)
        want = a @ w.T
        err = (down[torch.float32][mask].double() - want).norm() / want.norm().clamp_min(1e-30)
        assert float(err) <= 1e-4, (e, n)  # the FP8 instruction's own sums
    assert torch.equal(down[torch.float32].to(torch.bfloat16), down[torch.bfloat16])


@pytest.mark.parametrize("mean", [16, 40, 105, 300])
def test_expert_operands_off_alignment(dev, mean):
    """Codes 8 bytes and FP8 outputs one byte off alignment: the aligned
    call's results, and no byte outside them."""
    import torch
    from akas_amd import ops

    experts, top, h, f = 8, 2, 384, 256
    r = mean * experts // top
    g = torch.Generator(device=dev)
    g.manual_seed(mean)
    w1, s1 = _bank(torch, g, experts, f, h, torch.float32, dev)
    w3, s3 = _bank(torch, g, experts, f, h, torch.float32, dev)
    w2, s2 = _bank(torch, g, experts, h, f, torch.float32, dev)
    ids = torch.rand((r, experts), generator=g, device=dev).topk(top, -1).indices.to(torch.int32)
    codes, scales = ops.quantize(torch.randn((r, h), generator=g, device=dev))
    counts, routes = ops.quantized_routes(ids, torch.ones(r, dtype=torch.int32, device=dev),
                                          experts=experts)

    def off(t, n=8):
        moved = torch.empty(t.numel() + n, dtype=t.dtype, device=dev)[n:].view(t.shape)
        return moved.copy_(t)

    kw = dict(r=r, top=top, product_dtype=torch.bfloat16, activation_dtype=torch.bfloat16)
    act, acs = ops.fp8_expert_swiglu(codes, scales, w1, s1, w3, s3, counts, routes, **kw)
    down = ops.expert_partial(act, acs, w2, s2, counts, routes, r=r, top=top, routed_input=True)
    buf = torch.full((r * top * f + 17,), 99, dtype=torch.uint8, device=dev)
    for x, a, b in ((off(codes), w1, w3), (codes, off(w1), w3), (codes, w1, off(w3)),
                    (codes, w1, w3)):
        buf.fill_(99)
        out = buf[1:1 + act.numel()].view(act.shape)
        ops.fp8_expert_swiglu(x, scales, a, s1, b, s3, counts, routes, out=out, **kw)
        assert torch.equal(out, act)
        assert int(buf[0]) == 99 and bool((buf[1 + act.numel():] == 99).all())
    for x, w in ((off(act), w2), (act, off(w2))):
        assert torch.equal(down, ops.expert_partial(x, acs, w, s2, counts, routes, r=r, top=top,
                                                    routed_input=True))
