"""Route tables at the sizes where the chunked scan can go wrong: entry
counts at and around its chunks, several passes per chunk, rows that straddle
threads, inactive rows, ids outside the experts and ids off 16-byte
alignment.  Bit-exact against the oracle (src/akas/ops/moe/kernel.py:121-151)."""

import numpy as np
import pytest

from oracle import moe as omoe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,top,experts", [
    (1, 1, 3), (341, 3, 7), (1023, 4, 64), (1024, 4, 64), (1025, 4, 64), (1366, 3, 16),
    (4095, 4, 64), (4096, 4, 64), (4097, 4, 64), (8193, 2, 32), (2049, 8, 256), (513, 33, 40),
    (52431, 5, 8), (65537, 4, 4),
    # one chunk of several passes (256 experts and more), one rank over many
    # chunks, ranks in fours over two and four chunks
    (5000, 4, 257), (3001, 8, 256), (20001, 1, 8), (9000, 8, 128), (17001, 12, 64),
    # four ranks, rows in fours: routes4_kernel's first and last sizes (one
    # pass, and several with more experts than CUs), and those beside them
    (2500, 4, 64), (2504, 4, 64), (4092, 4, 16), (4100, 4, 64), (9004, 4, 300)])
@pytest.mark.parametrize("shift", [0, 1])
def test_routes_around_chunks(dev, rows, top, experts, shift):
    import torch
    from akas_amd import ops

    rng = np.random.default_rng(rows + top + shift)
    ids = np.argsort(rng.random((rows, experts)), axis=1)[:, :top].astype(np.int32)
    ids[rng.random(rows) < 0.02] = experts + 1  # a row that routes nowhere
    ids[rng.random(rows) < 0.02, 0] = -1
    active = (rng.random(rows) > 0.1).astype(np.int32)
    buf = torch.full((rows * top + 8,), -1, dtype=torch.int32, device=dev)
    tid = buf[shift:shift + rows * top].view(rows, top)
    tid.copy_(torch.from_numpy(ids))
    counts, routes = ops.quantized_routes(tid, torch.from_numpy(active).to(dev), experts=experts)
    want_counts, want_routes = omoe.quantized_routes(ids, active, experts)
    np.testing.assert_array_equal(counts.cpu().numpy(), want_counts)
    np.testing.assert_array_equal(routes.cpu().numpy(), want_routes)


@pytest.mark.parametrize("rows,top,experts", [(4, 33, 40), (5001, 2, 8), (2050, 4, 16),
                                              (9001, 8, 300), (1700, 5, 4)])
def test_routes_without_flags(dev, rows, top, experts):
    """A null activity table means every row: the tables of the one-call
    gate/up kind on batches past its own scan, against the oracle."""
    import torch
    from akas_amd import ops

    rng = np.random.default_rng(rows)
    top = min(top, experts)
    ids = np.argsort(rng.random((rows, experts)), axis=1)[:, :top].astype(np.int32)
    ids[rng.random(rows) < 0.02] = experts + 1
    x = torch.ones((rows, 128), dtype=torch.uint8, device=dev)
    xs = torch.ones((rows, 1), dtype=torch.float32, device=dev)
    w = torch.ones((experts, 128, 128), dtype=torch.uint8, device=dev)
    ws = torch.ones((experts, 1, 1), dtype=torch.float32, device=dev)
    counts, routes, _, _ = ops.routed_fp8_expert_swiglu(torch.from_numpy(ids).to(dev), None, x, xs,
                                                        w, ws, w, ws)
    want_counts, want_routes = omoe.quantized_routes(ids, np.ones(rows, np.int32), experts)
    np.testing.assert_array_equal(counts.cpu().numpy(), want_counts)
    np.testing.assert_array_equal(routes.cpu().numpy(), want_routes)


def test_routes_past_grid_y(dev):
    """More experts than the y or z extent of a launch grid takes."""
    import torch
    from akas_amd import ops

    experts, rows, top = 70001, 5, 3
    rng = np.random.default_rng(3)
    ids = rng.permutation(experts)[:rows * top].astype(np.int32).reshape(rows, top)
    ids[0, 0], ids[4, 2] = experts - 1, 65536
    active = np.array([1, 1, 0, 1, 1], np.int32)
    counts, routes = ops.quantized_routes(torch.from_numpy(ids).to(dev),
                                          torch.from_numpy(active).to(dev), experts=experts)
    want_counts, want_routes = omoe.quantized_routes(ids, active, experts)
    np.testing.assert_array_equal(counts.cpu().numpy(), want_counts)
    np.testing.assert_array_equal(routes.cpu().numpy(), want_routes)
