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
    (52431, 5, 8), (65537, 4, 4)])
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
