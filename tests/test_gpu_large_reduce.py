"""Reduced gradients of more windows of sorted positions than one launch has
threads for: two tables of eight positions a window (dims past 128, and off the
vector grid), 68 million references each.  Sums of 16 small whole numbers are
exact in any order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_reduce_past_a_launch(torch_gpu, pkg):
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    dims, rows, repeats = (132, 3), 4_250_000, 16
    n = rows * repeats
    assert 2 * n // 8 * 256 > 1 << 32
    print(f"case: dims={dims} references={n} each", flush=True)
    shard = H.DeviceShard(torch, [W.TableSpec(i, d, rows) for i, d in enumerate(dims)], max_occurrences=2 * n)
    none, feats = np.zeros(0, np.uint64), []
    for i, d in enumerate(dims):
        f = H.DeviceFeature(torch, W.Feature(i, i, W.SUM, none, none, none))
        f.occurrences, f.bags, f.rows = n, 1, 1
        f.indices = torch.arange(rows, device="cuda").flip(0).repeat(repeats)
        f.offsets = torch.tensor([0, n], device="cuda")
        f.gradient = torch.arange(1, d + 1, dtype=torch.float32, device="cuda").view(1, d)
        feats.append(f)
    slots, tables, occurrences, count = shard.unique(feats)
    assert int(count.item()) == 2 * rows
    values = shard.reduce(feats, occurrences, 2 * rows)
    torch.cuda.synchronize()
    assert torch.equal(values[:rows], (feats[0].gradient * repeats).expand(rows, -1))
    assert torch.equal(values[rows:, :3], (feats[1].gradient * repeats).expand(rows, -1))
    assert not values[rows:, 3:].any()
