"""Rows loaded from pinned host memory, whose launch has a bounded grid: counts
around one pass of that grid (64 blocks of 256 16-byte pieces), ragged last
passes and rows off the vector grid, exact."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 341, 342, 683, 3001])
@pytest.mark.parametrize("dim", [3, 4, 64, 300])
def test_load_rows_from_pinned_memory(torch_gpu, pkg, dim, count):
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    rows = 4001
    print(f"case: dim={dim} count={count}", flush=True)
    gen = torch.Generator().manual_seed(dim * 10_007 + count)
    shard = H.DeviceShard(torch, [W.TableSpec(0, dim, rows, seed=3)])
    shard.init_rows()
    want = shard.state[0].reshape(rows, 3 * dim).cpu().clone()
    slots = torch.randperm(rows, generator=gen)[:count]
    packed = torch.empty(count, 3 * dim, dtype=torch.float32, pin_memory=True)
    packed.copy_(torch.rand(count, 3 * dim, generator=gen))
    packed[count // 2, 3 * dim - 1] = 77.0
    want[slots] = packed
    shard.load_rows(0, slots.cuda(), packed)
    torch.cuda.synchronize()
    assert torch.equal(shard.state[0].reshape(rows, 3 * dim).cpu(), want)
    back = torch.empty_like(packed, pin_memory=True)
    shard.read_rows(0, slots.cuda(), out=back)
    torch.cuda.synchronize()
    assert torch.equal(back, packed)
