"""Pooled gathers at the edges of the load widths (4, 2 or 1 floats, by the
dimension and the buffers' alignment), of rows wider than a wavefront's
columns, of sequence copies and of bags past what a block stages at a time,
bit-exact against the oracle (sums are taken in occurrence order)."""
import numpy as np
import pytest

from parity import assert_close, oracle_store
from test_gpu_pull import expected, random_feature

pytestmark = pytest.mark.gpu


def check(torch, W, H, dim, pooling, rng, offset=0, **bags):
    spec = W.TableSpec(5, dim, 700, seed=77 + dim)
    f = random_feature(W, rng, spec, pooling, **bags)
    print(f"case: dim={dim} pooling={pooling} offset={offset} occurrences={len(f.keys)}", flush=True)
    shard = H.DeviceShard(torch, [spec])
    shard.init_rows()
    rows = len(f.keys) if pooling == 2 else len(f.valid_lengths)
    flat = torch.full((rows * dim + offset + 3,), -7.0, device="cuda")
    out = flat[offset: offset + rows * dim].view(rows, dim)
    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    shard.lookup([H.DeviceFeature(torch, f)], [out], status=status)
    torch.cuda.synchronize()
    assert int(status.item()) == 0
    assert (flat[:offset] == -7).all() and (flat[offset + rows * dim:] == -7).all(), "a value outside the output"
    assert_close(out.cpu().numpy(), expected(oracle_store(spec), f, dim), f"gather dim={dim}", strict_ulp=0)


@pytest.mark.parametrize("dim", [1, 2, 3, 4, 5, 6, 10, 50, 62, 64, 66, 126, 130, 254, 256, 258, 260, 300, 1028])
@pytest.mark.parametrize("pooling", [0, 1, 2, 3])
def test_widths(torch_gpu, pkg, dim, pooling):
    check(torch_gpu, pkg.workloads, pkg.eps_hip, dim, pooling, np.random.default_rng(dim * 4 + pooling), bags=130)


@pytest.mark.parametrize("dim,offset", [(64, 1), (64, 2), (64, 3), (256, 2), (260, 2), (6, 1)])
@pytest.mark.parametrize("pooling", [1, 2])
def test_output_alignment(torch_gpu, pkg, dim, offset, pooling):
    check(torch_gpu, pkg.workloads, pkg.eps_hip, dim, pooling, np.random.default_rng(dim + offset), offset=offset, bags=70)


@pytest.mark.parametrize("dim", [3, 4, 10, 64, 300])
@pytest.mark.parametrize("pooling", [0, 1, 3])
def test_bags_past_the_stage(torch_gpu, pkg, dim, pooling):
    """Blocks of 4 to 64 bags with up to 40,000 occurrences between them."""
    check(torch_gpu, pkg.workloads, pkg.eps_hip, dim, pooling, np.random.default_rng(dim * 7 + pooling), bags=67,
          max_len=1200)
