"""Row runs of pushes too small to fill the chip, whose windows are shorter than
their rows: rows that span many windows and the cuts between XCDs, and hot rows
among them, bit-exact against the oracle."""
import numpy as np
import pytest

import oracle
from parity import assert_close, oracle_store
from test_gpu_long_rows import feature_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 20, 150, 1500])
@pytest.mark.parametrize("dims", [(8,), (32,), (256,), (4, 64, 128)])
def test_push_small_windows(torch_gpu, pkg, dims, rows):
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    rng = np.random.default_rng(rows * 7 + sum(dims))
    specs = [W.TableSpec(i, d, 2000, seed=11 + i) for i, d in enumerate(dims)]
    feats = []
    for spec in specs:
        lengths = rng.choice([1, 1, 1, 2, 3, 5, 17, 64, 100, 127, 128, 129, 300], rows)
        f = feature_of(W, rng, spec.dim, lengths, spec.rows)
        f.table = f.feature = spec.id
        feats.append(f)
    print(f"case: dims={dims} occurrences={[len(f.keys) for f in feats]}", flush=True)
    shard = H.DeviceShard(torch, specs)
    shard.init_rows()
    dev = [H.DeviceFeature(torch, f) for f in feats]
    shard.prepare(dev)
    assert shard.push(dev) & H.STATUS_ERRORS == 0
    for spec, f in zip(specs, feats):
        store = oracle_store(spec)
        store.prepare(f)
        assert oracle.push([store], [f], [0], [f.gradient]) == 0
        keys = store.keys()
        want, _ = store.read_many(keys)
        got = shard.read_rows(spec.id, torch.from_numpy(keys.view(np.int64)).cuda()).cpu().numpy()
        assert_close(got.reshape(want.shape), want, f"dim={spec.dim} rows={rows}", strict_ulp=0)
