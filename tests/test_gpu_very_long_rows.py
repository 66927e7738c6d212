"""Rows of 65,536 or more references, which the hot-row kernel gives a block
per unit, at the edges of their chunks (128 references of 32-column units, 256
of 16-column ones) and beside rows just below: bit-exact against the oracle.
With a spin limit of 0 such rows stall like every hot row and are not
written."""
import numpy as np
import pytest

import oracle
from parity import assert_close, oracle_store

pytestmark = pytest.mark.gpu
F32 = np.float32


def push_case(W, rng, dims, counts, others, pooling):
    """One feature per table; table 0's rows take `counts` references each,
    `others` more are spread over every table."""
    specs = [W.TableSpec(i, d, 3000, seed=40 + i) for i, d in enumerate(dims)]
    feats = []
    for t, spec in enumerate(specs):
        keys = rng.integers(100, spec.rows, others // len(specs)).astype(np.uint64)
        if t == 0:
            keys = rng.permutation(np.concatenate([keys, np.repeat(np.arange(len(counts), dtype=np.uint64), counts)]))
        lengths = np.full(len(keys) // 4 + 1, 4)
        lengths[-1] = len(keys) - 4 * (len(lengths) - 1)
        offsets = np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint64)
        weights = rng.random(len(keys)).astype(F32) if pooling == W.WEIGHTED_SUM else None
        grad = rng.normal(0, 1e-2, (len(lengths), spec.dim)).astype(F32)
        feats.append(W.Feature(t, t, pooling, keys, offsets, lengths.astype(np.uint64), weights, grad))
    return specs, feats


@pytest.mark.parametrize("dims", [(4,), (36, 8), (128,), (256, 64)])
@pytest.mark.parametrize("others", [2000, 150_000])
def test_very_long_rows(torch_gpu, pkg, dims, others):
    """2,000 other references: 16-column units; 150,000: over 262,144 in all,
    32-column units."""
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    rng = np.random.default_rng(sum(dims) + others)
    counts = [65_536, 65_535, 65_537, 129] if others > 2000 else [65_536 + 255, 65_535, 129]
    specs, feats = push_case(W, rng, dims, counts, others, W.MEAN if dims[0] % 8 else W.WEIGHTED_SUM)
    total = sum(len(f.keys) for f in feats)
    print(f"case: dims={dims} references={total}", flush=True)
    assert (total < 1 << 18) == (others == 2000)
    shard = H.DeviceShard(torch, specs)
    shard.init_rows()
    dev = [H.DeviceFeature(torch, f) for f in feats]
    shard.prepare(dev)
    assert shard.push(dev) & H.STATUS_ERRORS == 0
    for t, spec in enumerate(specs):
        store = oracle_store(spec)
        store.prepare(feats[t])
        assert oracle.push([store], [feats[t]], [0], [feats[t].gradient]) == 0
        keys = store.keys()
        want, _ = store.read_many(keys)
        got = shard.read_rows(t, torch.from_numpy(keys.view(np.int64)).cuda()).cpu().numpy()
        assert_close(got.reshape(want.shape), want, f"very long rows table {t}", strict_ulp=0)


@pytest.mark.parametrize("others", [2000, 150_000])
def test_very_long_row_stalls_unwritten(torch_gpu, pkg, others):
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    specs, feats = push_case(W, np.random.default_rng(9), (64,), [70_000, 66_000, 300], others, W.SUM)
    shard = H.DeviceShard(torch, specs)
    shard.init_rows()
    hot = torch.arange(3, device="cuda")
    before = shard.read_rows(0, hot).clone()
    dev = [H.DeviceFeature(torch, f) for f in feats]
    print(f"case: stalled very long rows, {others} others", flush=True)
    try:
        H.check(H.lib().eps_hip_debug_set_spin_limit(0))
        shard.prepare(dev)
        status = shard.push(dev)
    finally:
        H.check(H.lib().eps_hip_debug_set_spin_limit(1 << 22))
    assert status & H.STATUS_STALLED, f"{status:#x}"
    assert torch.equal(shard.read_rows(0, hot), before), "a stalled row was written"
