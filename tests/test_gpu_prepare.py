"""The device preparation at the edges of its routes: one block (up to 4,096
occurrences and 8,192 staged offsets) and tiles of 4,096 per feature; tables
whose digit counts each pass adds up itself (up to 32 tiles) and longer ones;
one to three radix passes; several features a table in mixed order; holes.
Unique rows, the occurrence map and the reduced sums are compared with the
oracle, and a push of the same features (which sorts without occurrence
indices) must leave the oracle's state, bit for bit."""
import numpy as np
import pytest

import oracle
from parity import assert_close, oracle_store
from test_gpu_push import HOLE, check_unique_reduce, live

pytestmark = pytest.mark.gpu
F32 = np.float32


def feature(W, rng, specs, table, index, occurrences, pooling, holes=0.0, empty=0, skew=1.3):
    """`occurrences` ids in bags of 0..3, behind `empty` empty bags."""
    lengths = [0] * empty
    left = occurrences
    while left:
        take = min(left, int(rng.integers(0, 4)))
        lengths.append(take)
        left -= take
    if pooling == W.SEQUENCE and not lengths:
        lengths = [0]
    lengths = np.array(lengths or [0])
    offsets = np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint64)
    keys = (rng.zipf(skew, occurrences) % specs[table].rows).astype(np.uint64)
    keys[rng.random(occurrences) < holes] = HOLE
    weights = rng.normal(0, 1, occurrences).astype(F32) if pooling == W.WEIGHTED_SUM else None
    rows = occurrences if pooling == W.SEQUENCE else len(lengths)
    grad = rng.normal(0, 1e-2, (rows, specs[table].dim)).astype(F32)
    return W.Feature(table, index, pooling, keys, offsets, lengths.astype(np.uint64), weights, grad)


def check(torch, W, H, specs, feats):
    check_unique_reduce(torch, W, H, specs, feats)
    shard = H.DeviceShard(torch, specs)
    shard.init_rows()
    dev = [H.DeviceFeature(torch, f) for f in feats]
    shard.prepare(dev)
    status = shard.push(dev)
    assert status & H.STATUS_ERRORS == 0, f"{status:#x}"
    for t, spec in enumerate(specs):
        sel = [live(f) for f in feats if f.table == t]
        if not sel:
            continue
        store = oracle_store(spec)
        for f in sel:
            store.prepare(f)
        assert oracle.push([store], sel, [0] * len(sel), [f.gradient for f in sel]) == 0
        keys = store.keys()
        if not len(keys):
            continue
        want, _ = store.read_many(keys)
        got = shard.read_rows(t, torch.from_numpy(keys.view(np.int64)).cuda()).cpu().numpy()
        assert_close(got.reshape(want.shape), want, f"push table {t}", strict_ulp=0)


@pytest.mark.parametrize("occurrences", [1, 2, 63, 64, 65, 129, 1023, 1025, 4095, 4096, 4097, 8193])
@pytest.mark.parametrize("weighted", [False, True])
def test_occurrence_counts(torch_gpu, pkg, occurrences, weighted):
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    rng = np.random.default_rng(occurrences)
    specs = [W.TableSpec(0, 4, 3000, seed=1)]
    pooling = W.WEIGHTED_SUM if weighted else W.MEAN
    print(f"case: {occurrences} occurrences, weighted {weighted}", flush=True)
    check(torch, W, H, specs, [feature(W, rng, specs, 0, 0, occurrences, pooling, holes=0.1)])


@pytest.mark.parametrize("pooled,sequences,occurrences", [(32, 0, 4096), (32, 0, 4097), (16, 3, 2049), (0, 32, 4096)])
def test_many_features(torch_gpu, pkg, pooled, sequences, occurrences):
    """As many features as a push holds, over three tables, in one block and in tiles."""
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    rng = np.random.default_rng(pooled + occurrences)
    specs = [W.TableSpec(i, d, 900, seed=20 + i) for i, d in enumerate([4, 64, 10])]
    count = pooled + sequences
    share = [occurrences // count + (i < occurrences % count) for i in range(count)]
    feats = [feature(W, rng, specs, i % 3, i, share[i],
                     W.SEQUENCE if i >= pooled else [W.SUM, W.MEAN, W.WEIGHTED_SUM][i % 3]) for i in range(count)]
    print(f"case: {pooled} pooled features, {sequences} sequences, {occurrences} occurrences", flush=True)
    check(torch, W, H, specs, feats)


@pytest.mark.parametrize("empty", [0, 5000, 8000, 9000])
def test_empty_bags_beside_the_staged_offsets(torch_gpu, pkg, empty):
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    rng = np.random.default_rng(empty)
    specs = [W.TableSpec(0, 4, 500, seed=2), W.TableSpec(1, 8, 70, seed=3)]
    print(f"case: {empty} empty bags", flush=True)
    check(torch, W, H, specs, [feature(W, rng, specs, 0, 0, 90, W.MEAN, empty=empty),
                               feature(W, rng, specs, 1, 1, 0, W.SUM),
                               feature(W, rng, specs, 1, 2, 40, W.SEQUENCE)])


@pytest.mark.parametrize("rows", [1, 2, 1000, 1024, 1025, 1 << 20, (1 << 20) + 1, 1 << 24])
@pytest.mark.parametrize("occurrences", [700, 9000])
def test_key_widths(torch_gpu, pkg, rows, occurrences):
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    rng = np.random.default_rng(rows % 1009 + occurrences)
    specs = [W.TableSpec(0, 4, rows, seed=4), W.TableSpec(1, 4, 77, seed=5)]
    feats = [feature(W, rng, specs, 0, 0, occurrences, W.SUM, skew=1.05),
             feature(W, rng, specs, 1, 1, 333, W.SEQUENCE)]
    feats[0].keys[:2] = [rows - 1, 0]
    print(f"case: {rows} rows, {occurrences} occurrences", flush=True)
    check(torch, W, H, specs, feats)


@pytest.mark.parametrize("weighted", [False, True])
def test_features_of_mixed_tables(torch_gpu, pkg, weighted):
    """Tables in an order of classes unlike the call's, several features each,
    features between, all holes in one of them."""
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    rng = np.random.default_rng(17)
    specs = [W.TableSpec(i, d, r, seed=6 + i) for i, (d, r) in enumerate([(64, 900), (6, 50), (4, 5000), (300, 40)])]
    plan = [(2, 5000), (0, 4096), (1, 300), (2, 4097), (3, 200), (0, 1), (2, 0), (0, 3000)]
    poolings = [W.MEAN, W.SUM, W.SEQUENCE, W.WEIGHTED_SUM if weighted else W.MEAN]
    feats = [feature(W, rng, specs, t, i, n, poolings[i % 4], holes=1.0 if i == 5 else 0.05)
             for i, (t, n) in enumerate(plan)]
    print(f"case: weighted {weighted}", flush=True)
    check(torch, W, H, specs, feats)


@pytest.mark.parametrize("occurrences", [131_072, 131_073, 210_000])
@pytest.mark.parametrize("weighted", [False, True])
def test_long_tables(torch_gpu, pkg, occurrences, weighted):
    """At most 32 tiles (counts added up by each block) and more, with a second
    table so that segments and groups of both meet."""
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    rng = np.random.default_rng(occurrences)
    specs = [W.TableSpec(0, 4, 40_000, seed=11), W.TableSpec(1, 4, 1_200_000, seed=12)]
    pooling = W.WEIGHTED_SUM if weighted else W.MEAN
    feats = [feature(W, rng, specs, 1, 0, 30_000, W.SUM, holes=0.02),
             feature(W, rng, specs, 0, 1, occurrences, pooling, holes=0.02),
             feature(W, rng, specs, 1, 2, 50_000, pooling, skew=1.1)]
    print(f"case: {occurrences} occurrences, weighted {weighted}", flush=True)
    check(torch, W, H, specs, feats)
