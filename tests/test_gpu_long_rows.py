"""Rows summed by a whole block (more than 32 references) beside rows summed by
one lane group, at the edges of both: the reduce entry point, a push of the
generic dimension class and CSR packets, bit-exact against the oracle (sums are
taken in reference order from +0, so the tolerance is 0 ULP)."""
import numpy as np
import pytest

import oracle
from parity import assert_close, oracle_store
from test_gpu_push import check_unique_reduce

pytestmark = pytest.mark.gpu
F32 = np.float32


def block_lengths(dim, widest=1 << 16):
    """Row lengths around the hand-over to the block, its tiles (4,096 products of 16-byte loads, 2,048 of scalar
    ones, a tile row the next power of two of the columns) and its groups of 128 references."""
    vector = dim % 4 == 0 and dim <= widest
    pitch = 32 if vector else 16
    while pitch < min(dim, 128):
        pitch *= 2
    tile = (4096 if vector else 2048) // pitch
    edges = [tile - 1, tile, tile + 1, 2 * tile - 1, 2 * tile, 3 * tile + 1, 127, 128, 129, 255, 256, 257]
    return [1, 2, 4, 5, 8, 9, 31, 32, 33, 48, 49] + sorted({max(e, 33) for e in edges})


def feature_of(W, rng, dim, lengths, rows):
    slots = rng.permutation(rows)[: len(lengths)].astype(np.uint64)
    keys = rng.permutation(np.repeat(slots, lengths))
    bags = len(keys) // 3 + 1
    cuts = np.sort(rng.integers(0, len(keys) + 1, bags - 1))
    offsets = np.concatenate([[0], cuts, [len(keys)]]).astype(np.uint64)
    weights = rng.normal(0, 1, len(keys)).astype(F32)
    grad = rng.normal(0, 1e-2, (bags, dim)).astype(F32)
    return W.Feature(0, 0, W.WEIGHTED_SUM, keys, offsets, np.diff(offsets), weights, grad)


@pytest.mark.parametrize("dim", [4, 12, 64, 100, 128, 256, 3, 10, 50, 257, 300, 520])
def test_reduce_long_rows(torch_gpu, pkg, dim):
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    rng = np.random.default_rng(dim)
    lengths = block_lengths(dim)
    specs = [W.TableSpec(0, dim, 400, seed=3)]
    feats = [feature_of(W, rng, dim, lengths, specs[0].rows)]
    print(f"case: dim={dim} row lengths {lengths}", flush=True)
    check_unique_reduce(torch, W, H, specs, feats)


@pytest.mark.parametrize("dim", [3, 50, 300])
def test_push_long_generic_rows(torch_gpu, pkg, dim):
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    rng = np.random.default_rng(1000 + dim)
    spec = W.TableSpec(0, dim, 400, seed=4)
    f = feature_of(W, rng, dim, block_lengths(dim), spec.rows)
    print(f"case: dim={dim} occurrences={len(f.keys)}", flush=True)
    shard = H.DeviceShard(torch, [spec])
    shard.init_rows()
    dev = [H.DeviceFeature(torch, f)]
    shard.prepare(dev)
    assert shard.push(dev) & H.STATUS_ERRORS == 0
    store = oracle_store(spec)
    store.prepare(f)
    assert oracle.push([store], [f], [0], [f.gradient]) == 0
    keys = store.keys()
    want, _ = store.read_many(keys)
    got = shard.read_rows(0, torch.from_numpy(keys.view(np.int64)).cuda()).cpu().numpy()
    assert_close(got.reshape(want.shape), want, f"generic push dim={dim}", strict_ulp=0)


def crowded_lengths(rng, dim, short):
    """The edges among `short` rows of 1 to 6 references: more than 1,024 windows of 8 positions."""
    return list(rng.permutation(np.concatenate([block_lengths(dim), [1000], rng.integers(1, 7, short)])))


# (520 and 514: rows of three units of columns, of 16-byte and scalar loads.)
@pytest.mark.parametrize("dim", [3, 50, 300, 520, 514])
def test_push_long_generic_rows_apart(torch_gpu, pkg, dim):
    """A push of enough positions that its short and long rows are launched apart."""
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    rng = np.random.default_rng(5000 + dim)
    spec = W.TableSpec(0, dim, 4000, seed=4)
    f = feature_of(W, rng, dim, crowded_lengths(rng, dim, 3000), spec.rows)
    assert len(f.keys) > 8 * 1024
    print(f"case: dim={dim} occurrences={len(f.keys)}", flush=True)
    shard = H.DeviceShard(torch, [spec])
    shard.init_rows()
    dev = [H.DeviceFeature(torch, f)]
    shard.prepare(dev)
    assert shard.push(dev) & H.STATUS_ERRORS == 0
    store = oracle_store(spec)
    store.prepare(f)
    assert oracle.push([store], [f], [0], [f.gradient]) == 0
    keys = store.keys()
    want, _ = store.read_many(keys)
    got = shard.read_rows(0, torch.from_numpy(keys.view(np.int64)).cuda()).cpu().numpy()
    assert_close(got.reshape(want.shape), want, f"generic push dim={dim}", strict_ulp=0)


def test_reduce_long_rows_apart(torch_gpu, pkg):
    """Every class in one call, short and long rows apart, rows that end with their class among them."""
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    rng = np.random.default_rng(6000)
    dims = [4, 300, 64, 10, 128, 256, 520, 32]
    specs = [W.TableSpec(i, d, 1500, seed=3 + i) for i, d in enumerate(dims)]
    feats = []
    for i, d in enumerate(dims):
        f = feature_of(W, rng, d, crowded_lengths(rng, d, 700), 1500)
        f.keys[f.keys == f.keys.max()] = 1499  # the last slot
        f.table = i
        feats.append(f)
    print(f"case: dims={dims} occurrences={sum(len(f.keys) for f in feats)}", flush=True)
    check_unique_reduce(torch, W, H, specs, feats)


@pytest.mark.parametrize("dims", [[300], [50, 64, 3]])
def test_checked_apply_of_long_rows(torch_gpu, pkg, dims):
    """The two-pass update (a bound the guard cannot prove safe) over short and long rows of vector and generic
    classes leaves the state of the fused one."""
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    rng = np.random.default_rng(7000 + len(dims))
    specs = [W.TableSpec(i, d, 4000, seed=5 + i) for i, d in enumerate(dims)]
    feats = []
    for i, d in enumerate(dims):
        f = feature_of(W, rng, d, crowded_lengths(rng, d, 2500), 4000)
        f.table = i
        feats.append(f)
    print(f"case: dims={dims} occurrences={sum(len(f.keys) for f in feats)}", flush=True)
    states = []
    for bound in (None, 2e30):
        shard = H.DeviceShard(torch, specs)
        shard.init_rows()
        if bound:
            shard.bounds.view(torch.float32)[0] = bound
        dev = [H.DeviceFeature(torch, f) for f in feats]
        shard.prepare(dev)
        status = shard.push(dev)
        assert status & H.STATUS_ERRORS == 0 and bool(status & H.STATUS_CHECKED_PATH) == bool(bound)
        states.append([s.cpu().numpy() for s in shard.state])
    assert all(np.array_equal(a, b) for a, b in zip(*states))


def check_compact(torch, W, H, dim, lengths, rng, table_rows, checked=False):
    spec = W.TableSpec(0, dim, table_rows, seed=5)
    lengths = np.asarray(lengths)
    rows, count = len(lengths), 300
    slots = rng.permutation(spec.rows)[:rows]
    offsets = np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint64)
    sources = rng.integers(0, count, int(offsets[-1])).astype(np.uint64)
    scales = rng.random(len(sources)).astype(F32)
    values = rng.normal(0, 1e-2, (count, dim)).astype(F32)
    print(f"case: dim={dim} rows={rows} references={len(sources)} checked={checked}", flush=True)
    shard = H.DeviceShard(torch, [spec])
    shard.init_rows()
    if checked:  # a bound that the guard cannot prove safe: validated first, then applied
        shard.bounds.view(torch.float32)[0] = 2e30
    at = torch.from_numpy(slots).cuda()
    before = shard.read_rows(0, at).cpu().numpy().reshape(rows, 3, dim)
    cuda = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    status = shard.adam_compact(0, at, cuda(offsets.view(np.int64)), cuda(sources.view(np.int64)), cuda(scales),
                                cuda(values))
    assert status & H.STATUS_ERRORS == 0 and bool(status & H.STATUS_CHECKED_PATH) == checked, f"{status:#x}"
    g = np.zeros((rows, dim), F32)
    for j in range(int(lengths.max())):  # reference j of every row that has one
        live = np.flatnonzero(lengths > j)
        r = offsets[live].astype(np.int64) + j
        g[live] = g[live] + values[sources[r].astype(np.int64)] * scales[r][:, None]
    rc, w, m, v = oracle.adam_rows_ctx(before[:, 0], before[:, 1], before[:, 2], g, spec.beta1, spec.beta2, spec.eps,
                                       spec.lr, spec.b1p, spec.b2p)
    assert rc == 0
    got = shard.read_rows(0, at).cpu().numpy().reshape(rows, 3, dim)
    assert_close(got, np.stack([w, m, v], 1), f"compact dim={dim}", strict_ulp=0)


@pytest.mark.parametrize("checked", [False, True])
@pytest.mark.parametrize("dim", [4, 64, 100, 256, 3, 50, 300, 514])
def test_compact_long_rows(torch_gpu, pkg, dim, checked):
    # An empty row, the edges, and enough short rows for several blocks.
    rng = np.random.default_rng(2000 + dim)
    lengths = [0] + block_lengths(dim, 256) + list(rng.integers(0, 7, 700))
    check_compact(torch_gpu, pkg.workloads, pkg.eps_hip, dim, lengths, rng, 4000, checked)


def test_compact_many_rows(torch_gpu, pkg):
    """More rows than are looked at one by one for long ones, the long ones first and last."""
    rng = np.random.default_rng(2100)
    lengths = np.concatenate([block_lengths(8), rng.integers(0, 3, 290_011), [40, 33, 1, 700]])
    check_compact(torch_gpu, pkg.workloads, pkg.eps_hip, 8, lengths, rng, 400_000)


@pytest.mark.parametrize("dim", [4, 16, 64, 256, 6, 33, 260, 301])
def test_reduce_rows_of_several_tiles(torch_gpu, pkg, dim):
    """Rows of several tiles and groups of 128 references: the last one full, one short and one over."""
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    rng = np.random.default_rng(3000 + dim)
    lengths = [33, 63, 64, 65, 127, 129, 255, 256, 257, 511, 513, 768, 769, 1025, 1281]
    specs = [W.TableSpec(0, dim, 400, seed=3)]
    feats = [feature_of(W, rng, dim, lengths, specs[0].rows)]
    print(f"case: dim={dim} row lengths {lengths}", flush=True)
    check_unique_reduce(torch, W, H, specs, feats)


@pytest.mark.parametrize("dim", [260, 300])
def test_gradients_off_the_vector_grid(torch_gpu, pkg, dim):
    """Gradient rows four bytes past a 16-byte boundary take the scalar loads: the same bits as aligned ones."""
    torch, W, H = torch_gpu, pkg.workloads, pkg.eps_hip
    rng = np.random.default_rng(4000 + dim)
    f = feature_of(W, rng, dim, [1, 33, 300, 700, 5], 500)
    states = []
    for shift in (0, 1):
        dev = H.DeviceFeature(torch, f)
        rows = torch.zeros(f.gradient.size + 1, device="cuda")[shift:][: f.gradient.size].view(f.gradient.shape)
        rows.copy_(dev.gradient)
        dev.gradient = rows
        print(f"case: dim={dim} gradients {rows.data_ptr() % 16} bytes past a 16-byte boundary", flush=True)
        shard = H.DeviceShard(torch, [W.TableSpec(0, dim, 500, seed=6)])
        shard.init_rows()
        shard.prepare([dev])
        assert shard.push([dev]) & H.STATUS_ERRORS == 0
        states.append(shard.state[0].cpu().numpy())
    assert np.array_equal(states[0], states[1])
