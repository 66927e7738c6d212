"""Pooled gathers at the edges of the load widths (4, 2 or 1 floats, by the
dimension and the buffers' alignment), of rows wider than a wavefront's
columns, of sequence copies, of bags past what a block stages at a time and of
sources read by 64-bit offsets, bit-exact against the oracle (sums are taken in
occurrence order)."""
import ctypes as C

import numpy as np
import pytest

from parity import assert_close, oracle_store
from test_gpu_pull import expected, random_feature

pytestmark = pytest.mark.gpu


def check(torch, W, H, dim, pooling, rng, offset=0, rows=700, lengths=None, **bags):
    spec = W.TableSpec(5, dim, rows, seed=77 + dim)
    f = random_feature(W, rng, spec, pooling, **bags)
    if lengths is not None:
        lengths = np.asarray(lengths)
        offsets = np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint64)
        n = int(offsets[-1])
        f = W.Feature(0, 0, pooling, rng.integers(0, rows, n).astype(np.uint64), offsets, lengths.astype(np.uint64),
                      rng.random(n).astype(np.float32) if pooling == W.WEIGHTED_SUM else None)
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


@pytest.mark.parametrize("dim", [1, 2, 4, 16, 50, 64, 256, 300])
@pytest.mark.parametrize("pooling", [0, 1, 3])
def test_bags_around_a_groups_entries(torch_gpu, pkg, dim, pooling):
    """A group of G lanes stages 4 * G occurrences at a time where its block's bags hold more than 1,024:
    bags around one and two of those, empty ones and one of many beside them, in no order."""
    width = 4 if dim % 4 == 0 else 2 if dim % 2 == 0 else 1
    lanes = 4
    while lanes < 64 and lanes * width < dim:
        lanes *= 2
    room = 4 * lanes
    rng = np.random.default_rng(dim * 11 + pooling)
    lengths = [0, 1, lanes, room - 1, room, room + 1, 2 * room - 1, 2 * room, 2 * room + 3, 5, 0, 2500, 0, 7, 8, 9]
    check(torch_gpu, pkg.workloads, pkg.eps_hip, dim, pooling, rng, lengths=rng.permutation(np.tile(lengths, 5)))


@pytest.mark.parametrize("dim", [1, 2, 4, 64, 256, 300, 16_385])
@pytest.mark.parametrize("pooling", [0, 1, 3])
def test_one_bag_of_a_block(torch_gpu, pkg, dim, pooling):
    """A block's only occurrences are one bag's, past the 1,024 that it stages at a time: alone, the first and the
    last of empty ones, and beside one of a single occurrence."""
    W, H = pkg.workloads, pkg.eps_hip
    rng = np.random.default_rng(dim * 13 + pooling)
    for lengths in ([1025], [2048], [0] * 70 + [1500], [3001] + [0] * 70, [0] * 66 + [1, 1100]):
        check(torch_gpu, W, H, dim, pooling, rng, rows=100, lengths=lengths)


@pytest.mark.parametrize("dim", [256, 257, 258, 260, 300, 1028, 1030, 16_384, 16_385, 16_386, 16_388])
@pytest.mark.parametrize("pooling", [0, 1, 3])
def test_bags_of_one_row(torch_gpu, pkg, dim, pooling):
    """Bags of at most one occurrence, holes among them: copies where a row is wider than a wavefront's columns."""
    check(torch_gpu, pkg.workloads, pkg.eps_hip, dim, pooling, np.random.default_rng(dim * 17 + pooling), rows=60,
          bags=45, max_len=1, holes=0.3)


# The last dimension read through a 32-bit buffer range, and the first ones past it: loads of 1, 2 and 4 floats.
@pytest.mark.parametrize("dim", [16_384, 16_385, 16_386, 16_388])
@pytest.mark.parametrize("pooling", [0, 1, 2, 3])
def test_sources_past_a_buffer_range(torch_gpu, pkg, dim, pooling):
    check(torch_gpu, pkg.workloads, pkg.eps_hip, dim, pooling, np.random.default_rng(dim + pooling), rows=60, bags=13,
          max_len=20, holes=0.2)


@pytest.mark.parametrize("dim", [16_385, 16_386, 16_388])
@pytest.mark.parametrize("pooling", [0, 1, 3])
def test_bags_past_the_stage_past_a_buffer_range(torch_gpu, pkg, dim, pooling):
    check(torch_gpu, pkg.workloads, pkg.eps_hip, dim, pooling, np.random.default_rng(dim * 3 + pooling), rows=60,
          bags=6, max_len=700, holes=0.2)


@pytest.mark.parametrize("dim", [64, 50, 3, 16_385, 16_386, 16_388])
@pytest.mark.parametrize("pooling", [0, 1, 2, 3])
def test_only_holes(torch_gpu, pkg, dim, pooling):
    check(torch_gpu, pkg.workloads, pkg.eps_hip, dim, pooling, np.random.default_rng(dim), rows=60, bags=9, max_len=30,
          holes=1.0)


@pytest.mark.parametrize("dim", [64, 258, 300, 1028, 16_385, 16_388])
@pytest.mark.parametrize("lengths", [[1] * 40, [0, 1, 0, 3], [700, 1, 900, 1], [2000]])
def test_occurrences_claimed_without_indices(torch_gpu, pkg, dim, lengths):
    """Offsets that claim occurrences of a part without indices are bad indices: zeros, and the status bit."""
    torch, H = torch_gpu, pkg.eps_hip
    print(f"case: dim={dim} bags={len(lengths)}", flush=True)
    source = torch.full((60, dim), 3.0, device="cuda")
    offsets = torch.from_numpy(np.concatenate([[0], np.cumsum(lengths)])).cuda()
    valid = torch.from_numpy(np.asarray(lengths)).cuda()
    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    for pooling in (H.SUM, H.MEAN, H.WEIGHTED_SUM):
        out = torch.full((len(lengths), dim), -7.0, device="cuda")
        part = H.GatherPart(source.data_ptr(), None, None, offsets.data_ptr(),
                            valid.data_ptr() if pooling == H.MEAN else None, None, out.data_ptr(), dim, len(lengths),
                            60, 0, dim, pooling)
        status.zero_()
        H.check(H.lib().eps_hip_gather(C.byref(part), 1, status.data_ptr(), stream))
        torch.cuda.synchronize()
        assert int(status) & H.STATUS_BAD_INDEX
        assert not out.any()
