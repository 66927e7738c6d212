"""The shard's kept argument arrays follow every reassignment of a feature's
arrays, also of features that are only ever looked up (on the CPU: a stand-in
library records the pointers that a call passes)."""
import numpy as np
import pytest


class Recorder:
    """Stands in for the HIP library: sizes a shard asks for, and the arguments of its calls."""

    def __init__(self, H):
        self.H, self.parts, self.features = H, [], []

    def eps_hip_device_check(self, device):
        return 0

    def eps_hip_bounds_bytes(self):
        return 1024

    def eps_hip_update_workspace_bytes(self):
        return 1024

    def eps_hip_push_workspace_bytes(self, occurrences):
        return 1024

    def eps_hip_gather(self, parts, count, status, stream):
        self.parts = [{name: getattr(parts[i], name) for name, _ in self.H.GatherPart._fields_} for i in range(count)]
        return 0

    def eps_hip_prepare(self, tables, table_count, features, count, workspace, workspace_bytes, stream):
        self.features = [{name: getattr(features[i], name) for name, _ in self.H.PushFeature._fields_}
                         for i in range(count)]
        return 0


class Stream:
    cuda_stream = 0


@pytest.fixture
def shard(pkg, monkeypatch):
    import torch
    W, H = pkg.workloads, pkg.eps_hip
    recorder = Recorder(H)
    monkeypatch.setattr(H, "lib", lambda: recorder)
    return torch, W, H, recorder, H.DeviceShard(torch, [W.TableSpec(0, 4, 50)], device="cpu")


def feature(torch, W, H, pooling):
    keys, offsets = np.arange(6, dtype=np.uint64), np.array([0, 2, 6], np.uint64)
    weights = np.ones(6, np.float32) if pooling == W.WEIGHTED_SUM else None
    return H.DeviceFeature(torch, W.Feature(0, 0, pooling, keys, offsets, np.diff(offsets), weights,
                                            np.ones((2, 4), np.float32)), device="cpu")


@pytest.mark.parametrize("pushed", [False, True])
@pytest.mark.parametrize("field,argument", [("indices", "indices"), ("offsets", "offsets"), ("weights", "weights"),
                                            ("valid_lengths", "valid_lengths"), ("rows", "rows")])
def test_lookup_follows_reassignment(shard, field, argument, pushed):
    torch, W, H, recorder, shard = shard
    f = feature(torch, W, H, W.MEAN if field == "valid_lengths" else W.WEIGHTED_SUM)
    out = torch.zeros(2, 4)
    if pushed:
        shard.prepare([f], stream=Stream)
    shard.lookup([f], [out], stream=Stream)
    kept = []  # (so that no new array takes an old one's address)
    for _ in range(3):
        kept.append(getattr(f, field))
        setattr(f, field, kept[-1].clone() if torch.is_tensor(kept[-1]) else 3 - kept[-1])
        if pushed:
            shard.prepare([f], stream=Stream)
        shard.lookup([f], [out], stream=Stream)
        now = getattr(f, field)
        assert recorder.parts[0][argument] == (now.data_ptr() if torch.is_tensor(now) else now)
        assert recorder.parts[0]["output"] == out.data_ptr()


def test_prepare_follows_reassignment(shard):
    torch, W, H, recorder, shard = shard
    f = feature(torch, W, H, W.SUM)
    kept = []
    for _ in range(3):
        shard.prepare([f], stream=Stream)
        assert recorder.features[0]["indices"] == f.indices.data_ptr()
        kept.append(f.indices)
        f.indices = kept[-1].clone()


def test_kept_arguments_are_reused(shard):
    """Nothing is rebuilt while nothing changes."""
    torch, W, H, recorder, shard = shard
    f, out = feature(torch, W, H, W.SUM), torch.zeros(2, 4)
    shard.lookup([f], [out], stream=Stream)
    first = next(iter(shard._args_cache.values()))
    shard.lookup([f], [out], stream=Stream)
    assert len(shard._args_cache) == 1 and next(iter(shard._args_cache.values())) is first
