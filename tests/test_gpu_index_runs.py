"""Key index with buckets probed four at a time (inserts of 2^20 keys and more:
one): indexes smaller than a run, runs around the end, an index without an empty
bucket, and keys that are not in it."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("capacity,count", [(2, 1), (2, 2), (4, 3), (8, 8), (256, 250), (1024, 1024), (1 << 16, 30_011),
                                            (1 << 21, 1 << 20)])
def test_insert_remove_resolve(torch_gpu, pkg, capacity, count):
    torch, H = torch_gpu, pkg.eps_hip
    lib = H.lib()
    print(f"case: capacity={capacity} count={count}", flush=True)
    rng = np.random.default_rng(capacity + count)
    keys = rng.choice(1 << 40, 3 * count + 8, replace=False).astype(np.int64)
    first, second, absent = keys[:count], keys[count:2 * count], keys[2 * count:]
    index = torch.empty(lib.eps_hip_index_bytes(capacity) // 8, dtype=torch.int64, device="cuda")
    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    device = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()

    def insert(k, slots):
        k, slots = device(k), device(slots)
        H.check(lib.eps_hip_index_insert(index.data_ptr(), capacity, k.data_ptr(), slots.data_ptr(), len(k),
                                         status.data_ptr(), stream))
        torch.cuda.synchronize()

    def remove(k):
        k = device(k)
        H.check(lib.eps_hip_index_remove(index.data_ptr(), capacity, k.data_ptr(), len(k), status.data_ptr(), stream))
        torch.cuda.synchronize()

    def resolve(k):
        k, out = device(k), torch.empty(len(k), dtype=torch.int64, device="cuda")
        H.check(lib.eps_hip_resolve(index.data_ptr(), capacity, k.data_ptr(), None, None, 0, len(k), out.data_ptr(),
                                    status.data_ptr(), stream))
        return out.cpu().numpy()

    H.check(lib.eps_hip_index_clear(index.data_ptr(), capacity, stream))
    insert(first, np.arange(count))
    assert (resolve(first) == np.arange(count)).all() and (resolve(absent) == -1).all()
    gone = count // 2 + 1
    remove(first[:gone])
    assert (resolve(first[:gone]) == -1).all() and (resolve(first[gone:]) == np.arange(gone, count)).all()
    insert(second[:gone], 1000 + np.arange(gone))  # takes the removed buckets' place
    assert (resolve(second[:gone]) == 1000 + np.arange(gone)).all()
    assert (resolve(first[gone:]) == np.arange(gone, count)).all() and (resolve(absent) == -1).all()
    assert int(status) == 0
    remove(absent[:1])
    assert int(status) & H.STATUS_ERRORS
