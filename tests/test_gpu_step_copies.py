"""GPU: a request-loop step's copies, whose host ends are pinned memory (whole or its inside, aligned or
not) or ordinary memory."""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def announce(msg):
    print(f"[gpu-case] {msg}", flush=True)


@pytest.mark.parametrize("pinned", [True, False])
@pytest.mark.parametrize("shift", [0, 1, 3])
@pytest.mark.parametrize("queries", [1, 37, 300])
def test_step_copies(pinned, shift, queries):
    import torch

    from simd_set_operations_amd import _native
    from simd_set_operations_amd.intersect import algo_id

    rng = np.random.Generator(np.random.PCG64(queries))
    sets = [np.unique(rng.integers(0, 900, rng.integers(1, 400))).astype(np.uint32) for _ in range(40)]
    beg = np.concatenate([[0], np.cumsum([s.size for s in sets])]).astype(np.uint64)
    pool = torch.from_numpy(np.concatenate(sets).view(np.int32)).cuda()
    ids = rng.integers(0, len(sets), (queries, 3))
    n = np.array([s.size for s in sets], np.uint64)
    rows = np.concatenate([beg[ids[:, 0]], beg[ids[:, 0]] + n[ids[:, 0]], beg[ids[:, 1]], beg[ids[:, 1]] + n[ids[:, 1]],
                           np.arange(queries + 1, dtype=np.uint64), beg[ids[:, 2]], beg[ids[:, 2]] + n[ids[:, 2]]])
    na, nb = (np.ascontiguousarray(n[ids[:, k]]) for k in (0, 1))
    need = int(np.minimum(na, nb).sum())

    def host(count, dtype, off):
        t = torch.full((count + off + 4,), 7, dtype=dtype)
        return (t.pin_memory() if pinned else t)[off:off + count]

    h_idx = host(rows.size, torch.int64, shift)
    h_idx.copy_(torch.from_numpy(rows.astype(np.uint64).view(np.int64)))
    h_off, h_out = host(queries + 1, torch.int64, shift), host(need, torch.int32, shift)
    d_idx = torch.zeros(rows.size, dtype=torch.int64, device="cuda")
    out = torch.zeros(need + 8, dtype=torch.int32, device="cuda")
    off = torch.zeros(queries + 1, dtype=torch.int64, device="cuda")
    cnt = torch.full((queries,), 9, dtype=torch.int32, device="cuda")
    tot = torch.zeros(2, dtype=torch.int64, device="cuda")
    lib = _native.hip()
    h = ctypes.c_void_p()
    one = torch.zeros(4, dtype=torch.int64, device="cuda")
    _native.check(lib.setops_hip_batch_create_gather(
        ctypes.byref(h), algo_id("hip_galloping"), pool.data_ptr(), None, pool.numel(), one.data_ptr(),
        one.data_ptr() + 8, pool.data_ptr(), None, pool.numel(), one.data_ptr() + 16, one.data_ptr() + 24, 1))
    announce(f"step copies pinned={pinned} shift={shift} queries={queries}")
    for _ in range(2):
        _native.check(lib.setops_hip_batch_step(
            h, h_idx.data_ptr(), d_idx.data_ptr(), queries, queries, na.ctypes.data, nb.ctypes.data, out.data_ptr(),
            need, off.data_ptr(), cnt.data_ptr(), tot.data_ptr(), h_off.data_ptr(), h_out.data_ptr(), need,
            torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        assert np.array_equal(d_idx.cpu().numpy().view(np.uint64), rows.astype(np.uint64))
        exp = [oracle.svs("branchless_merge", [sets[i] for i in q]) for q in ids]
        assert np.array_equal(cnt.cpu().numpy(), [e.size for e in exp])
        assert np.array_equal(np.diff(h_off.numpy()), [e.size for e in exp])
        total = int(h_off[-1])
        assert np.array_equal(h_out[:total].numpy().view(np.uint32), np.concatenate(exp))
        assert (h_out[total:] == 0).all()  # what the device buffer holds there
    lib.setops_hip_batch_destroy(h)
