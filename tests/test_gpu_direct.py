"""GPU: batches and single pairs that run without a plan launch (the tile kernels' direct form and the
fused placement, which writes offsets and counts), at the edges of tiles and of the form's limits, as
plain, int32 and BSR sets, with and without counts, and the planned form beside them."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def announce(msg):
    print(f"[gpu-case] {msg}", flush=True)


def pair(rng, na, nb, signed=False):
    u = 2 * (na + nb) + 8
    a = np.sort(rng.choice(u, na, replace=False))
    b = np.sort(rng.choice(u, nb, replace=False))
    if signed:
        a, b = a - u // 2, b - u // 2
    dt = np.int32 if signed else np.uint32
    return a.astype(dt), b.astype(dt)


# pair sizes of a batch: one tile; a pair over several tiles beside tiny and empty ones; tiles that start with a
# pair; about the fused placement's 1,024 tiles of 5,120 units and one more
SIZES = {
    "one tile": [(5, 9), (0, 7), (1000, 900), (0, 0), (3, 0)],
    "mixed": [(3, 1), (0, 0), (20000, 7000), (1, 1), (0, 12000), (9000, 0)] + [(17, 40)] * 300 + [(2560, 2520)] * 5,
    "whole tiles": [(2540, 2540)] * 6 + [(1, 1)],
    "tiny": [(1, 2)] * 700,
    "limit": [(2500, 2580)] * 1022,
    "beyond": [(2500, 2580)] * 1026,
}


@pytest.mark.parametrize("name", ["hip_branchless_merge", "hip_shuffling", "hip_galloping"])
@pytest.mark.parametrize("signed", [False, True])
@pytest.mark.parametrize("sizes", list(SIZES))
def test_direct_batches(name, signed, sizes):
    from simd_set_operations_amd import _native
    from simd_set_operations_amd.batch import DeviceBatch

    rng = np.random.Generator(np.random.PCG64(len(SIZES[sizes]) + signed))
    pairs = [pair(rng, na, nb, signed) for na, nb in SIZES[sizes]]
    off = [np.concatenate([[0], np.cumsum([p[s].size for p in pairs])]).astype(np.uint64) for s in (0, 1)]
    A, B = (np.concatenate([p[s] for p in pairs]) for s in (0, 1))
    announce(f"direct {name} signed={signed} {sizes}")
    db = DeviceBatch(name, A, off[0], B, off[1])
    exp = [np.intersect1d(a, b, assume_unique=True) for a, b in pairs]
    counts = np.array([e.size for e in exp])
    for rep in range(3):
        db.d_counts.fill_(7)
        db.d_out_off.fill_(7)
        db.run(count_only=rep == 1)
        out_off, cnt, data = db.results()
        assert np.array_equal(cnt, counts)
        assert np.array_equal(out_off, np.concatenate([[0], np.cumsum(counts)]))
        assert db.totals() == (counts.sum(), counts.sum())
        if rep != 1:
            assert np.array_equal(data, np.concatenate(exp))
    # offsets alone (no counts asked for)
    db.d_out_off.fill_(7)
    _native.check(_native.hip().setops_hip_batch_run(db.handle, db.d_out.data_ptr(), None, db.d_out.numel(),
                                                     db.d_out_off.data_ptr(), None, None,
                                                     db.torch.cuda.current_stream().cuda_stream))
    assert np.array_equal(db.d_out_off.cpu().numpy(), np.concatenate([[0], np.cumsum(counts)]))
    db.close()


@pytest.mark.parametrize("na,nb", [(0, 0), (1, 0), (2500, 2500), (2540, 2540), (2541, 2541), (5000, 5001), (40000, 3),
                                   (3, 40000), (65536, 65536), (2621000, 2621000), (2700000, 2700000)])
def test_direct_single_pairs(na, nb):
    from simd_set_operations_amd import _native
    from simd_set_operations_amd.batch import to_device_u32
    from simd_set_operations_amd.bsr import BsrVec
    from simd_set_operations_amd.intersect import algo_id
    import torch

    rng = np.random.Generator(np.random.PCG64(na + 3 * nb))
    a, b = pair(rng, na, nb)
    exp = np.intersect1d(a, b, assume_unique=True)
    announce(f"direct pair {na} {nb}")
    lib = _native.hip()
    stream = torch.cuda.current_stream().cuda_stream
    tot = torch.zeros(2, dtype=torch.int64, device="cuda")
    calls = [lib.setops_hip_intersect2_dev] + ([lib.setops_hip_intersect2_dev_noalloc] if na + nb <= 1 << 22 else [])
    da, db = to_device_u32(a, torch), to_device_u32(b, torch)
    for call in calls:
        for cap in (min(na, nb), exp.size // 2):  # the second clips the writes
            out = torch.full((max(min(na, nb), 1) + 8,), -1, dtype=torch.int32, device="cuda")
            tot.fill_(7)
            _native.check(call(algo_id("hip_branchless_merge"), da.data_ptr(), None, na, db.data_ptr(), None, nb,
                               out.data_ptr(), None, cap, tot.data_ptr(), stream))
            got = out.cpu().numpy()
            n = min(cap, exp.size)
            assert tot.tolist() == [exp.size, exp.size]
            assert np.array_equal(got[:n].view(np.uint32), exp[:n]) and (got[max(n, 1):] == -1).all()
        tot.fill_(7)
        _native.check(call(algo_id("hip_branchless_merge"), da.data_ptr(), None, na, db.data_ptr(), None, nb, None, None,
                           0, tot.data_ptr(), stream))
        assert tot.tolist() == [exp.size, exp.size]
    va, vb, ve = BsrVec.from_sorted(a), BsrVec.from_sorted(b), BsrVec.from_sorted(exp)
    n = min(va.bases.size, vb.bases.size)
    dv = [to_device_u32(x, torch) for x in (va.bases, va.states, vb.bases, vb.states)]
    ob, os_ = (torch.full((n + 8,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    _native.check(lib.setops_hip_intersect2_dev(
        algo_id("hip_branchless_merge_bsr"), dv[0].data_ptr(), dv[1].data_ptr(), va.bases.size, dv[2].data_ptr(),
        dv[3].data_ptr(), vb.bases.size, ob.data_ptr(), os_.data_ptr(), n, tot.data_ptr(), stream))
    w = ve.bases.size
    assert tot.tolist() == [w, exp.size]
    assert np.array_equal(ob[:w].cpu().numpy().view(np.uint32), ve.bases)
    assert np.array_equal(os_[:w].cpu().numpy().view(np.uint32), ve.states)
