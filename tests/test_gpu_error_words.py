"""GPU: what setops_hip_batch_check reports of inputs that are no sets (values repeated so often that a
tile finds more results than sets can have), whatever form the run takes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def announce(msg):
    print(f"[gpu-case] {msg}", flush=True)


def csr_batch(name, pairs):
    from simd_set_operations_amd.batch import DeviceBatch

    off = [np.concatenate([[0], np.cumsum([p[s].size for p in pairs])]).astype(np.uint64) for s in (0, 1)]
    A, B = (np.concatenate([p[s] for p in pairs]) for s in (0, 1))
    st = {}
    if name.endswith("_bsr"):
        st = dict(A_states=np.full(A.size, 3, np.uint32), B_states=np.full(B.size, 1, np.uint32))
    return DeviceBatch(name, A, off[0], B, off[1], **st)


# pairs of 2,500 + 2,580 before and after the one whose A holds a value 12,000 times: the tiles that drop
# their results lie directly behind the first one, far behind it, and beyond the direct form's 1,024 tiles
@pytest.mark.parametrize("before,after", [(1, 0), (1, 40), (900, 3), (1100, 0)])
@pytest.mark.parametrize("name", ["hip_branchless_merge", "hip_branchless_merge@3", "hip_branchless_merge_bsr"])
def test_dropped_results_are_reported(name, before, after):
    from simd_set_operations_amd import _native

    a, b = np.arange(0, 5000, 2, dtype=np.uint32), np.arange(0, 7740, 3, dtype=np.uint32)
    n = before + after
    announce(f"dropped results {name} {before} {after}")
    for odd, ok in ((np.full(12000, 7, np.uint32), False), (np.arange(12000, dtype=np.uint32), True)):
        pairs = [(a, b)] * before + [(odd, np.array([7], np.uint32))] + [(a, b)] * after
        db = csr_batch(name, pairs)
        for rep in range(4):
            db.run(count_only=rep % 2 == 1)
            if ok:
                db.check()
                each = np.intersect1d(a, b).size
                assert db.totals() == (n * each + 1, n * each + 1)
            else:
                with pytest.raises(_native.SetopsError) as ei:
                    db.check()
                assert ei.value.code == _native.SETOPS_ERR_INVALID
        db.close()


# one tile whose A repeats values: more results than the output holds, none written past it
@pytest.mark.parametrize("name,a,b", [
    ("hip_shuffling", [np.repeat(np.arange(500), 4)], [np.arange(500)]),
    ("hip_shuffling", [np.repeat(np.arange(100), 4), np.repeat(np.arange(300), 3)], [np.arange(100), np.arange(300)]),
    ("hip_branchless_merge", [np.full(1004, 5), np.arange(0)], [np.array([5]), np.arange(1000)]),
])
def test_one_tile_stays_inside_the_output(name, a, b):
    import torch

    from simd_set_operations_amd import _native
    from simd_set_operations_amd.batch import to_device_u32
    from simd_set_operations_amd.intersect import algo_id

    a, b = ([x.astype(np.uint32) for x in s] for s in (a, b))
    total, results = sum(x.size for x in a), np.concatenate(a)  # every element of A is found
    cap = (total + sum(x.size for x in b)) // 2
    announce(f"one tile {name} {len(a)} pairs, {total} results, room for {cap}")
    assert total > cap
    db = csr_batch(name, list(zip(a, b)))
    assert db.info()["tiles"] == 1
    lib, stream = _native.hip(), torch.cuda.current_stream().cuda_stream
    out = torch.full((cap + 4096,), -1, dtype=torch.int32, device="cuda")
    for _ in range(2):
        _native.check(lib.setops_hip_batch_run(db.handle, out.data_ptr(), None, cap, db.d_out_off.data_ptr(),
                                               db.d_counts.data_ptr(), db.d_totals.data_ptr(), stream))
        with pytest.raises(_native.SetopsError) as ei:
            db.check()
        assert ei.value.code == _native.SETOPS_ERR_CAPACITY
        assert db.totals()[0] == total
        assert np.array_equal(out[:cap].cpu().numpy().view(np.uint32), results[:cap]) and (out[cap:] == -1).all()
    db.close()
    # a single pair has room for the smaller set
    cap = min(a[0].size, b[0].size)
    out.fill_(-1)
    da, d_b = to_device_u32(a[0], torch), to_device_u32(b[0], torch)
    tot = torch.zeros(2, dtype=torch.int64, device="cuda")
    _native.check(lib.setops_hip_intersect2_dev(algo_id(name), da.data_ptr(), None, a[0].size, d_b.data_ptr(), None,
                                                b[0].size, out.data_ptr(), None, cap, tot.data_ptr(), stream))
    torch.cuda.synchronize()
    assert (out[cap:] == -1).all()


def test_one_search_tile_of_wrong_sizes_stays_inside_the_output():
    """Device sizes beyond those given to setops_hip_batch_rebind: reported, and written no further than the
    room that the given sizes ask for."""
    import torch

    from simd_set_operations_amd import _native
    from simd_set_operations_amd.batch import GatherBatch

    P = 10
    pool = np.tile(np.arange(40, dtype=np.uint32), P)
    beg = np.arange(P, dtype=np.uint64) * np.uint64(40)
    announce("one search tile, sizes that differ")
    gb = GatherBatch("hip_galloping", pool, beg, beg + np.uint64(40), pool, beg, beg + np.uint64(40))
    lib, stream = _native.hip(), torch.cuda.current_stream().cuda_stream
    one = np.ones(P, np.uint64)
    _native.check(lib.setops_hip_batch_rebind(gb.handle, gb.dA_beg.data_ptr(), gb.dA_end.data_ptr(),
                                              gb.dB_beg.data_ptr(), gb.dB_end.data_ptr(), P, one.ctypes.data,
                                              one.ctypes.data))
    assert gb.info()["tiles"] == 1
    out = torch.full((P + 1024,), -1, dtype=torch.int32, device="cuda")
    _native.check(lib.setops_hip_batch_run(gb.handle, out.data_ptr(), None, P, gb.d_out_off.data_ptr(),
                                           gb.d_counts.data_ptr(), gb.d_totals.data_ptr(), stream))
    with pytest.raises(_native.SetopsError) as ei:
        gb.check()
    assert ei.value.code == _native.SETOPS_ERR_INVALID and "differ" in str(ei.value)
    assert (out[P:] == -1).all()
    gb.close()


def test_host_pair_with_repeated_values_copies_only_what_was_written():
    """A host call whose A repeats values: the count may exceed the smaller set's size, but nothing past the
    results that the kernels wrote (rounded up to the call's 256-byte pieces) reaches the caller."""
    from simd_set_operations_amd import intersect

    a, b = np.repeat(np.arange(500, dtype=np.uint32), 4), np.arange(500, dtype=np.uint32)
    announce("host pair, repeated values")
    out = np.full(2500, 0xABCD1234, np.uint32)
    n = intersect.intersect2_c("hip_shuffling", a, b, out)
    assert n == a.size and np.array_equal(out[:500], a[:500]) and (out[576:] == 0xABCD1234).all()


@pytest.mark.parametrize("further", [[], [np.arange(5000)], [np.arange(300), np.arange(5000)]])
def test_ksets_with_repeated_values_are_refused(further):
    """A fold that finds more results than its smaller set has elements ends the call with a capacity error,
    before a further fold reads that many from a buffer of the set's size."""
    from simd_set_operations_amd import _native, intersect

    sets = [np.repeat(np.arange(500), 4), np.arange(500)] + further
    announce(f"k-set with repeated values, {len(sets)} sets")
    with pytest.raises(_native.SetopsError) as ei:
        intersect.run_kset([s.astype(np.uint32) for s in sets], "hip_shuffling")
    assert ei.value.code == _native.SETOPS_ERR_CAPACITY


# pairs in one workgroup's scan, in several workgroups' shares of one, in group scans
@pytest.mark.parametrize("P", [300, 5000, 9000])
@pytest.mark.parametrize("name,units", [("hip_galloping", 512), ("hip_branchless_merge", 5120)])
def test_sizes_beyond_the_device_are_reported(name, units, P):
    """Host sizes given to setops_hip_batch_rebind that make 3,000 tiles more than the device offsets: the
    tiles past the pairs' end find no pair, and the run is reported; right sizes then give the results."""
    from simd_set_operations_amd import _native
    from simd_set_operations_amd.batch import GatherBatch

    rng = np.random.Generator(np.random.PCG64(P))
    sets = [np.unique(rng.integers(0, 4000, rng.integers(8, 60))).astype(np.uint32) for _ in range(50)]
    off = np.concatenate([[0], np.cumsum([s.size for s in sets])]).astype(np.uint64)
    pool = np.concatenate(sets)
    ia, ib = rng.integers(0, 50, P), rng.integers(0, 50, P)
    announce(f"sizes beyond the device {name} P={P}")
    gb = GatherBatch(name, pool, off[ia], off[ia + 1], pool, off[ib], off[ib + 1])
    na, nb = (np.ascontiguousarray(off[i + 1] - off[i]) for i in (ia, ib))
    tiles = gb.info()["tiles"]
    exp = [np.intersect1d(sets[i], sets[j], assume_unique=True) for i, j in zip(ia, ib)]
    for more in (3000 * units, 0):
        hna, hnb = na.copy(), nb.copy()
        hna[-1] += np.uint64(more)
        hnb[-1] += np.uint64(more if name == "hip_galloping" else 0)
        _native.check(_native.hip().setops_hip_batch_rebind(
            gb.handle, gb.dA_beg.data_ptr(), gb.dA_end.data_ptr(), gb.dB_beg.data_ptr(), gb.dB_end.data_ptr(), P,
            hna.ctypes.data, hnb.ctypes.data))
        for rep in range(2):
            gb.run(count_only=rep == 1)
            if more:
                assert gb.info()["tiles"] >= tiles + 2990
                with pytest.raises(_native.SetopsError) as ei:
                    gb.check()
                assert ei.value.code == _native.SETOPS_ERR_INVALID and "differ" in str(ei.value)
            else:
                o, cnt, data = gb.results()
                assert np.array_equal(cnt, [e.size for e in exp])
                if rep == 0:
                    assert np.array_equal(data, np.concatenate(exp))
    gb.close()
