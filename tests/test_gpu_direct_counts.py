"""GPU: count-only search batches that run without a plan launch (at most 256 pairs, at most 1,024 tiles),
and the first ones beyond each limit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def announce(msg):
    print(f"[gpu-case] {msg}", flush=True)


def batch(rng, sizes):
    a, b = [], []
    for na, nb in sizes:
        u = 2 * (na + nb) + 8
        a.append(np.sort(rng.choice(u, na, replace=False)).astype(np.uint32))
        b.append(np.sort(rng.choice(u, nb, replace=False)).astype(np.uint32))
    return a, b


# one tile of 512 probes, with and without padding and empty pairs; tiles that end with a pair; the most pairs
# and one more; about the most tiles and more
SIZES = {
    "one pair": [(9, 700)],
    "one tile": [(5, 9), (0, 7), (100, 900), (0, 0), (300, 3)],
    "whole tiles": [(512, 600)] * 4,
    "tiles": [(3, 1), (0, 0), (20000, 700), (1, 1), (0, 12000), (900, 4000)] * 9,
    "256 pairs": [(17, 40)] * 256,
    "257 pairs": [(17, 40)] * 257,
    "1,024 tiles": [(2048, 2100)] * 256,
    "more tiles": [(2100, 2100)] * 256,
}


@pytest.mark.parametrize("name", ["hip_galloping", "hip_binary_search@1", "hip_simd_galloping@2"])
@pytest.mark.parametrize("sizes", list(SIZES))
def test_count_only_search_batches(name, sizes):
    from simd_set_operations_amd import _native
    from simd_set_operations_amd.batch import DeviceBatch

    a, b = batch(np.random.Generator(np.random.PCG64(len(sizes))), SIZES[sizes])
    off = [np.concatenate([[0], np.cumsum([x.size for x in s])]).astype(np.uint64) for s in (a, b)]
    announce(f"counts {name} {sizes}")
    db = DeviceBatch(name, np.concatenate(a), off[0], np.concatenate(b), off[1])
    counts = np.array([np.intersect1d(x, y, assume_unique=True).size for x, y in zip(a, b)])
    ends = np.concatenate([[0], np.cumsum(counts)])
    for rep in range(3):
        db.d_counts.fill_(7)
        db.d_out_off.fill_(7)
        db.run(count_only=rep != 1)
        out_off, cnt, _ = db.results()
        assert np.array_equal(cnt, counts)
        assert np.array_equal(out_off, ends)
        assert db.totals() == (counts.sum(), counts.sum())
    # offsets alone, then counts alone
    lib, s = _native.hip(), db.torch.cuda.current_stream().cuda_stream
    db.d_out_off.fill_(7)
    _native.check(lib.setops_hip_batch_run(db.handle, None, None, 0, db.d_out_off.data_ptr(), None, None, s))
    assert np.array_equal(db.d_out_off.cpu().numpy(), ends)
    db.d_counts.fill_(7)
    _native.check(lib.setops_hip_batch_run(db.handle, None, None, 0, None, db.d_counts.data_ptr(), None, s))
    assert np.array_equal(db.d_counts.cpu().numpy(), counts)
    db.close()


@pytest.mark.parametrize("queries", [1, 40, 256, 300])
def test_count_only_kset_batches(queries):
    from simd_set_operations_amd.batch import KsetBatch

    rng = np.random.Generator(np.random.PCG64(queries))
    lists = [np.sort(rng.choice(6000, n, replace=False)).astype(np.uint32) for n in rng.integers(1, 2500, 60)]
    beg = np.concatenate([[0], np.cumsum([x.size for x in lists])]).astype(np.uint64)
    groups = [sorted(rng.choice(60, rng.integers(2, 6), replace=False), key=lambda i: lists[i].size)
              for _ in range(queries)]
    ids = np.concatenate(groups)
    announce(f"k-set counts {queries}")
    kb = KsetBatch("hip_galloping", np.concatenate(lists), beg[ids], beg[ids + 1],
                   np.concatenate([[0], np.cumsum([len(g) for g in groups])]), index=True)
    exp = []
    for g in groups:
        r = lists[g[0]]
        for i in g[1:]:
            r = np.intersect1d(r, lists[i], assume_unique=True)
        exp.append(r.size)
    for rep in range(2):
        kb.d_counts.fill_(7)
        kb.run(count_only=True)
        out_off, cnt, _ = kb.results()
        assert np.array_equal(cnt, exp)
        assert np.array_equal(out_off, np.concatenate([[0], np.cumsum(exp)]))
    kb.close()
