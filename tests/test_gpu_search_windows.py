"""GPU: search tiles whose larger windows are staged whole, sampled (one line or many per sample) or too
many for LDS, in A and in B, in plain, int32 and BSR form, with and without the B-pool index, with
sets that start and end inside a 32-element line."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def announce(msg):
    print(f"[gpu-case] {msg}", flush=True)


def make_sets(small, large, npairs, signed):
    """npairs pairs of about `small` against `large` elements, a few of them shared; odd sizes, and the
    larger set on either side."""
    rng = np.random.Generator(np.random.PCG64(small * 7919 + large))
    a, b = [], []
    for p in range(npairs):
        u = 4 * large + 64
        big = np.sort(rng.choice(u, large + p % 3, replace=False))
        own = rng.choice(u, max(small - small // 3, 1), replace=False)
        ends = big[[0, -1]] if p % 2 else big[[large // 2]]
        sm = np.unique(np.concatenate([own, rng.choice(big, small // 3), ends]))
        if signed:
            big, sm = big - u // 2, sm - u // 2
        dt = np.int32 if signed else np.uint32
        x, y = sm.astype(dt), big.astype(dt)
        a.append(y if p % 4 == 3 else x)
        b.append(x if p % 4 == 3 else y)
    return a, b


def csr(sets):
    return np.concatenate(sets), np.concatenate([[0], np.cumsum([s.size for s in sets])]).astype(np.uint64)


# (probes per pair, larger set, pairs): staged; one line a sample; the fewest samples; many lines a sample;
# pairs over several tiles; more windows than LDS holds
SHAPES = [(100, 500, 9), (300, 9000, 7), (3, 700, 300), (2, 90000, 40), (6000, 60000, 2), (5000, 9000, 3),
          (4, 2300, 1000), (1, 33, 500)]


@pytest.mark.parametrize("small,large,npairs", SHAPES)
@pytest.mark.parametrize("name,signed", [("hip_galloping", False), ("hip_binary_search@2", True),
                                         ("hip_simd_galloping@1", False)])
@pytest.mark.parametrize("indexed", [False, True])
def test_search_windows(name, signed, indexed, small, large, npairs):
    from simd_set_operations_amd.batch import DeviceBatch

    a, b = make_sets(small, large, npairs, signed)
    A, ao = csr(a)
    B, bo = csr(b)
    announce(f"windows {name} signed={signed} indexed={indexed} {small} against {large} x {npairs}")
    db = DeviceBatch(name, A, ao, B, bo)
    if indexed:
        db.index_b()
    exp = [np.intersect1d(x, y, assume_unique=True) for x, y in zip(a, b)]
    for _ in range(2):
        db.run()
        off, cnt, data = db.results()
        assert np.array_equal(cnt, [e.size for e in exp])
        assert np.array_equal(data, np.concatenate(exp))
    db.run(count_only=True)
    assert db.totals()[0] == sum(e.size for e in exp)
    db.close()


@pytest.mark.parametrize("small,large,npairs", SHAPES)
def test_search_windows_bsr(small, large, npairs):
    from simd_set_operations_amd.batch import DeviceBatch
    from simd_set_operations_amd.bsr import BsrVec

    a, b = make_sets(small, large, npairs, False)
    va, vb = [BsrVec.from_sorted(x) for x in a], [BsrVec.from_sorted(x) for x in b]
    A, ao = csr([v.bases for v in va])
    B, bo = csr([v.bases for v in vb])
    announce(f"windows bsr {small} against {large} x {npairs}")
    db = DeviceBatch("hip_galloping_bsr", A, ao, B, bo, A_states=np.concatenate([v.states for v in va]),
                     B_states=np.concatenate([v.states for v in vb]))
    db.run()
    off, cnt, data, states = db.results()
    for p in range(npairs):
        exp = BsrVec.from_sorted(oracle.branchless_merge(a[p], b[p]))
        o, n = int(off[p]), int(cnt[p])
        assert n == exp.bases.size
        assert np.array_equal(data[o:o + n], exp.bases) and np.array_equal(states[o:o + n], exp.states)
    db.close()
