"""GPU: batches of BSR sets that run without a plan launch (states, counts and offsets over several tiles), at the
edges of tiles and of the direct form's limits, and the planned form beside them."""
import numpy as np
import pytest

from test_gpu_direct import announce, pair

pytestmark = pytest.mark.gpu

# words per pair; a BSR tile has 2,560 units, a pair 20 units of padding
SIZES = {
    "one tile": [(5, 9), (0, 7), (500, 300), (0, 0), (3, 0)],
    "mixed": [(3, 1), (0, 0), (20000, 7000), (1, 1), (0, 12000), (9000, 0)] + [(17, 40)] * 300 + [(1280, 1260)] * 5,
    "whole tiles": [(1270, 1270)] * 6 + [(1, 1)],
    "tiny": [(1, 2)] * 700,
    "limit": [(1260, 1280)] * 1022,
    "beyond": [(1260, 1280)] * 1026,
}


@pytest.mark.parametrize("name", ["hip_branchless_merge_bsr", "hip_shuffling_bsr", "hip_qfilter_bsr"])
@pytest.mark.parametrize("sizes", list(SIZES))
def test_direct_bsr_batches(name, sizes):
    from simd_set_operations_amd.batch import DeviceBatch

    rng = np.random.Generator(np.random.PCG64(len(SIZES[sizes])))
    pairs = [pair(rng, na, nb) for na, nb in SIZES[sizes]]
    # the states of few bits: some common bases have no common bit
    states = [[(1 << rng.integers(0, 3, s.size)).astype(np.uint32) | np.uint32(8) * (s % 5 == 0) for s in p] for p in pairs]
    off = [np.concatenate([[0], np.cumsum([p[s].size for p in pairs])]).astype(np.uint64) for s in (0, 1)]
    A, B = (np.concatenate([p[s] for p in pairs]) for s in (0, 1))
    As, Bs = (np.concatenate([p[s] for p in states]).astype(np.uint32) for s in (0, 1))
    words, bits = [], []
    for (a, b), (sa, sb) in zip(pairs, states):
        w, i, j = np.intersect1d(a, b, assume_unique=True, return_indices=True)
        s = (sa[i] & sb[j]).astype(np.uint32)
        words.append(w[s != 0])
        bits.append(s[s != 0])
    counts = np.array([w.size for w in words])
    elems = sum(bin(s).count("1") for s in np.concatenate(bits))
    announce(f"direct bsr {name} {sizes}")
    db = DeviceBatch(name, A, off[0], B, off[1], A_states=As, B_states=Bs)
    for rep in range(3):
        db.d_counts.fill_(7)
        db.d_out_off.fill_(7)
        db.run(count_only=rep == 1)
        out_off, cnt, data, st = db.results()
        assert np.array_equal(cnt, counts)
        assert np.array_equal(out_off, np.concatenate([[0], np.cumsum(counts)]))
        assert db.totals() == (counts.sum(), elems)
        if rep != 1:
            assert np.array_equal(data, np.concatenate(words)) and np.array_equal(st, np.concatenate(bits))
    db.close()
