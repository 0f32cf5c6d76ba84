"""GPU: the unit scan and tile maps of gather and search batches at the edges of its groups (1,024
pairs), of the one-launch form (8,192 pairs) and of pairs that span no tile, part of one or many."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def announce(msg):
    print(f"[gpu-case] {msg}", flush=True)


def make_pairs(npairs, long_every):
    """CSR pairs over small universes: most sizes 0..9 (some empty), every `long_every`-th pair long."""
    rng = np.random.Generator(np.random.PCG64(npairs * 31 + long_every))
    a, b = [], []
    for p in range(npairs):
        n = 5000 if p % long_every == long_every - 1 else 9
        a.append(np.unique(rng.integers(0, 3 * n, rng.integers(0, n + 1))).astype(np.uint32))
        b.append(np.unique(rng.integers(0, 3 * n, rng.integers(0, n + 1))).astype(np.uint32))
    off = [np.concatenate([[0], np.cumsum([s.size for s in x])]).astype(np.uint64) for x in (a, b)]
    return a, b, np.concatenate(a), off[0], np.concatenate(b), off[1]


@pytest.mark.parametrize("npairs,long_every", [(1, 1), (2, 1), (1023, 500), (1024, 3), (1025, 1025), (8192, 4000),
                                                (8193, 900), (20000, 7001)])
@pytest.mark.parametrize("name", ["hip_galloping", "hip_branchless_merge"])
def test_plan_of_gather_and_search_batches(name, npairs, long_every):
    from simd_set_operations_amd.batch import GatherBatch

    a, b, A, ao, B, bo = make_pairs(npairs, long_every)
    announce(f"plan {name} npairs={npairs} long_every={long_every}")
    gb = GatherBatch(name, A, ao[:-1], ao[1:], B, bo[:-1], bo[1:])
    exp = [np.intersect1d(x, y, assume_unique=True) for x, y in zip(a, b)]
    for _ in range(3):
        gb.run()
        off, cnt, data = gb.results()
        assert np.array_equal(cnt, [e.size for e in exp])
        assert np.array_equal(data, np.concatenate(exp))
        assert np.array_equal(np.diff(off.astype(np.int64)), cnt)
    gb.close()
