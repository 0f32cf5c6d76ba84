"""GPU: search tiles whose first pair's probes all fall into a gap of its larger set (an empty window, at the
first staged word), before pairs whose windows are staged."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def announce(msg):
    print(f"[gpu-case] {msg}", flush=True)


def make_pairs(probes, gap_at):
    """Pair 0: `probes` probes, those from `gap_at` on between two neighbours of the larger set (64 apart, so
    that BSR words differ too); then small pairs with a few common elements."""
    small = np.arange(probes, dtype=np.uint32) * np.uint32(64)
    large = np.concatenate([small[:gap_at:2], np.arange(3 * probes, dtype=np.uint32) * np.uint32(64) + small[-1] + np.uint32(640)])
    pairs = [(small, large)]
    for k in range(40):
        pairs.append((np.arange(3 + k, dtype=np.uint32) * np.uint32(96), np.arange(50 + k, dtype=np.uint32) * np.uint32(64)))
    return pairs


@pytest.mark.parametrize("name", ["hip_galloping", "hip_binary_search@1", "hip_simd_galloping@2", "hip_galloping_bsr"])
@pytest.mark.parametrize("probes,gap_at", [(300, 100), (600, 256), (600, 512), (1500, 1024), (2100, 5)])
@pytest.mark.parametrize("indexed", [False, True])
def test_probes_in_a_gap(name, probes, gap_at, indexed):
    from simd_set_operations_amd.batch import DeviceBatch
    from simd_set_operations_amd.bsr import BsrVec

    pairs = make_pairs(probes, gap_at)
    exp = [oracle.branchless_merge(a, b) for a, b in pairs]
    announce(f"gap {name} {probes} {gap_at} indexed={indexed}")
    sides, kw = [[p[s] for p in pairs] for s in (0, 1)], {}
    if name.endswith("_bsr"):
        vecs = [[BsrVec.from_sorted(x) for x in s] for s in sides]
        kw = {f"{n}_states": np.concatenate([v.states for v in s]) for n, s in zip("AB", vecs)}
        sides, exp = [[v.bases for v in s] for s in vecs], [BsrVec.from_sorted(e).bases for e in exp]
    off = [np.concatenate([[0], np.cumsum([x.size for x in s])]).astype(np.uint64) for s in sides]
    db = DeviceBatch(name, np.concatenate(sides[0]), off[0], np.concatenate(sides[1]), off[1], **kw)
    if indexed:
        db.index_b()
    for _ in range(2):
        db.run()
        o, cnt, data = db.results()[:3]
        assert np.array_equal(cnt, [e.size for e in exp])
        assert np.array_equal(data, np.concatenate(exp))
    db.close()
