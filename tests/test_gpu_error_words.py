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
