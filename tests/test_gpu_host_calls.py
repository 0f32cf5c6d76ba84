"""GPU: host-pointer calls at the edges of how their inputs (read in place, moved by a copy kernel, copied
by the runtime) and results (in pinned memory, on the device) travel."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def announce(msg):
    print(f"[gpu-case] {msg}", flush=True)


def pair(na, nb, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    u = 2 * max(na, nb) + 8
    return tuple(np.sort(rng.choice(u, n, replace=False)).astype(np.uint32) for n in (na, nb))


# inputs of about 96 KiB, 4 MiB and more; results of up to 2 MiB and more
@pytest.mark.parametrize("na,nb", [(0, 5), (1, 1), (12156, 12284), (12156, 12285), (524156, 524284), (524157, 524284),
                                   (524284, 524157), (700000, 900000), (1000, 1100000)])
@pytest.mark.parametrize("name", ["hip_branchless_merge", "hip_galloping"])
def test_host_pairs(name, na, nb):
    from simd_set_operations_amd import _native, intersect
    from simd_set_operations_amd.bsr import BsrVec

    a, b = pair(na, nb, na + nb)
    exp = np.intersect1d(a, b, assume_unique=True)
    announce(f"host pair {name} {na} {nb}")
    out = np.full(min(na, nb) + 4, 7, np.uint32)
    for _ in range(2):
        n = intersect.intersect2_c(name, a, b, out)
        assert n == exp.size and np.array_equal(out[:n], exp) and (out[n:] == 7).all()
    assert intersect.intersect2_c(name, a, b) == exp.size
    if exp.size:
        with pytest.raises(_native.SetopsError):
            intersect.intersect2_c(name, a, b, np.zeros(exp.size - 1, np.uint32))
    got, elems = intersect.intersect2_bsr(name + "_bsr", BsrVec.from_sorted(a), BsrVec.from_sorted(b))
    assert elems == exp.size and np.array_equal(got.to_sorted_set(), exp)


@pytest.mark.parametrize("name", ["hip_branchless_merge", "hip_galloping", "hip_small_adaptive"])
@pytest.mark.parametrize("sizes", [(3, 4, 5), (500, 800, 900, 2000), (30000, 40000, 200000, 250000, 300000),
                                   (30000, 40000, 400000, 450000, 500000), (600000, 700000, 800000), (40, 0, 90),
                                   (900, 1000) + (1100,) * 12])
def test_host_ksets(name, sizes):
    from simd_set_operations_amd import intersect

    rng = np.random.Generator(np.random.PCG64(sum(sizes)))
    u = 2 * max(sizes) + 8
    common = rng.choice(u, min(sizes) // 2, replace=False)
    sets = [np.unique(np.concatenate([common, rng.choice(u, n, replace=False)]) if n else common[:0]).astype(np.uint32)
            for n in sizes]
    announce(f"host k-set {name} {sizes}")
    exp = oracle.svs("branchless_merge", sets)
    for _ in range(2):
        assert np.array_equal(intersect.run_kset(sets, name), exp)
