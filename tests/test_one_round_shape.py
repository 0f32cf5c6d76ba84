"""The probes per lane of a resident-pool batch: as few as leave no tile waiting."""
from simd_set_operations_amd import tuning


def test_one_round_shape():
    r = tuning.ONE_ROUND_TILES * 256
    for probes, shape in ((1, "@1"), (r, "@1"), (r + 1, ""), (2 * r, ""), (2 * r + 1, "@2"), (4 * r, "@2")):
        assert tuning.one_round_shape("hip_binary_search@2", probes) == "hip_binary_search" + shape
    assert tuning.one_round_shape("hip_galloping@1", 4 * r + 1) == "hip_galloping@1"
    assert tuning.one_round_shape("hip_branchless_merge@3", 5) == "hip_branchless_merge@3"
