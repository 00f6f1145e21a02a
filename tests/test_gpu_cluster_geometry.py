"""Clustered norms: a workgroup's strip and sequence come of its number by the strips' reciprocal, its launch tags lane by lane.  Many and
odd numbers of strips and sequences, for every number of members (forced, so that a launch may have more workgroups than compute
units: they run in order and none waits for one behind it for longer than the bound)."""
import pytest

import test_gpu_ragged_rows as R

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def br():
    import ane_amd.bridge as b
    b.init()
    return b


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("members,B,C,S", [(2, 1, 512, 31 * 64), (2, 7, 520, 3 * 128 + 9), (4, 5, 520, 11 * 64 + 5), (4, 16, 1024, 256),
                                           (8, 1, 768, 256), (8, 3, 1000, 9 * 64 + 1), (2, 125, 512, 64), (8, 4, 2048, 7 * 64 + 3)])
def test_strips_and_members(br, members, B, C, S, bf16):
    br.lib.mi355_tune_set(b"rms_cluster", members)
    try:
        R.test_rmsnorm_family_on_rows_of_any_length(br, B, C, S, bf16, 0)
    finally:
        br.lib.mi355_tune_set(b"rms_cluster", 0)


def test_every_reciprocal_divides():
    """cluster * ceil(2^20 / strips) >> 20 is cluster / strips for every pair that a launch can have."""
    for strips in range(1, 1025):
        recip = ((1 << 20) + strips - 1) // strips
        assert all(n * recip >> 20 == n // strips and n * recip < 1 << 32 for n in range(1024)), strips
