"""Clustered norms: a workgroup's strip and sequence come of its number by the strips' reciprocal (cluster_words.h, which
test_cluster_words.py checks for every launch), its launch tags lane by lane.  Many and odd numbers of strips and sequences, for every
number of members, forced, so that a launch may have more workgroups than compute units: they run in order and none waits for one
behind it for longer than the bound.  Where all are resident no wait may expire: a workgroup with a wrong tag or partner would take the
way of an expired wait, to the same values."""
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
    strips = -(-S // (128 if bf16 else 64))
    expired = br.exchange_fallbacks()[0]
    br.lib.mi355_tune_set(b"rms_cluster", members)
    try:
        R.test_rmsnorm_family_on_rows_of_any_length(br, B, C, S, bf16, 0)
    finally:
        br.lib.mi355_tune_set(b"rms_cluster", 0)
    if members * strips * B <= br.device_info()[2]:
        assert br.exchange_fallbacks()[0] == expired
