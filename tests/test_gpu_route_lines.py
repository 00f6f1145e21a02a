"""Both sides of lines at which the clustered norms and the fp32 QK-norm + RoPE forward change their kernel: members whose rows fill
half of a tile, a row more and fewer; tensors from which on rows of any length are read past the caches; eight rows per lane
with the residual; rows of a head without conditions, by the workgroups to one of 256 compute units and the fill of a strip."""
import pytest

import test_gpu_qk_whole_tiles as Q
import test_gpu_ragged_rows as R

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def br():
    import ane_amd.bridge as b
    b.init()
    return b


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("B,C,S", [(1, 512, 32), (2, 512, 33), (1, 513, 100), (3, 520, 64), (1, 1024, 54), (1, 1032, 54),     # rows of a member
                                   (11, 512, 100), (12, 512, 100), (31, 768, 100), (32, 768, 100), (33, 520, 65),             # clusters, not large enough
                                   (15, 1000, 100), (15, 1000, 99), (30, 1000, 101), (31, 1000, 97),                          # values of a tensor
                                   (40, 1024, 100), (50, 1000, 67), (64, 768, 33)])                                           # rows per lane
def test_norm_clusters(br, B, C, S, bf16):
    R.test_rmsnorm_family_on_rows_of_any_length(br, B, C, S, bf16, 1)


@pytest.mark.parametrize("hd,B,S", [(64, 32, 33), (64, 33, 33), (64, 32, 100), (64, 33, 100), (64, 40, 81), (64, 41, 81), (128, 24, 100), (128, 25, 100),
                                    (128, 32, 80), (128, 33, 80), (128, 40, 70), (128, 41, 70), (128, 32, 64), (128, 33, 63)])
def test_qknorm_rope_rows(br, hd, B, S):
    Q.test_qknorm_rope_ragged_strips(br, hd, 8, 8, B, S, False)
