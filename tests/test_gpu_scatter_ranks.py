"""The ordered embedding gradient by columns around 32768 positions, where a workgroup begins to rank 128 positions instead of 64:
the same bits as the reference loop, ids out of range skipped, last workgroups with 1, 63, 64, 65 and 127 positions."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def br():
    import ane_amd.bridge as b
    b.init()
    yield b
    b.tune("scatter_cols", 0)


@pytest.mark.parametrize("V", [3, 700, 40000])
@pytest.mark.parametrize("N", [32768, 32769, 32831, 32832, 32833, 32895, 40960, 49153])
def test_scatter_ranks(br, N, V):
    print("[case] scatter ranks N=%d V=%d" % (N, V), flush=True)
    D = 5
    rng = np.random.default_rng(820)
    ids = np.minimum(rng.zipf(1.2, N) - 1, V - 1).astype(np.int32) if V > 3 else rng.integers(0, V, N).astype(np.int32)
    ids[rng.choice(N, 9, replace=False)] = [-1, V, V + 1, -2 ** 31, 2 ** 31 - 1, -7, V, V, -1]
    dx, dE = H.normal(821, (1, D, N)), H.normal(822, (V, D))
    br.tune("scatter_cols", 1)
    Ed, xd, idd = br.DevArray.from_numpy(dE), br.DevArray.from_numpy(dx), br.DevArray.from_numpy(ids)
    br.check(br.lib.mi355_embed_scatter_add_dev(Ed.ptr, xd.ptr, idd.ptr, V, D, N, 1))
    keep = (ids >= 0) & (ids < V)
    want = dE.copy()
    np.add.at(want, ids[keep], dx[0].T[keep])          # one addition after the other, in order of position
    assert Ed.numpy().tobytes() == want.tobytes()
