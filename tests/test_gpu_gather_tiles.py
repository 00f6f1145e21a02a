"""mi355_embed_gather_dev at the edges of its tiles: 64 x 32 for few positions, in the order of the grid and by XCD, 64 x 64 for rows of
whole 128-byte lines, 256 x 32 and 256 x 16 for others, x and the table at any float, positions of several sequences in a tile, ids out of range."""
import numpy as np
import pytest

import helpers as H
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def br():
    import ane_amd.bridge as b
    b.init()
    return b


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("V,D,B,S,oob", [(50, 65, 2, 32, 3), (50, 64, 1, 64, 0), (300, 68, 3, 96, 0), (300, 17, 1, 255, 5), (300, 16, 1, 256, 0),
                                         (300, 33, 1, 257, 1), (300, 15, 5, 3, 2), (700, 1023, 130, 127, 9), (700, 1028, 66, 250, 0), (9, 1, 7, 73, 0),
                                         (300, 260, 33, 130, 4), (300, 515, 34, 250, 3), (300, 513, 64, 256, 2)])
def test_gather_tiles(br, V, D, B, S, oob, off):
    print("[case] gather tiles V=%d D=%d B=%d S=%d off=%d" % (V, D, B, S, off), flush=True)
    rng = np.random.default_rng(800)
    ids = rng.integers(0, V, B * S).astype(np.int32)
    ids[rng.choice(B * S, oob, replace=False)] = rng.choice([-1, V, V + 7, -2 ** 31], oob)
    ids = ids.reshape(B, S)
    E = H.normal(801, (V, D)); pre = H.normal(802, (B, D, S))
    put = lambda a: br.DevArray.from_numpy(np.concatenate([np.full(off, 7.0, np.float32), a.ravel(), np.full(3, 7.0, np.float32)]))
    Ed, xd, idd = put(E), put(pre), br.DevArray.from_numpy(ids)
    br.check(br.lib.mi355_embed_gather_dev(xd.ptr + 4 * off, Ed.ptr + 4 * off, idd.ptr, V, D, S, B))
    want, _ = O.embed_lookup(E, ids, out=pre)
    got = xd.numpy()
    assert got[off:off + pre.size].tobytes() == want.tobytes()
    assert np.all(got[:off] == 7.0) and np.all(got[off + pre.size:] == 7.0)
