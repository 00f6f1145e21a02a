"""The plan of the column form of the embedding gradient: tokens that all fall into one workgroup's group (distinct ones and equal ones,
64 and 512 to a wave and one more or less), more entries than one pass ranks, blocks that are nearly empty, more blocks than one
pair of launches takes, and calls with other numbers of blocks in turn.  The bits of the reference loop."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu

BLOCK = 8192


@pytest.fixture(scope="module")
def br():
    import ane_amd.bridge as b
    b.init()
    yield b
    b.tune("scatter_cols", 0)


def scatter(br, ids, V, D=2):
    N = ids.size
    print("[case] scatter plan N=%d V=%d" % (N, V), flush=True)
    br.tune("scatter_cols", 1)
    dx, dE = H.normal(911, (1, D, N)), H.normal(912, (V, D))
    Ed, xd, idd = br.DevArray.from_numpy(dE), br.DevArray.from_numpy(dx), br.DevArray.from_numpy(ids.astype(np.int32))
    br.check(br.lib.mi355_embed_scatter_add_dev(Ed.ptr, xd.ptr, idd.ptr, V, D, N, 1))
    keep = (ids >= 0) & (ids < V)
    want = dE.copy()
    np.add.at(want, ids[keep], dx[0].T[keep])          # one addition after the other, in order of position
    assert Ed.numpy().tobytes() == want.tobytes()


def one_group(V, nblk, g=3):
    """the tokens that one workgroup of a block ranks"""
    groups = max(16, min(128, 256 // nblk))
    k = np.arange(V, dtype=np.uint64)
    h = (((k * 0x9E3779 & 0xffffffff) >> 8 & 0xffff) * groups) >> 16
    return np.flatnonzero(h == g)


@pytest.mark.parametrize("V", [(1 << 19) - 1, 32000])
@pytest.mark.parametrize("nblk", [1, 2, 5])
def test_tokens_of_one_group(br, V, nblk):
    pool, rng = one_group(V, nblk), np.random.default_rng(nblk)
    N = nblk * BLOCK
    scatter(br, np.resize(rng.permutation(pool), N), V)              # as many distinct ones as there are: several passes of entries
    scatter(br, np.resize(pool[:700], N), V)                         # 700 tokens over and over
    scatter(br, rng.choice(pool[:40], N), V)
    ids = np.full(N, -1, np.int64)                                   # and few positions of a wave's 512, the others elsewhere
    for wave, n in enumerate([0, 1, 11, 12, 13, 63, 64, 65, 127, 128, 129, 511, 512]):
        at = wave * 512 + np.sort(rng.permutation(512)[:n])
        ids[at] = np.resize(pool[:max(1, n // (1 + wave % 3))], n)
    scatter(br, ids, V)


@pytest.mark.parametrize("N", [513, 8191, 8192, 8193, 16384 + 1, 5 * 8192 + 511])
def test_equal_and_distinct_tokens(br, N):
    rng = np.random.default_rng(N)
    V = 60000
    scatter(br, np.full(N, V - 1), V)
    scatter(br, np.full(N, V), V)                                    # none in range
    scatter(br, rng.permutation(V)[:N], V)
    ids = np.minimum(rng.zipf(1.1, N) - 1, V - 1)
    ids[rng.choice(N, 9, replace=False)] = [-1, V, V + 1, -2 ** 31, 2 ** 31 - 1, -7, V, V, -1]
    scatter(br, ids, V)
    scatter(br, rng.integers(0, 1 << 15, N), 1 << 15)
    scatter(br, np.zeros(N, np.int64), 1)


def test_more_blocks_than_a_launch_takes(br):
    rng = np.random.default_rng(64)
    for N in (64 * BLOCK, 64 * BLOCK + 5, 700, 66 * BLOCK + 4099, 3 * BLOCK):
        scatter(br, np.minimum(rng.zipf(1.2, N) - 1, 9999), 10000, D=1)


@pytest.mark.parametrize("recorded", [False, True])
@pytest.mark.parametrize("nblk", [1, 3])
def test_a_plan_whose_sums_are_not_launched(br, nblk, recorded):
    """An error that another call has left behind ends a call between its plan and its sums; the calls after it start from cleared counts."""
    rng, V = np.random.default_rng(nblk), 5000
    N = nblk * BLOCK - 3
    texts = [np.minimum(rng.zipf(1.2, N) - 1, V - 1) for _ in range(3)]
    for ids in texts:
        scatter(br, ids, V)
    Ed, xd, idd = br.DevArray((V, 2)), br.DevArray((2, N)), br.DevArray.from_numpy(texts[0].astype(np.int32))
    unrecorded = [br.Event(), br.Event()]
    for times in range(1, 4):
        if recorded:
            br.check(br.lib.mi355_graph_begin())
        for _ in range(times):
            assert br.lib.mi355_event_elapsed_ms(unrecorded[0].handle, unrecorded[1].handle) < 0
            assert br.lib.mi355_embed_scatter_add_dev(Ed.ptr, xd.ptr, idd.ptr, V, 2, N, 1) == -1 and "plan" in br.last_error()
        if recorded:
            graph = br.lib.mi355_graph_end()
            assert graph
            for _ in range(3):
                br.check(br.lib.mi355_graph_launch(graph))
                scatter(br, texts[times - 1], V)
            br.lib.mi355_graph_free(graph)
        for ids in texts:
            scatter(br, ids, V)
