"""The ordered scatter-add in its column form where sequences are of any length, dx starts at any 4-byte boundary and
positions are many: bit-identical to the reference loop, and taken from the second call of a shape on."""
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


@pytest.mark.parametrize("V,D,B,S,shift", [
    (500, 6, 1, 513, 0),          # one position more than the one-launch kernel; the last group has one position
    (500, 770, 171, 3, 0),        # groups of four positions over two sequences, each; 257 workgroups
    (40, 5, 600, 1, 0),           # ... over four
    (900, 1024, 42, 197, 0),      # blocks of 8192 positions that end inside a sequence
    (900, 33, 8193, 1, 0),        # a second block of one position
    (3000, 64, 3, 256, 1),        # whole sequences at an odd element
    (3000, 64, 5, 4097, 3),       # both, 20485 positions
])
def test_column_form_at_any_length_and_alignment(br, V, D, B, S, shift):
    ids = H.zipf_ids(7, B * S, V).astype(np.int32).reshape(B, S)
    ids[0, 0] = V                                       # skipped
    dx = H.normal(8, (B, D, S)); dE0 = H.normal(9, (V, D))
    dxd = br.DevArray.from_numpy(np.concatenate([np.zeros(shift, np.float32), dx.ravel()]))
    dEd, idd = br.DevArray.from_numpy(dE0), br.DevArray.from_numpy(ids)
    br.tune("scatter_cols", 1)
    try:
        br.check(br.lib.mi355_embed_scatter_add_dev(dEd.ptr, dxd.ptr + 4 * shift, idd.ptr, V, D, S, B))
    finally:
        br.tune("scatter_cols", 0)
    assert dEd.numpy().tobytes() == O.embed_backward(dE0, dx, ids).tobytes()


@pytest.mark.parametrize("B,S", [(80, 256), (131, 125)])        # 20480 positions; 16375 in sequences of an odd length
def test_form_is_learned_from_the_last_call_of_the_shape(br, B, S):
    V, D = 32000, 96
    text = H.zipf_ids(11, B * S, V).astype(np.int32).reshape(B, S)
    flat = np.random.default_rng(12).integers(0, V, (B, S)).astype(np.int32)
    dx = H.normal(13, (B, D, S)); dE0 = H.normal(14, (V, D))
    dxd = br.DevArray.from_numpy(dx)
    form = lambda: br.lib.mi355_embed_scatter_add_form(V, D, S, B, 1)

    def call(ids):
        dEd = br.DevArray.from_numpy(dE0)
        idd = br.DevArray.from_numpy(ids)
        br.check(br.lib.mi355_embed_scatter_add_dev(dEd.ptr, dxd.ptr, idd.ptr, V, D, S, B))
        br.sync()
        assert dEd.numpy().tobytes() == O.embed_backward(dE0, dx, ids).tobytes()

    assert form() == -1                 # nothing known yet
    call(text)
    assert form() == 1
    call(text)
    call(np.roll(text, 1))
    assert form() == 1
    call(flat)
    assert form() == -1                 # ids that hardly repeat: rows, and there it stays
    call(flat)
    assert form() == -1
    call(text)
    assert form() == 1


def test_graph_records_a_short_sequence_of_any_length_into_a_large_vocabulary(br):
    """Up to 512 positions the plan and the sums are one launch, which takes any length; the row form of so large a
    vocabulary would call the library sort, which cannot be recorded."""
    L = br.lib
    V, D, B, S = 300000, 8, 2, 197
    ids = H.zipf_ids(15, B * S, V).astype(np.int32).reshape(B, S)
    dx = H.normal(16, (B, D, S)); dE0 = H.normal(17, (V, D))
    dEd, idd, dxd = br.DevArray.from_numpy(dE0), br.DevArray.from_numpy(ids), br.DevArray.from_numpy(dx)
    br.sync()
    br.check(L.mi355_graph_begin())
    got = L.mi355_embed_scatter_add_dev(dEd.ptr, dxd.ptr, idd.ptr, V, D, S, B)
    why = br.last_error()
    g = L.mi355_graph_end()
    try:
        assert got == 0 and g, why
        want = dE0
        for _ in range(3):
            br.check(L.mi355_graph_launch(g))
            want = O.embed_backward(want, dx, ids)
            br.sync()
            assert dEd.numpy().tobytes() == want.tobytes()
    finally:
        if g: L.mi355_graph_free(g)


@pytest.mark.parametrize("V,D,B,S,shift", [(300000, 8, 5, 197, 1), (3000, 12, 27, 607, 0)])    # 985 positions; 16389
def test_graph_records_sequences_of_any_length_that_the_library_would_sort(br, V, D, B, S, shift):
    """The column form reads sequences of any length at any element, so it stands in for the library sort there too."""
    L = br.lib
    ids = H.zipf_ids(18, B * S, V).astype(np.int32).reshape(B, S)
    dx = H.normal(19, (B, D, S)); dE0 = H.normal(20, (V, D))
    dEd, idd = br.DevArray.from_numpy(dE0), br.DevArray.from_numpy(ids)
    dxd = br.DevArray.from_numpy(np.concatenate([np.zeros(shift, np.float32), dx.ravel()]))
    call = lambda e: L.mi355_embed_scatter_add_dev(e.ptr, dxd.ptr + 4 * shift, idd.ptr, V, D, S, B)
    eager = br.DevArray.from_numpy(dE0)
    br.check(call(eager))                               # also sizes the workspace
    br.sync()
    br.check(L.mi355_graph_begin())
    got = call(dEd)
    why = br.last_error()
    g = L.mi355_graph_end()
    try:
        assert got == 0 and g, why
        want = dE0
        for _ in range(3):
            br.check(L.mi355_graph_launch(g))
            want = O.embed_backward(want, dx, ids)
            assert dEd.numpy().tobytes() == want.tobytes()
            br.check(call(eager))                       # the program's own eager work between replays
            br.sync()
        assert eager.numpy().tobytes() == O.embed_backward(want, dx, ids).tobytes()
    finally:
        if g: L.mi355_graph_free(g)
