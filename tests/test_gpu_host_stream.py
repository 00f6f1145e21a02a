"""Elementwise calls on host arrays, whose chunks are packed, computed over the link and unpacked at the same time: sizes at the ends of
chunks (16384, 21504, 32768 values ...) and of a round, results over their own inputs, arrays that overlap otherwise or lie
in a resident table (which take the other way), and what lies beside the arrays.  The bytes are those of the device call."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def br():
    import ane_amd.bridge as b
    b.init()
    return b


def guarded(n):
    buf = np.full(n + 2, 3.0, np.float32)
    return buf[1:-1], lambda: buf[0] == 3.0 and buf[-1] == 3.0


def on_device(br, name, outs, ins, *rest):
    o, i = [br.DevArray(ins[0].size) for _ in range(outs)], [br.DevArray.from_numpy(x) for x in ins]
    br.check(getattr(br.lib, name)(*[x.ptr for x in o + i], *rest))
    return [x.numpy() for x in o]


SIZES = [1, 3, 1023, 16384, 21504, 32769, 65536 + 1024, 131071, 700001, (2 << 20) + 1, (2796202 & ~4095) + 1]


@pytest.mark.parametrize("n", SIZES)
def test_results_in_arrays_of_their_own(br, n):
    print("[case] host stream n=%d" % n, flush=True)
    a, b, c = H.normal(960, n), H.normal(961, n), H.normal(962, n)
    p = lambda x: x.ctypes.data
    (y, y_ok), (z, z_ok) = guarded(n), guarded(n)
    br.lib.mi355_swiglu_fwd(p(y), p(a), p(b), n)
    assert y.tobytes() == on_device(br, "mi355_swiglu_fwd_dev", 1, [a, b], n)[0].tobytes() and y_ok()
    br.lib.mi355_swiglu_bwd(p(y), p(z), p(a), p(b), p(c), n)
    want = on_device(br, "mi355_swiglu_bwd_dev", 2, [a, b, c], n)
    assert y.tobytes() == want[0].tobytes() and z.tobytes() == want[1].tobytes() and y_ok() and z_ok()
    for mode in range(3):
        br.lib.mi355_axpby(p(y), p(a), p(b), 0.3, n, mode)
        assert y.tobytes() == on_device(br, "mi355_axpby_dev", 1, [a, b], 0.3, n, mode)[0].tobytes() and y_ok()


@pytest.mark.parametrize("n", SIZES)
def test_adam(br, n):
    print("[case] host stream adam n=%d" % n, flush=True)
    arrays = [guarded(n) for _ in range(4)]
    for k, (x, _) in enumerate(arrays):
        x[...] = H.normal(970 + k, n)
    arrays[3][0][...] **= 2
    dev = [br.DevArray.from_numpy(x) for x, _ in arrays]
    rest = (n, 7, 3e-4, 0.9, 0.95, 1e-8, 0.1)
    br.check(br.lib.mi355_adam_update_dev(*[d.ptr for d in dev], *rest, 1.0, None, 0))
    br.lib.mi355_adam_update(*[x.ctypes.data for x, _ in arrays], *rest)
    for (x, ok), d in zip(arrays, dev):
        assert x.tobytes() == d.numpy().tobytes() and ok()


@pytest.mark.parametrize("shift", [0, 1, -1, 40000, -40000])
def test_results_over_inputs(br, shift):
    """y = 0.3 b + a with y `shift` values behind a or b: every input is read before any result is written"""
    n = 300007
    for over in (0, 1):
        buf = H.normal(980, n + 80000)
        x, other = buf[40000:40000 + n], H.normal(981, n)
        y = buf[40000 + shift:40000 + shift + n]
        a, b = (x, other) if over == 0 else (other, x)
        want = b * np.float32(0.3) + a
        br.lib.mi355_axpby(y.ctypes.data, a.ctypes.data, b.ctypes.data, 0.3, n, 0)
        assert y.tobytes() == want.tobytes()


@pytest.mark.parametrize("n", [300007, (3 << 20) + 5])       # several chunks of one round, two rounds
@pytest.mark.parametrize("fail", [1, 2, 4])
def test_results_over_inputs_stay_when_a_chunk_does_not_come_back(br, n, fail):
    x, other, h1, h3 = H.normal(985, n), H.normal(986, n), H.normal(987, n), H.normal(988, n)
    was = [a.copy() for a in (x, h1, h3)]
    p = lambda a: a.ctypes.data
    try:
        br.tune("host_stage_fail", fail)
        br.lib.mi355_axpby(p(x), p(x), p(other), 0.3, n, 0)
        br.lib.mi355_swiglu_bwd(p(h1), p(h3), p(other), p(h1), p(h3), n)
    finally:
        br.tune("host_stage_fail", 0)
    for a, b in zip((x, h1, h3), was):
        assert a.tobytes() == b.tobytes()


def test_results_over_inputs_stay_whichever_chunk_does_not_come_back(br):
    """Every chunk of a call of one round and of two, the second round's among them, whose inputs stand where the first one has written
    its results by then: the old values come from the log."""
    p = lambda a: a.ctypes.data

    def calls(n):
        x, y, z, w = H.normal(1020, n), H.normal(1021, n), H.normal(1022, n), H.normal(1023, n) ** 2
        yield [x], lambda: br.lib.mi355_axpby(p(x), p(x), p(y), 0.3, n, 0)
        yield [x, z], lambda: br.lib.mi355_swiglu_bwd(p(x), p(z), p(y), p(x), p(z), n)
        yield [x, y, w], lambda: br.lib.mi355_adam_update(p(x), p(z), p(y), p(w), n, 7, 3e-4, 0.9, 0.95, 1e-8, 0.1)

    chunks = {}
    try:
        # values of the round of a pinned block of 32 MB, by the arrays of the calls
        for n in (None, (3 << 20) + 5):
            for k, parts in enumerate((3, 5, 4)):
                m = n or ((32 << 20) // (4 * parts) & ~4095)
                arrays, call = list(calls(m))[k]
                was = [a.tobytes() for a in arrays]
                fail = 0
                while [a.tobytes() for a in arrays] == was:
                    fail += 1
                    assert fail <= 100
                    br.tune("host_stage_fail", fail)
                    call()
                chunks[n, k] = fail - 1
    finally:
        br.tune("host_stage_fail", 0)
    for k in range(3):
        print("[case] chunks of a round, of two: %d %d" % (chunks[None, k], chunks[(3 << 20) + 5, k]), flush=True)
        assert 2 < chunks[None, k] <= 32 and chunks[(3 << 20) + 5, k] > chunks[None, k]


@pytest.mark.parametrize("fail", [1, 2, 5])
def test_nothing_is_written_when_a_chunk_is_not_launched(br, fail):
    """results over inputs and results in arrays of their own alike"""
    n = 700001
    a, b, c = H.normal(1000, n), H.normal(1001, n), H.normal(1002, n) ** 2
    p = lambda x: x.ctypes.data
    y, z = np.full(n, 3.0, np.float32), np.full(n, 4.0, np.float32)
    calls = [lambda: br.lib.mi355_axpby(p(y), p(a), p(b), 0.3, n, 0), lambda: br.lib.mi355_axpby(p(y), p(a), None, 0.3, n, 1),
             lambda: br.lib.mi355_axpby(p(a), p(a), p(b), 0.3, n, 0), lambda: br.lib.mi355_swiglu_fwd(p(y), p(a), p(b), n),
             lambda: br.lib.mi355_swiglu_bwd(p(y), p(z), p(a), p(b), p(c), n), lambda: br.lib.mi355_swiglu_bwd(p(b), p(z), p(a), p(b), p(c), n),
             lambda: br.lib.mi355_adam_update(p(a), p(b), p(y), p(c), n, 7, 3e-4, 0.9, 0.95, 1e-8, 0.1)]
    was = [x.tobytes() for x in (a, b, c, y, z)]
    try:
        br.tune("host_stage_fail", -fail)
        for k, call in enumerate(calls):
            call()
            assert "refused" in br.last_error() and [x.tobytes() for x in (a, b, c, y, z)] == was, k
            br.lib.mi355_axpby(None, None, None, 0.3, n, 0)                       # (another error's text)
    finally:
        br.tune("host_stage_fail", 0)


def test_weights_that_a_table_holds(br):
    """the table that an update steps is looked up on the device afterwards, with the values that the update left"""
    V, D, S = 300, 64, 50
    w, g, m, v = H.normal(990, (V, D)), H.normal(991, (V, D)), H.normal(992, (V, D)), H.normal(993, (V, D)) ** 2
    tok = np.random.default_rng(994).integers(0, V, S).astype(np.uint16)
    x = np.zeros((D, S), np.float32)
    for _ in range(2):
        br.lib.mi355_embed_lookup(x.ctypes.data, w.ctypes.data, tok.ctypes.data, V, D, S)
        assert x.tobytes() == np.ascontiguousarray(w[tok].T).tobytes()
        br.lib.mi355_adam_update(w.ctypes.data, g.ctypes.data, m.ctypes.data, v.ctypes.data, V * D, 3, 3e-4, 0.9, 0.95, 1e-8, 0.1)
    br.lib.mi355_embed_lookup(x.ctypes.data, w.ctypes.data, tok.ctypes.data, V, D, S)
    assert x.tobytes() == np.ascontiguousarray(w[tok].T).tobytes()
    br.lib.mi355_host_table_invalidate(w.ctypes.data)
