"""The way of host arrays to the device and back (host_stage.h): sizes at the ends of its pieces (64 KB), copies (256 KB, 512 KB ...)
and rounds (32 MB), results over their own inputs, rows of a table that end inside a piece, calls far apart (the helper
threads sleep then), and what lies beside the arrays."""
import time

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


def guarded(a):
    """A copy of the array between guard values, and a check that they are still there."""
    buf = np.full(a.size + 2, 3.0, np.float32)
    buf[1:-1] = a.ravel()
    view = buf[1:-1].reshape(a.shape)
    return view, lambda: buf[0] == 3.0 and buf[-1] == 3.0


# floats of an array; a call sends two and gets one back
@pytest.mark.parametrize("n", [1, 63, 16383, 16384, 16385, 65536, 65537, 200001, 3 << 20, (4 << 20) + 17, (11 << 20) + 5])
def test_axpby_sizes(br, n):
    print("[case] host axpby n=%d" % n, flush=True)
    a, a_ok = guarded(H.normal(900, n)); b, b_ok = guarded(H.normal(901, n)); y, y_ok = guarded(np.zeros(n, np.float32))
    want = O.axpby(a, b, 0.3, 0) if hasattr(O, "axpby") else (b * np.float32(0.3) + a)
    for far_apart in (False, True):
        if far_apart:
            time.sleep(0.02)
        y[...] = 0
        br.lib.mi355_axpby(y.ctypes.data, a.ctypes.data, b.ctypes.data, 0.3, n, 0)
        assert y.tobytes() == want.tobytes() and a_ok() and b_ok() and y_ok()
    br.lib.mi355_axpby(a.ctypes.data, a.ctypes.data, b.ctypes.data, 0.3, n, 0)          # over its own input
    assert a.tobytes() == want.tobytes() and a_ok()


@pytest.mark.parametrize("n", [5, 70001, (9 << 20) + 3])
def test_adam_gets_three_arrays_back(br, n):
    print("[case] host adam n=%d" % n, flush=True)
    w, w_ok = guarded(H.normal(910, n, 0, 0.02)); g = H.normal(911, n); m, m_ok = guarded(H.normal(912, n, 0, 0.01))
    v, v_ok = guarded(H.normal(913, n, 0, 0.01) ** 2)
    dev = [br.DevArray.from_numpy(np.array(x)) for x in (w, g, m, v)]
    br.check(br.lib.mi355_adam_update_dev(*[d.ptr for d in dev], n, 7, 3e-4, 0.9, 0.95, 1e-8, 0.1, 1.0, None, 0))
    br.lib.mi355_adam_update(w.ctypes.data, g.ctypes.data, m.ctypes.data, v.ctypes.data, n, 7, 3e-4, 0.9, 0.95, 1e-8, 0.1)
    for host, d, ok in ((w, dev[0], w_ok), (m, dev[2], m_ok), (v, dev[3], v_ok)):
        assert host.tobytes() == d.numpy().tobytes() and ok()


@pytest.mark.parametrize("V,D,S", [(50, 1, 1), (40, 5000, 30), (500, 768, 512), (3000, 1021, 2048)])
def test_rows_of_a_table(br, V, D, S):
    print("[case] host embed_backward V=%d D=%d S=%d" % (V, D, S), flush=True)
    tok = H.zipf_ids(920, S, V).astype(np.uint16)
    dx = H.normal(921, (D, S))
    dE, ok = guarded(H.normal(922, (V, D)))
    want = O.embed_backward(np.array(dE), dx[None], tok.astype(np.int32)[None])
    br.lib.mi355_embed_backward(dE.ctypes.data, dx.ctypes.data, tok.ctypes.data, V, D, S)
    assert dE.tobytes() == want.tobytes() and ok()


def test_loss_and_gradient_come_back_together(br):
    for V, S in ((1, 1), (37, 5), (5000, 256), (40000, 256)):
        print("[case] host cross_entropy V=%d S=%d" % (V, S), flush=True)
        logits = H.normal(930, (V, S), 0, 2.0)
        tok = np.random.default_rng(931).integers(0, V, S).astype(np.uint16)
        dl, ok = guarded(np.zeros((V, S), np.float32))
        loss = br.lib.mi355_cross_entropy_loss(dl.ctypes.data, logits.ctypes.data, tok.ctypes.data, V, S)
        rl, rd = O.cross_entropy(logits, tok.astype(np.int32))
        assert abs(loss - rl) <= 1e-5 * max(abs(rl), 1e-3) and H.err_std(dl, rd) <= 1e-5 and ok()
        over = logits.copy()                            # the gradient over the logits
        br.lib.mi355_cross_entropy_loss(over.ctypes.data, over.ctypes.data, tok.ctypes.data, V, S)
        assert over.tobytes() == dl.tobytes()


def updates(br):
    """Calls that update host arrays: name, the arrays, what makes the call of them."""
    def adam(n):
        w, g, m, v = H.normal(940, n, 0, 0.02), H.normal(941, n), H.normal(942, n, 0, 0.01), H.normal(943, n, 0, 0.01) ** 2
        return [w, m, v], lambda a: br.lib.mi355_adam_update(a[0].ctypes.data, g.ctypes.data, a[1].ctypes.data, a[2].ctypes.data, n, 7, 3e-4, 0.9, 0.95, 1e-8, 0.1)

    def norm(d, S):
        x, dy, w, dx = H.normal(944, (d, S)), H.normal(945, (d, S)), H.normal(946, d, 1, 0.02), np.zeros((d, S), np.float32)
        return [H.normal(947, d)], lambda a: br.lib.mi355_rmsnorm_bwd(dx.ctypes.data, a[0].ctypes.data, dy.ctypes.data, x.ctypes.data, w.ctypes.data, d, S)

    def table(V, D, S):
        tok, dx = np.random.default_rng(948).integers(0, V, S).astype(np.uint16), H.normal(949, (D, S))
        return [H.normal(950, (V, D))], lambda a: br.lib.mi355_embed_backward(a[0].ctypes.data, dx.ctypes.data, tok.ctypes.data, V, D, S)

    def rope(hd, S):
        return [H.normal(951, (4 * hd, S))], lambda a: br.lib.mi355_rope_backward_inplace(a[0].ctypes.data, S, 4 * hd, hd)

    return {"adam small": lambda: adam(70001), "adam rounds": lambda: adam((9 << 20) + 3), "norm": lambda: norm(768, 1000),
            "table": lambda: table(500, 768, 512), "table rounds": lambda: table(2500, 8000, 2000), "rope": lambda: rope(64, 3000)}


@pytest.mark.parametrize("name", ["adam small", "adam rounds", "norm", "table", "table rounds", "rope"])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_arrays_that_are_updated_stay_when_a_copy_back_fails(br, name, mode):
    print("[case] host failure %s mode %d" % (name, mode), flush=True)
    start, call = updates(br)[name]()
    want = [np.array(a) for a in start]
    call(want)
    failures = 0
    br.tune("host_stage", mode)
    try:
        for n in (1, 2, 3, 8, 10 ** 6):          # the copy that fails; the last is never reached
            got = [np.array(a) for a in start]
            br.tune("host_stage_fail", n)
            call(got)
            kept = all(g.tobytes() == a.tobytes() for g, a in zip(got, start))
            failures += kept
            assert kept or (n > 1 and all(g.tobytes() == a.tobytes() for g, a in zip(got, want)))
        assert failures >= 1 and not kept
    finally:
        br.tune("host_stage", 0)
        br.tune("host_stage_fail", 0)


@pytest.mark.parametrize("mode", [1, 2])
def test_without_helper_threads_and_without_pinned_memory(br, mode):
    """The same bits as with both, for each kind of part: inputs, results, a result in an input's place, rows of a table."""
    n, V, S = 300007, 5000, 256
    a, b = H.normal(952, n), H.normal(953, n)
    logits, tok = H.normal(954, (V, S), 0, 2.0), H.zipf_ids(955, S, V).astype(np.uint16)
    got = []
    try:
        for m in (0, mode, 0):
            br.tune("host_stage", m)
            y, dl = np.zeros(n, np.float32), np.zeros((V, S), np.float32)
            br.lib.mi355_axpby(y.ctypes.data, a.ctypes.data, b.ctypes.data, 0.3, n, 0)
            loss = br.lib.mi355_cross_entropy_loss(dl.ctypes.data, logits.ctypes.data, tok.ctypes.data, V, S)
            arrays = [y, dl, np.float32(loss)]
            for make in updates(br).values():
                start, call = make()
                call(start)
                arrays += start
            got.append([x.tobytes() for x in arrays])
    finally:
        br.tune("host_stage", 0)
    assert got[0] == got[1] == got[2]
