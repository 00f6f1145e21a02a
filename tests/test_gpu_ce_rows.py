"""The one-launch softmax cross-entropy on rows of any length and every number of row steps: row counts around the
variants' limits (8 and 16 steps of 64 rows in each of the members, and the LDS rows beyond), strips that do not divide the
row, short last groups, rows of whole 128-byte lines and others, tensors that start within a line."""
import numpy as np
import pytest

import helpers as H
import oracle as O

pytestmark = pytest.mark.gpu


def run(br, logits, tgt, bf16, scale, off=0, one_launch=1):
    """off: elements between the start of an allocation and the tensor, on both sides; one_launch: the knob's value"""
    dt = np.uint16 if bf16 else np.float32
    raw = O.cvt_f32_bf16(logits) if bf16 else logits
    ld = br.DevArray.from_numpy(np.concatenate([np.zeros(off, dt), raw.ravel()]))
    td, dl, loss = br.DevArray.from_numpy(tgt), br.DevArray(off + logits.size, dt), br.DevArray(1)
    fn, at = br.lib.mi355_softmax_ce_bf16_dev if bf16 else br.lib.mi355_softmax_ce_dev, off * dt().itemsize
    br.tune("ce_resident", one_launch)
    try:
        br.check(fn(dl.ptr + at, loss.ptr, ld.ptr + at, td.ptr, logits.shape[0], logits.shape[1], scale))
    finally:
        br.tune("ce_resident", 0)
    return loss.numpy().tobytes(), dl.numpy()[off:].reshape(logits.shape)


# 64 members at S = 197 and 52, 51 at S = 300, 16 at S = 1000: 64 * 512 = 32768 rows are the last that fit 8 steps, 65536 the
# last that fit 16; (1, 4) and (65, 7): members without rows, one short group
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("V,S", [(1, 4), (65, 7), (32768, 197), (32769, 52), (65600, 37), (9000, 1000), (20001, 999), (26113, 300), (110000, 65)])
def test_one_launch_on_rows_of_any_length(br, V, S, bf16):
    print("[case] one-launch ce V=%d S=%d bf16=%d" % (V, S, bf16), flush=True)
    logits = H.normal(400, (V, S), 0, 2.0)
    if bf16:
        logits = O.cvt_bf16_f32(O.cvt_f32_bf16(logits))
    tgt = np.random.default_rng(401).integers(0, V, S).astype(np.int32)
    tgt[0] = V - 1; tgt[S - 1] = 0
    if S > 4:
        tgt[1] = V; tgt[S - 2] = -1                       # out-of-range targets are skipped
    rl, rd = O.cross_entropy(logits, tgt, 256.0)
    expired = br.exchange_fallbacks()[1]
    loss, dl = run(br, logits, tgt, bf16, 256.0)
    assert br.exchange_fallbacks()[1] == expired
    got = O.cvt_bf16_f32(dl) if bf16 else dl
    assert abs(float(np.frombuffer(loss, np.float32)[0]) - rl) <= 1e-5 * max(abs(rl), 1e-3)
    assert H.rel_err(got, rd) <= (5e-3 if bf16 else 1e-5)         # the parity bars of the two storage types
    try:
        br.tune("xch_take_nothing", 1)                            # every partner's partial recomputed: the same bits
        loss2, dl2 = run(br, logits, tgt, bf16, 256.0)
        assert br.exchange_fallbacks()[1] > expired
    finally:
        br.tune("xch_take_nothing", 0)
    assert loss2 == loss and dl2.tobytes() == dl.tobytes()


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("V,S", [(9000, 256), (70000, 128)])
def test_rows_of_whole_lines_at_any_element(br, V, S, bf16):
    """The same bits wherever the tensors start: past the caches on a line or half a line, through them elsewhere."""
    logits = H.normal(402, (V, S), 0, 2.0)
    tgt = np.random.default_rng(403).integers(0, V, S).astype(np.int32)
    loss, dl = run(br, logits, tgt, bf16, 1.0)
    rl, rd = O.cross_entropy(O.cvt_bf16_f32(O.cvt_f32_bf16(logits)) if bf16 else logits, tgt, 1.0)
    assert H.rel_err(O.cvt_bf16_f32(dl) if bf16 else dl, rd) <= (5e-3 if bf16 else 1e-5)
    assert abs(float(np.frombuffer(loss, np.float32)[0]) - rl) <= 1e-5 * abs(rl)
    for off in (1, 4, 16, 64):
        loss2, dl2 = run(br, logits, tgt, bf16, 1.0, off)
        assert loss2 == loss and dl2.tobytes() == dl.tobytes(), off


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("S", [37, 64])
def test_a_single_strip_of_a_large_vocabulary_takes_three_launches(br, S, bf16):
    """14 row steps of 64 rows in 64 members are the last that one launch takes there (fp32), and the other form needs no
    call that sizes a workspace before a graph is recorded, as the one launch does not."""
    for V in (57344, 57345):
        logits = H.normal(404, (V, S), 0, 2.0)
        tgt = np.random.default_rng(405).integers(0, V, S).astype(np.int32)
        want = run(br, logits, tgt, bf16, 1.0, 0, 0)
        rl, rd = O.cross_entropy(O.cvt_bf16_f32(O.cvt_f32_bf16(logits)) if bf16 else logits, tgt, 1.0)
        assert H.rel_err(O.cvt_bf16_f32(want[1]) if bf16 else want[1], rd) <= (5e-3 if bf16 else 1e-5)
        assert abs(float(np.frombuffer(want[0], np.float32)[0]) - rl) <= 1e-5 * abs(rl)
        expired = br.exchange_fallbacks()[1]
        try:
            br.tune("xch_take_nothing", 1)                    # counted by the one launch only
            got = run(br, logits, tgt, bf16, 1.0, 0, 0)
        finally:
            br.tune("xch_take_nothing", 0)
        assert (br.exchange_fallbacks()[1] > expired) == (bf16 or V == 57344)
        assert got[0] == want[0] and got[1].tobytes() == want[1].tobytes()
    if bf16:
        return
    L = br.lib
    ld, td, dl, loss = br.DevArray.from_numpy(logits), br.DevArray.from_numpy(tgt), br.DevArray((V, S)), br.DevArray(1)
    ws = L.mi355_workspace_size()
    br.check(L.mi355_graph_begin())
    br.check(L.mi355_softmax_ce_dev(dl.ptr, loss.ptr, ld.ptr, td.ptr, V, S, 1.0))
    g = L.mi355_graph_end()
    assert g, br.last_error()
    assert L.mi355_workspace_size() == ws
    for _ in range(3):
        br.check(L.mi355_graph_launch(g))
        assert loss.numpy().tobytes() == want[0] and dl.numpy().tobytes() == want[1].tobytes()
        run(br, logits[:40000], np.zeros(S, np.int32), False, 2.0, 0, -1)         # other values in the scratch
        br.check(L.mi355_buf_zero(dl.handle))
        br.sync()
    L.mi355_graph_free(g)


@pytest.mark.parametrize("V,S,bf16", [(65536, 1000, False), (262144, 5, True)])
def test_one_launch_up_to_64_row_steps(br, V, S, bf16):
    """16 members at S = 1000, 64 at S = 5: the last V that one launch takes, and the next, which are three; the two forms
    sum in different orders and agree within the parity bar."""
    for v, one in ((V, True), (V + 1, False)):
        logits = np.random.default_rng(406).standard_normal((v, S), dtype=np.float32)
        tgt = np.random.default_rng(407).integers(0, v, S).astype(np.int32)
        loss, dl = run(br, logits, tgt, bf16, 1.0, 0, -1)
        try:
            br.tune("xch_take_nothing", 1)                    # counted by the one launch only
            expired = br.exchange_fallbacks()[1]
            loss1, dl1 = run(br, logits, tgt, bf16, 1.0, 0, 0)
        finally:
            br.tune("xch_take_nothing", 0)
        assert (br.exchange_fallbacks()[1] > expired) == one
        assert abs(np.frombuffer(loss1, np.float32)[0] / np.frombuffer(loss, np.float32)[0] - 1) <= 1e-5
        a, b = (O.cvt_bf16_f32(d) if bf16 else d for d in (dl1, dl))
        assert np.max(np.abs(a - b) / np.maximum(np.abs(b), np.float32(1e-3 / v / S))) <= (2.0 ** -7 if bf16 else 1e-5)
