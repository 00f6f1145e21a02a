"""The one-launch softmax cross-entropy on rows of any length and every number of row steps: row counts around the
variants' limits (8 and 16 steps of 64 rows in each of the members, and the LDS rows beyond), strips that do not divide the
row, short last groups, rows of whole 128-byte lines and others, tensors that start within a line."""
import numpy as np
import pytest

import helpers as H
import oracle as O

pytestmark = pytest.mark.gpu


def run(br, logits, tgt, bf16, scale, off=0):
    """off: elements between the start of an allocation and the tensor, on both sides"""
    dt = np.uint16 if bf16 else np.float32
    raw = O.cvt_f32_bf16(logits) if bf16 else logits
    ld = br.DevArray.from_numpy(np.concatenate([np.zeros(off, dt), raw.ravel()]))
    td, dl, loss = br.DevArray.from_numpy(tgt), br.DevArray(off + logits.size, dt), br.DevArray(1)
    fn, at = br.lib.mi355_softmax_ce_bf16_dev if bf16 else br.lib.mi355_softmax_ce_dev, off * dt().itemsize
    br.check(fn(dl.ptr + at, loss.ptr, ld.ptr + at, td.ptr, logits.shape[0], logits.shape[1], scale))
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
