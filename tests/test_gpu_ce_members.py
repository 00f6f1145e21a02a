"""The one-launch softmax cross-entropy with up to 128 members to a strip: rows of one and two strips (bfloat16: three) around the row
counts where it begins, where eight row steps end and where rows are read twice; every partial handed over, and recomputed."""
import numpy as np
import pytest

import helpers as H
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def br():
    import ane_amd.bridge as b
    b.init()
    yield b
    b.tune("xch_take_nothing", 0)


@pytest.mark.parametrize("V,S,bf16", [(28672, 64, False), (28673, 64, False), (57344, 37, False), (65536, 65, False), (65537, 128, False), (140001, 68, False),
                                      (28673, 5, True), (65536, 64, True), (65537, 127, True), (213001, 6, True), (49152, 192, True), (49153, 192, True), (50001, 133, True), (131072, 192, True), (131073, 192, True), (140001, 133, True)])
def test_members(br, V, S, bf16):
    print("[case] ce members V=%d S=%d bf16=%d" % (V, S, bf16), flush=True)
    logits = np.random.default_rng(830).standard_normal((V, S), dtype=np.float32) * np.float32(2.0)
    raw = O.cvt_f32_bf16(logits) if bf16 else logits
    if bf16:
        logits = O.cvt_bf16_f32(raw)
    tgt = np.random.default_rng(831).integers(0, V, S).astype(np.int32)
    tgt[0], tgt[S - 1] = V - 1, 0
    tgt[1], tgt[S - 2] = V, -1                            # out-of-range targets are skipped
    ld, td = br.DevArray.from_numpy(raw), br.DevArray.from_numpy(tgt)
    fn = br.lib.mi355_softmax_ce_bf16_dev if bf16 else br.lib.mi355_softmax_ce_dev

    def run():
        dl, loss = br.DevArray(raw.shape, raw.dtype), br.DevArray(1)
        br.check(fn(dl.ptr, loss.ptr, ld.ptr, td.ptr, V, S, 256.0))
        return loss.numpy(), dl.numpy()

    expired = br.exchange_fallbacks()[1]
    loss, dl = run()
    assert br.exchange_fallbacks()[1] == expired
    rl, rd = O.cross_entropy(logits, tgt, 256.0)
    assert abs(float(loss[0]) - rl) <= 1e-5 * max(abs(rl), 1e-3)
    assert H.rel_err(O.cvt_bf16_f32(dl) if bf16 else dl, rd) <= (5e-3 if bf16 else 1e-5)         # the parity bars of the two storage types
    br.tune("xch_take_nothing", 1)
    try:
        loss2, dl2 = run()
    finally:
        br.tune("xch_take_nothing", 0)
    assert br.exchange_fallbacks()[1] > expired           # (it is the one launch)
    assert loss2.tobytes() == loss.tobytes() and dl2.tobytes() == dl.tobytes()
