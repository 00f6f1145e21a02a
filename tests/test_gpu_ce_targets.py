"""The one-launch softmax cross-entropy where its targets lie: all columns on one row (the first and last of the tensor, of a member, of a
row step), a lane's columns on rows of different steps, targets out of range, with scales that round; and the
numbers of row steps at which its smallest variants change (4 steps of 64 rows in each member)."""
import numpy as np
import pytest

import helpers as H
import oracle as O
from test_gpu_ce_rows import run

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def br():
    import ane_amd.bridge as b
    b.init()
    return b


def targets(kind, V, S):
    t = np.arange(S, dtype=np.int64)
    if kind == "first":
        t[:] = 0
    elif kind == "last":
        t[:] = V - 1
    elif kind == "steps":               # 64 rows apart: one lane's columns, one row step after the other
        t = t * 64 % V
    elif kind == "border":              # both sides of the members' borders
        rows = -(-V // max(1, min(256 // -(-S // 64), 64)))
        t = np.minimum((t // 2 + 1) * rows - t % 2, V - 1)
    elif kind == "outside":
        t = np.where(t % 3 == 0, -1 - t, np.where(t % 3 == 1, V + t, V // 2))
    return t.astype(np.int32)


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("kind", ["first", "last", "steps", "border", "outside"])
@pytest.mark.parametrize("V,S", [(60, 256), (300, 1000), (16384, 256), (16385, 200), (20000, 52), (33000, 61)])
def test_targets(br, V, S, kind, bf16):
    print("[case] ce targets V=%d S=%d %s bf16=%d" % (V, S, kind, bf16), flush=True)
    logits = H.normal(404, (V, S), 0, 2.0)
    if bf16:
        logits = O.cvt_bf16_f32(O.cvt_f32_bf16(logits))
    tgt = targets(kind, V, S)
    rl, rd = O.cross_entropy(logits, tgt, 0.37)
    loss, dl = run(br, logits, tgt, bf16, 0.37)
    got = O.cvt_bf16_f32(dl) if bf16 else dl
    assert abs(float(np.frombuffer(loss, np.float32)[0]) - rl) <= 1e-5 * max(abs(rl), 1e-3)
    assert H.rel_err(got, rd) <= (5e-3 if bf16 else 1e-5)         # the parity bars of the two storage types
    ok = (tgt >= 0) & (tgt < V)
    assert H.rel_err(got[tgt[ok], np.flatnonzero(ok)], rd[tgt[ok], np.flatnonzero(ok)]) <= (5e-3 if bf16 else 1e-5)
