"""The softmax ops on columns that hold NaNs and infinities: such a column is NaN from top to bottom and so is the loss that
counts it, as in the sequential loop; its neighbours are untouched."""
import numpy as np
import pytest

import helpers as H
import oracle as O

pytestmark = pytest.mark.gpu


def columns(V, S):
    x = H.normal(420, (V, S), 0, 2.0)
    x[V // 3, 0] = np.nan
    x[V - 1, 1] = np.inf
    x[:, 2] = np.nan
    x[:, 3] = -np.inf
    x[::2, 4] = -np.inf                              # ordinary: half of the column masked
    x[:, 5] = np.nan; x[V // 2, 5] = 1.0             # groups of rows that are NaN throughout
    x[7 % V:, 6] = -np.inf; x[0, 6] = np.nan         # ... and -inf throughout
    x[V // 5, S - 1] = np.nan
    return x, [0, 1, 2, 3, 5, 6, S - 1]


# one launch with one, two and more row steps, whole 128-byte lines and others; three launches with one and with four columns
# per lane; in place, which is three launches
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("V,S,form", [(40, 9, 0), (4608, 128, 0), (70001, 70, 0), (4608, 128, -1), (23500, 256, -1), (40, 9, "in place")])
def test_cross_entropy_keeps_nan_and_inf(br, V, S, form, bf16):
    print("[case] non-finite ce V=%d S=%d form=%s bf16=%d" % (V, S, form, bf16), flush=True)
    x, bad = columns(V, S)
    if bf16:
        x = O.cvt_bf16_f32(O.cvt_f32_bf16(x))
    tgt = np.random.default_rng(421).integers(0, V, S).astype(np.int32)
    tgt[1] = V                                       # (an out-of-range target: no loss term, the column still NaN)
    fn = br.lib.mi355_softmax_ce_bf16_dev if bf16 else br.lib.mi355_softmax_ce_dev
    put = lambda a: br.DevArray.from_numpy(O.cvt_f32_bf16(a) if bf16 else a)
    good = [t for t in range(S) if t not in bad]
    for counted in (True, False):
        if not counted:
            tgt[bad] = -1                            # no NaN column is counted: the loss is a number
        with np.errstate(all="ignore"):
            rl, rd = O.cross_entropy(x, tgt, 256.0)
        assert np.isnan(rd[:, bad]).all() and np.isfinite(rd[:, good]).all() and np.isnan(rl) == counted
        ld, td, loss = put(x), br.DevArray.from_numpy(tgt), br.DevArray(1)
        dl = ld if form == "in place" else put(np.zeros_like(x))
        br.tune("ce_resident", form if form == -1 else 0)
        try:
            br.check(fn(dl.ptr, loss.ptr, ld.ptr, td.ptr, V, S, 256.0))
        finally:
            br.tune("ce_resident", 0)
        got = O.cvt_bf16_f32(dl.numpy()) if bf16 else dl.numpy()
        assert np.isnan(got[:, bad]).all()
        assert H.rel_err(got[:, good], rd[:, good]) <= (5e-3 if bf16 else 1e-5)       # the parity bars of the storage types
        l = float(loss.numpy()[0])
        assert np.isnan(l) if counted else abs(l - rl) <= 1e-5 * abs(rl)


@pytest.mark.parametrize("V,S", [(40, 9), (4608, 128)])
def test_softmax_cols_keeps_nan_and_inf(br, V, S):
    x, bad = columns(V, S)
    with np.errstate(all="ignore"):
        want = O.softmax_cols(x)
    xd, pd = br.DevArray.from_numpy(x), br.DevArray((V, S))
    br.check(br.lib.mi355_softmax_cols_dev(pd.ptr, xd.ptr, V, S))
    got = pd.numpy()
    good = [t for t in range(S) if t not in bad]
    assert np.isnan(want[:, bad]).all() and np.isnan(got[:, bad]).all()
    assert H.rel_err(got[:, good], want[:, good]) <= 1e-5
