"""The sums of partial weight gradients at the numbers of partial rows where their kernel changes how many it asks for at a time (64,
128, 512 and what is left behind a multiple of 512): by one row group of columns per sequence, QK-norm backward of batches of one
to 1025 slabs, against the oracle's sum over the same rows.  Bits are the same from run to run, and queued or not."""
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
    b.check(b.lib.mi355_dw_defer(0))


# slabs of [4][8]: one workgroup, so one partial row, each
@pytest.mark.parametrize("rows", [1, 31, 33, 63, 64, 65, 96, 127, 128, 129, 161, 479, 481, 500, 511, 512, 513, 575, 577, 640, 641, 1000, 1024, 1025])
def test_partial_rows(br, rows):
    print("[case] dw rows %d" % rows, flush=True)
    hd, S = 4, 8
    x, dy, w, dw0 = H.normal(995, (rows, hd, S)), H.normal(996, (rows, hd, S)), H.normal(997, hd, 1, 0.02), H.normal(998, hd)
    cos, sin = br.rope_tables_dev(S, hd, 1e4)
    D = br.DevArray.from_numpy
    xd, gd, wd = D(x), D(dy), D(w)
    got = []
    for defer in (0, 0, 1):
        br.check(br.lib.mi355_dw_defer(defer))
        out, dwd = br.DevArray(x.shape), D(dw0)
        br.check(br.lib.mi355_qknorm_rope_bwd_dev(out.ptr, None, dwd.ptr, None, gd.ptr, None, xd.ptr, None, wd.ptr, None, 1, 0, hd, S, rows, cos, sin,
                                                  1e-5, 0))
        br.check(br.lib.mi355_dw_flush())
        got.append(dwd.numpy())
    br.check(br.lib.mi355_dw_defer(0))
    assert got[0].tobytes() == got[1].tobytes() == got[2].tobytes()
    # 64-bit: dw[c] = sum over slabs and columns of (gradient un-rotated) * x / rms
    x64, g64 = x.astype(np.float64), dy.astype(np.float64)
    i = np.arange(hd // 2)[:, None]
    ang = np.arange(S)[None] * 1e4 ** (-2.0 * i / hd)
    c, s = np.cos(ang), np.sin(ang)
    d = np.empty_like(g64)
    d[:, 0::2] = g64[:, 0::2] * c + g64[:, 1::2] * s
    d[:, 1::2] = -g64[:, 0::2] * s + g64[:, 1::2] * c
    terms = d * x64 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + 1e-5)
    want = dw0 + terms.sum((0, 2))
    # fp32 terms (a few roundings each, tables to 1e-7 of a turn) summed in fp32: 2e-6 of the sum of magnitudes is well above both
    assert np.all(np.abs(got[0] - want) <= 2e-6 * (np.abs(dw0) + np.abs(terms).sum((0, 2))))
