"""Converts and the attention-gradient finish on rows of any length and pitch, at any element: the last lane of a row takes
the row's last whole group again.  Conversions, copies and sums in a stated order: the same bits as the oracle."""
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


@pytest.mark.parametrize("rows,cols,dst_ld,src_ld,shift", [
    (33, 197, 1221, 197, 0),      # a surface whose rows hold something else behind
    (5, 8, 9, 11, 1),             # one group
    (700, 9, 10, 9, 1),           # two groups that share seven elements
    (31, 197, 197, 197, 1),       # no gaps: one row of 6107 elements
    (1, 7, 7, 7, 0), (2, 7, 7, 7, 1), (3, 7, 8, 7, 0),      # fewer than a group; 14 without gaps; rows of 7
    (64, 256, 256, 260, 3),
])
def test_cvt_rows_of_any_length(br, rows, cols, dst_ld, src_ld, shift):
    src = H.normal(150, (rows, src_ld), 0, 30.0)
    half0 = np.random.default_rng(151).integers(0, 65536, shift + rows * dst_ld).astype(np.uint16)
    sd = br.DevArray.from_numpy(np.concatenate([np.zeros(shift, np.float32), src.ravel()]))
    hd = br.DevArray.from_numpy(half0)
    br.check(br.lib.mi355_cvt_f32_f16_dev(hd.ptr + 2 * shift, dst_ld, sd.ptr + 4 * shift, src_ld, rows, cols))
    want = half0.copy()
    want[shift:].reshape(rows, dst_ld)[:, :cols] = O.cvt_f32_f16(src[:, :cols])
    assert np.array_equal(hd.numpy(), want)
    back0 = H.normal(152, shift + rows * src_ld)
    bd = br.DevArray.from_numpy(back0)
    br.check(br.lib.mi355_cvt_f16_f32_dev(bd.ptr + 4 * shift, src_ld, hd.ptr + 2 * shift, dst_ld, rows, cols))
    wantb = back0.copy()
    wantb[shift:].reshape(rows, src_ld)[:, :cols] = O.cvt_f16_f32(want[shift:].reshape(rows, dst_ld)[:, :cols])
    assert np.array_equal(bd.numpy().view(np.uint32), wantb.view(np.uint32))


@pytest.mark.parametrize("S", [4, 5, 8, 9, 15, 197, 256])
@pytest.mark.parametrize("in_f16,shift,in_place", [(1, 0, False), (1, 1, False), (0, 0, False), (0, 1, False), (0, 0, True)])
def test_finish_rows_of_any_length(br, S, in_f16, shift, in_place):
    B, heads, kvh, hd, theta = 3, 4, 4 if in_place else 2, 8, 1e4
    ratio, full, kv = heads // kvh, (B, heads * hd, S), (B, kvh * hd, S)
    src = [H.normal(160 + i, full) for i in range(3)]
    ins = [O.cvt_f32_f16(a) for a in src] if in_f16 else src
    size = 2 if in_f16 else 4
    ind = [br.DevArray.from_numpy(np.concatenate([np.zeros(shift, a.dtype), a.ravel()])) for a in ins]
    outs = ind if in_place else [br.DevArray(int(np.prod(s)) + shift) for s in (full, kv, kv)]
    cosd, sind = br.rope_tables_dev(S, hd, theta)
    br.check(br.lib.mi355_attn_grads_finish_dev(*[o.ptr + 4 * shift for o in outs], *[a.ptr + size * shift for a in ind],
                                                in_f16, 0, 0, 0, heads, kvh, hd, S, B, cosd, sind))
    cv = O.cvt_f16_f32 if in_f16 else (lambda a: a)
    q = cv(ins[0])
    k, v = (np.stack([O.gqa_reduce(cv(a[b]), kvh, ratio, hd) for b in range(B)]) for a in ins[1:])
    for got, ref in zip(outs, (O.rope(q, hd, theta, -1), O.rope(k, hd, theta, -1), v)):
        assert np.array_equal(got.numpy().ravel()[shift:].view(np.uint32), ref.ravel().view(np.uint32))
