"""Rows whose length is no multiple of a lane's columns, and tensors that start at any element: the last lane of such a
row takes columns that are also its neighbour's (lane_cols in tile.h), in place as well as out of place.

S = 65 and 257 leave a last strip shorter than a lane (in place: the one-column tiles), 67 and 197 one that holds the
short group and its neighbour, 9 and 4 rows of about one lane."""
import numpy as np
import pytest

import helpers as H
import oracle as O

pytestmark = pytest.mark.gpu
TOL, TOL16 = 1e-5, 5e-3         # the parity bars of fp32 and of bfloat16 results
ALPHA = np.float32(0.7)


class Store:
    """fp32 or bfloat16 device tensors that start `off` elements behind an aligned address."""

    def __init__(self, br, bf16, off):
        self.br, self.off, self.dtype, self.tol = br, off, (np.uint16 if bf16 else np.float32), (TOL16 if bf16 else TOL)
        self.bf16, self.keep = bf16, []

    def values(self, a):
        return O.cvt_bf16_f32(O.cvt_f32_bf16(a)) if self.bf16 else a

    def put(self, a):
        raw = O.cvt_f32_bf16(a) if self.bf16 else a
        d = self.br.DevArray.from_numpy(np.concatenate([np.zeros(self.off, self.dtype), raw.ravel()]))
        self.keep.append(d)
        return d.ptr + self.off * self.dtype().itemsize

    def new(self, shape):
        return self.put(np.zeros(shape, np.float32))

    def get(self, ptr, shape):
        d = [d for d in self.keep if d.ptr + self.off * self.dtype().itemsize == ptr][0]
        raw = d.numpy()[self.off:].reshape(shape)
        return O.cvt_bf16_f32(raw) if self.bf16 else raw

    def fn(self, name):
        return getattr(self.br.lib, "mi355_%s_bf16_dev" % name if self.bf16 else "mi355_%s_dev" % name)


SHAPES = [(2, 768, 197), (1, 768, 65), (3, 1030, 67), (1, 5000, 9), (2, 100, 257), (2, 48, 4), (8, 600, 511), (70, 768, 131)]


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("B,C,S", SHAPES)
def test_rmsnorm_family_on_rows_of_any_length(br, B, C, S, bf16, off):
    print("[case] ragged rmsnorm B=%d C=%d S=%d bf16=%d off=%d" % (B, C, S, bf16, off), flush=True)
    st = Store(br, bf16, off)
    x, dy, res = (st.values(H.normal(300 + i, (B, C, S))) for i in range(3))
    w, dw0 = H.normal(310, C, 1.0, 0.02), H.normal(311, C)
    wd = br.DevArray.from_numpy(w)
    xd = st.put(x)
    want_y = O.rmsnorm(x, w)
    want_dx, want_dw = O.rmsnorm_bwd(dy, x, w, dw=dw0)
    want_r = O.axpby(x, res, ALPHA, 0)
    want_dxr = O.axpby(want_dx, res, 0.0, 2)
    for in_place in (False, True):
        y = st.put(x) if in_place else st.new(x.shape)
        br.check(st.fn("rmsnorm_fwd")(y, y if in_place else xd, wd.ptr, C, S, B, 1e-5))
        assert H.rel_err(st.get(y, x.shape), want_y) <= st.tol
        dyd, dwd = st.put(dy), br.DevArray.from_numpy(dw0)
        dx = dyd if in_place else st.new(x.shape)
        br.check(st.fn("rmsnorm_bwd")(dx, dwd.ptr, dyd, xd, wd.ptr, C, S, B, 1e-5, 0))
        assert H.rel_err(st.get(dx, x.shape), want_dx) <= st.tol and H.rel_err(dwd.numpy(), want_dw) <= TOL
        a, b, yn = st.put(x), st.put(res), st.new(x.shape)
        y2 = a if in_place else st.new(x.shape)
        br.check(st.fn("residual_rmsnorm_fwd")(y2, yn, a, b, ALPHA, wd.ptr, C, S, B, 1e-5))
        got = st.get(y2, x.shape)
        assert H.rel_err(got, want_r) <= st.tol and H.rel_err(st.get(yn, x.shape), O.rmsnorm(got, w)) <= st.tol
        for over in (["res", "dy"] if in_place else [None]):
            dyd, rd, dwd, dxs = st.put(dy), st.put(res), br.DevArray.from_numpy(dw0), st.new(x.shape)
            dx = rd if over == "res" else dyd if over == "dy" else st.new(x.shape)
            br.check(st.fn("rmsnorm_bwd_residual")(dx, dxs, dwd.ptr, dyd, xd, wd.ptr, rd, ALPHA, C, S, B, 1e-5, 0))
            assert H.rel_err(st.get(dx, x.shape), want_dxr) <= st.tol, over
            assert H.rel_err(st.get(dxs, x.shape), O.axpby(want_dxr, None, ALPHA, 1)) <= st.tol
            assert H.rel_err(dwd.numpy(), want_dw) <= TOL


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("B,heads,kvh,hd,S", [(2, 4, 2, 128, 197), (1, 2, 1, 64, 65), (1, 3, 3, 16, 257), (2, 2, 1, 128, 9), (1, 2, 2, 32, 4),
                                                # large enough for eight columns per lane: 16 and 8 lanes, 256 and 512 threads
                                                (9, 12, 12, 64, 197), (52, 12, 12, 64, 33), (6, 16, 8, 128, 197),
                                                (6, 16, 8, 128, 257), (32, 16, 8, 128, 33), (40, 12, 12, 32, 100)])
def test_rope_and_qknorm_on_rows_of_any_length(br, B, heads, kvh, hd, S, bf16):
    print("[case] ragged rope B=%d heads=%d/%d hd=%d S=%d bf16=%d" % (B, heads, kvh, hd, S, bf16), flush=True)
    st = Store(br, bf16, 1)
    q, gq = (st.values(H.normal(320 + i, (B, heads * hd, S))) for i in range(2))
    k, gk = (st.values(H.normal(330 + i, (B, kvh * hd, S))) for i in range(2))
    wq, wk = H.normal(340, hd, 1.0, 0.02), H.normal(341, hd, 1.0, 0.02)
    wqd, wkd = br.DevArray.from_numpy(wq), br.DevArray.from_numpy(wk)
    cd, sd = br.rope_tables_dev(S, hd, 1e4)
    tol = st.tol if hd >= 16 else 1e-3
    rdq, rdwq = O.qknorm_rope_bwd(gq, q, wq, hd, 1e4)
    rdk, rdwk = O.qknorm_rope_bwd(gk, k, wk, hd, 1e4)
    for in_place in (False, True):
        qd, kd, gqd, gkd = st.put(q), st.put(k), st.put(gq), st.put(gk)
        qo, ko = (qd, kd) if in_place else (st.new(q.shape), st.new(k.shape))
        br.check(st.fn("rope")(qo, ko, qd, kd, heads, kvh, hd, S, B, cd, sd, -1))
        assert H.rel_err(st.get(qo, q.shape), O.rope(q, hd, 1e4, -1)) <= st.tol
        assert H.rel_err(st.get(ko, k.shape), O.rope(k, hd, 1e4, -1)) <= st.tol
        qd, kd = st.put(q), st.put(k)
        qo, ko = st.new(q.shape), st.new(k.shape)
        br.check(st.fn("qknorm_rope_fwd")(qo, ko, qd, kd, wqd.ptr, wkd.ptr, heads, kvh, hd, S, B, cd, sd, 1e-5))
        assert H.rel_err(st.get(qo, q.shape), O.qknorm_rope_fwd(q, wq, hd, 1e4)) <= tol
        assert H.rel_err(st.get(ko, k.shape), O.qknorm_rope_fwd(k, wk, hd, 1e4)) <= tol
        dq, dk = (gqd, gkd) if in_place else (st.new(q.shape), st.new(k.shape))
        dwq, dwk = br.DevArray(hd), br.DevArray(hd)
        br.check(st.fn("qknorm_rope_bwd")(dq, dk, dwq.ptr, dwk.ptr, gqd, gkd, qd, kd, wqd.ptr, wkd.ptr, heads, kvh, hd, S,
                                          B, cd, sd, 1e-5, 0))
        assert H.rel_err(st.get(dq, q.shape), rdq) <= tol and H.rel_err(st.get(dk, k.shape), rdk) <= tol
        assert H.rel_err(dwq.numpy(), rdwq) <= TOL and H.rel_err(dwk.numpy(), rdwk) <= TOL


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("which", ["q", "k"])
def test_qknorm_of_one_operand_alone_is_not_in_place(br, which, bf16):
    """heads = 0 or kv_heads = 0 with NULL for what is absent: those equal pointers are no call in place, whose rows of this
    length go one column per lane, which holds no head of 256."""
    B, n, hd, S = 1, 2, 256, 257
    st = Store(br, bf16, 0)
    x, g, w = st.values(H.normal(350, (B, n * hd, S))), st.values(H.normal(351, (B, n * hd, S))), H.normal(352, hd, 1.0, 0.02)
    wd, xd, gd, dw = br.DevArray.from_numpy(w), st.put(x), st.put(g), br.DevArray(hd)
    cd, sd = br.rope_tables_dev(S, hd, 1e4)
    both = lambda a: (a, None) if which == "q" else (None, a)
    counts = (n, 0) if which == "q" else (0, n)
    y, dx = st.new(x.shape), st.new(x.shape)
    br.check(st.fn("qknorm_rope_fwd")(*both(y), *both(xd), *both(wd.ptr), *counts, hd, S, B, cd, sd, 1e-5))
    assert H.rel_err(st.get(y, x.shape), O.qknorm_rope_fwd(x, w, hd, 1e4)) <= st.tol
    br.check(st.fn("qknorm_rope_bwd")(*both(dx), *both(dw.ptr), *both(gd), *both(xd), *both(wd.ptr), *counts, hd, S, B, cd, sd, 1e-5, 0))
    rdx, rdw = O.qknorm_rope_bwd(g, x, w, hd, 1e4)
    assert H.rel_err(st.get(dx, x.shape), rdx) <= st.tol and H.rel_err(dw.numpy(), rdw) <= TOL
