"""QK-norm + RoPE and the RMSNorm backward with the residual where a tile is whole (every row pair of a head, every column of a
strip) and one step beside it (one column more, a head size that leaves rows of the tile empty), fp32 and bfloat16."""
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


def to_bf(x):
    return O.cvt_f32_bf16(np.ascontiguousarray(x, np.float32)).reshape(x.shape)


def widen(h):
    return O.cvt_bf16_f32(np.ascontiguousarray(h)).reshape(h.shape)


def err(a, r):
    """Largest difference over the value, or over the root mean square where that is larger."""
    r = r.astype(np.float64)
    return float(np.max(np.abs(a - r) / np.maximum(np.abs(r), np.sqrt(np.mean(r * r)))))


# hd 128 and 64 fill the tiles; batches beyond the line below which bfloat16 takes one column per lane
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("hd,heads,kv,B,S", [(128, 16, 8, 9, 128), (128, 16, 8, 5, 256), (128, 16, 8, 5, 257), (64, 12, 12, 14, 256), (64, 12, 12, 14, 255),
                                             (96, 8, 8, 9, 256), (128, 3, 1, 2, 64)])
def test_qknorm_rope_whole_and_ragged_tiles(br, hd, heads, kv, B, S, bf16):
    print("[case] qk tiles hd=%d heads=%d kv=%d B=%d S=%d bf16=%d" % (hd, heads, kv, B, S, bf16), flush=True)
    theta, eps = 1e6, 1e-5
    end = "_bf16_dev" if bf16 else "_dev"
    enc, dec = (to_bf, widen) if bf16 else (lambda a: np.array(a), lambda a: a)
    D = br.DevArray.from_numpy
    cos, sin = br.rope_tables_dev(S, hd, theta)
    wq, wk = H.normal(960, hd, 1.0, 0.02), H.normal(961, hd, 1.0, 0.02)
    q, k = enc(H.normal(962, (B, heads * hd, S))), enc(H.normal(963, (B, kv * hd, S)))
    gq, gk = enc(H.normal(964, (B, heads * hd, S))), enc(H.normal(965, (B, kv * hd, S)))
    qd, kd, gqd, gkd, wqd, wkd = (D(a) for a in (q, k, gq, gk, wq, wk))
    qo, ko, dq, dk = (br.DevArray(a.shape, a.dtype) for a in (q, k, q, k))
    dwq, dwk = br.DevArray(hd), br.DevArray(hd)
    br.check(getattr(br.lib, "mi355_qknorm_rope_fwd" + end)(qo.ptr, ko.ptr, qd.ptr, kd.ptr, wqd.ptr, wkd.ptr, heads, kv, hd, S, B, cos, sin, eps))
    br.check(getattr(br.lib, "mi355_qknorm_rope_bwd" + end)(dq.ptr, dk.ptr, dwq.ptr, dwk.ptr, gqd.ptr, gkd.ptr, qd.ptr, kd.ptr, wqd.ptr, wkd.ptr,
                                                            heads, kv, hd, S, B, cos, sin, eps, 0))
    # one rounding to 8 bits on store, relative to the value (2^-8); fp32: as the other QK-norm tests
    tol, tol_w = (2.0 ** -8 * 1.01, 1e-5) if bf16 else (1e-5, 1e-5)
    for x, g, w, out, dx, dw in ((q, gq, wq, qo, dq, dwq), (k, gk, wk, ko, dk, dwk)):
        y = O.qknorm_rope_fwd(dec(x), w, hd, theta, eps)
        rdx, rdw = O.qknorm_rope_bwd(dec(g), dec(x), w, hd, theta, eps)
        assert err(dec(out.numpy()), y) <= tol
        assert err(dec(dx.numpy()), rdx) <= tol
        assert err(dw.numpy(), rdw) <= tol_w


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("C,S,B", [(1024, 256, 16), (1024, 128, 3), (1024, 255, 16), (512, 256, 4), (768, 256, 8)])
def test_rmsnorm_bwd_residual_whole_and_ragged_tiles(br, C, S, B, bf16):
    print("[case] rmsnorm_bwd_residual C=%d S=%d B=%d bf16=%d" % (C, S, B, bf16), flush=True)
    end = "_bf16_dev" if bf16 else "_dev"
    enc, dec = (to_bf, widen) if bf16 else (lambda a: np.array(a), lambda a: a)
    x, dy, res = (enc(H.normal(970 + i, (B, C, S))) for i in range(3))
    w = H.normal(973, C, 1.0, 0.02)
    xd, dyd, rd, wd = (br.DevArray.from_numpy(a) for a in (x, dy, res, w))
    dx, dx2, dw = br.DevArray(x.shape, x.dtype), br.DevArray(x.shape, x.dtype), br.DevArray(C)
    br.check(getattr(br.lib, "mi355_rmsnorm_bwd_residual" + end)(dx.ptr, dx2.ptr, dw.ptr, dyd.ptr, xd.ptr, wd.ptr, rd.ptr, 0.25, C, S, B, 1e-5, 0))
    rdx, rdw = O.rmsnorm_bwd(dec(dy), dec(x), w)
    want = rdx.reshape(x.shape) + dec(res)
    tol = 2.0 ** -8 * 1.01 if bf16 else 1e-5
    assert err(dec(dx.numpy()), want) <= tol
    assert err(dec(dx2.numpy()), want * np.float32(0.25)) <= tol
    assert err(dw.numpy(), rdw) <= 1e-5


# whole rows of a tile beside columns that are not: one column in the last strip, the last group moved back over a strip's edge,
# strips that end inside a group; in place where the tile allows it and where another takes over (S % 128 < 8)
@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("hd,heads,kv,B,S", [(128, 16, 8, 9, 129), (128, 16, 8, 8, 147), (128, 16, 8, 4, 197), (128, 16, 8, 40, 33), (128, 16, 8, 60, 15),
                                             (64, 12, 12, 30, 131), (64, 12, 12, 30, 136), (128, 16, 8, 100, 8)])
def test_qknorm_rope_ragged_strips(br, hd, heads, kv, B, S, bf16):
    print("[case] qk strips hd=%d heads=%d kv=%d B=%d S=%d bf16=%d" % (hd, heads, kv, B, S, bf16), flush=True)
    end = "_bf16_dev" if bf16 else "_dev"
    enc, dec = (to_bf, widen) if bf16 else (lambda a: np.array(a), lambda a: a)
    theta, eps = 1e6, 1e-5
    D = br.DevArray.from_numpy
    cos, sin = br.rope_tables_dev(S, hd, theta)
    wq, wk = H.normal(980, hd, 1.0, 0.02), H.normal(981, hd, 1.0, 0.02)
    q, k = enc(H.normal(982, (B, heads * hd, S))), enc(H.normal(983, (B, kv * hd, S)))
    gq, gk = enc(H.normal(984, (B, heads * hd, S))), enc(H.normal(985, (B, kv * hd, S)))
    qd, kd, wqd, wkd = (D(a) for a in (q, k, wq, wk))
    guard = lambda a: D(np.concatenate([a.ravel(), np.full(64, 7, a.dtype)]))
    tol = 2.0 ** -8 * 1.01 if bf16 else 1e-5          # one rounding to 8 bits on store
    qo, ko = guard(np.zeros_like(q)), guard(np.zeros_like(k))
    br.check(getattr(br.lib, "mi355_qknorm_rope_fwd" + end)(qo.ptr, ko.ptr, qd.ptr, kd.ptr, wqd.ptr, wkd.ptr, heads, kv, hd, S, B, cos, sin, eps))
    for x, w, o in ((q, wq, qo), (k, wk, ko)):
        got = o.numpy()
        assert err(dec(got[:x.size].reshape(x.shape)), O.qknorm_rope_fwd(dec(x), w, hd, theta, eps)) <= tol
        assert np.all(got[x.size:] == 7)
    for in_place in (False, True):
        gqd, gkd = guard(gq), guard(gk)
        dq, dk = (gqd, gkd) if in_place else (guard(np.zeros_like(q)), guard(np.zeros_like(k)))
        dwq, dwk = br.DevArray(hd), br.DevArray(hd)
        br.check(getattr(br.lib, "mi355_qknorm_rope_bwd" + end)(dq.ptr, dk.ptr, dwq.ptr, dwk.ptr, gqd.ptr, gkd.ptr, qd.ptr, kd.ptr, wqd.ptr, wkd.ptr,
                                                       heads, kv, hd, S, B, cos, sin, eps, 0))
        for x, g, w, dx, dw in ((q, gq, wq, dq, dwq), (k, gk, wk, dk, dwk)):
            rdx, rdw = O.qknorm_rope_bwd(dec(g), dec(x), w, hd, theta, eps)
            got = dx.numpy()
            assert err(dec(got[:x.size].reshape(x.shape)), rdx) <= tol
            assert np.all(got[x.size:] == 7)
            assert err(dw.numpy(), rdw) <= 1e-5


# clusters whose members hold fewer rows than lanes, or a last strip of one column or of less than a group: every load in bounds,
# nothing counted twice
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("C,S,B", [(768, 129, 3), (768, 64, 5), (1024, 65, 4), (1024, 193, 6), (520, 9, 2), (513, 131, 2), (1000, 77, 3)])
def test_rmsnorm_ragged_clusters(br, C, S, B, bf16):
    print("[case] rmsnorm clusters C=%d S=%d B=%d bf16=%d" % (C, S, B, bf16), flush=True)
    end = "_bf16_dev" if bf16 else "_dev"
    enc, dec = (to_bf, widen) if bf16 else (lambda a: np.array(a), lambda a: a)
    x, dy, res = (enc(H.normal(990 + i, (B, C, S))) for i in range(3))
    w = H.normal(993, C, 1.0, 0.02)
    one = np.array([7], x.dtype)
    guard = lambda a: br.DevArray.from_numpy(np.concatenate([a.ravel(), np.repeat(one, 64)]))
    xd, dyd, rd, wd = guard(x), guard(dy), guard(res), br.DevArray.from_numpy(w)
    tol = 2.0 ** -8 * 1.01 if bf16 else 1e-5

    def check(d, want):
        got = d.numpy()
        assert err(dec(got[:x.size].reshape(x.shape)), want) <= tol
        assert np.all(got[x.size:] == one)

    y, yn, dx, dw = guard(np.zeros_like(x)), guard(np.zeros_like(x)), guard(np.zeros_like(x)), br.DevArray(C)
    br.check(getattr(br.lib, "mi355_rmsnorm_fwd" + end)(y.ptr, xd.ptr, wd.ptr, C, S, B, 1e-5))
    check(y, O.rmsnorm(dec(x), w).reshape(x.shape))
    br.check(getattr(br.lib, "mi355_residual_rmsnorm_fwd" + end)(y.ptr, yn.ptr, xd.ptr, rd.ptr, 0.25, wd.ptr, C, S, B, 1e-5))
    got_y = y.numpy()[:x.size].reshape(x.shape)
    check(y, dec(res) * np.float32(0.25) + dec(x))
    check(yn, O.rmsnorm(dec(got_y), w).reshape(x.shape))
    br.check(getattr(br.lib, "mi355_rmsnorm_bwd" + end)(dx.ptr, dw.ptr, dyd.ptr, xd.ptr, wd.ptr, C, S, B, 1e-5, 0))
    rdx, rdw = O.rmsnorm_bwd(dec(dy), dec(x), w)
    check(dx, rdx.reshape(x.shape))
    assert err(dw.numpy(), rdw) <= 1e-5


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("res", [False, True])
@pytest.mark.parametrize("C,S,B", [(768, 129, 3), (768, 256, 2), (513, 131, 2)])
def test_rmsnorm_bwd_clusters_pass_infinities_on(br, C, S, B, res, bf16):
    """Lanes without a row read row 0: an infinity there must not become a NaN in a sum that it would only make infinite."""
    print("[case] rmsnorm_bwd infinities C=%d S=%d B=%d res=%d bf16=%d" % (C, S, B, res, bf16), flush=True)
    end = "_bf16_dev" if bf16 else "_dev"
    enc, dec = (to_bf, widen) if bf16 else (lambda a: np.array(a), lambda a: a)
    x, dy, r = (enc(H.normal(995 + i, (B, C, S))) for i in range(3))
    dy[0, 0, 5] = enc(np.array([np.inf], np.float32))[0]
    dy[B - 1, 0, S - 1] = enc(np.array([-np.inf], np.float32))[0]
    w = H.normal(998, C, 1.0, 0.02)
    D = br.DevArray.from_numpy
    xd, dyd, rd, wd, dx, dw = D(x), D(dy), D(r), D(w), br.DevArray(x.shape, x.dtype), br.DevArray(C)
    if res:
        br.check(getattr(br.lib, "mi355_rmsnorm_bwd_residual" + end)(dx.ptr, None, dw.ptr, dyd.ptr, xd.ptr, wd.ptr, rd.ptr, 0.25, C, S, B, 1e-5, 0))
    else:
        br.check(getattr(br.lib, "mi355_rmsnorm_bwd" + end)(dx.ptr, dw.ptr, dyd.ptr, xd.ptr, wd.ptr, C, S, B, 1e-5, 0))
    with np.errstate(invalid="ignore"):
        rdx, _ = O.rmsnorm_bwd(dec(dy), dec(x), w)
        want = rdx.reshape(x.shape) + (dec(r) if res else np.float32(0))
    got = dec(dx.numpy())
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want))
    assert np.array_equal(np.isneginf(got), np.isneginf(want))


# an infinity in the table's first value reaches the column and the row pair that it belongs to, also where lanes without a row pair or
# without columns (heads and strips that do not fill the tile) load the table's first values in place of none
@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("hd,heads,kv,B,S", [(96, 8, 8, 9, 256), (96, 8, 8, 9, 100), (40, 8, 4, 9, 200), (192, 4, 4, 9, 72), (128, 2, 1, 1, 33), (128, 16, 8, 9, 129), (6, 3, 1, 2, 9)])
def test_qknorm_rope_bwd_infinite_table_value_stays_in_its_column(br, hd, heads, kv, B, S, bf16):
    print("[case] qk table hd=%d heads=%d kv=%d B=%d S=%d bf16=%d" % (hd, heads, kv, B, S, bf16), flush=True)
    end = "_bf16_dev" if bf16 else "_dev"
    enc, dec = (to_bf, widen) if bf16 else (lambda a: np.array(a), lambda a: a)
    D = br.DevArray.from_numpy
    angle = H.normal(990, (hd // 2, S))
    wq, wk = H.normal(991, hd, 1.0, 0.02), H.normal(992, hd, 1.0, 0.02)
    ops = [enc(H.normal(993 + i, (B, n * hd, S))) for i, n in enumerate((heads, kv, heads, kv))]
    gq, gk, q, k = ops
    gqd, gkd, qd, kd, wqd, wkd = (D(a) for a in (gq, gk, q, k, wq, wk))
    res = []
    for first in (np.float32(0.5), np.float32(np.inf)):
        cos, sin = np.cos(angle).astype(np.float32), np.sin(angle).astype(np.float32)
        cos[0, 0] = first
        cd, sd = D(cos), D(sin)
        dq, dk, dwq, dwk = br.DevArray(q.shape, q.dtype), br.DevArray(k.shape, k.dtype), br.DevArray(hd), br.DevArray(hd)
        br.check(getattr(br.lib, "mi355_qknorm_rope_bwd" + end)(dq.ptr, dk.ptr, dwq.ptr, dwk.ptr, gqd.ptr, gkd.ptr, qd.ptr, kd.ptr, wqd.ptr, wkd.ptr,
                                                                heads, kv, hd, S, B, cd.ptr, sd.ptr, 1e-5, 0))
        res.append([a.numpy() for a in (dq, dk, dwq, dwk)])
    for i in (0, 1):
        assert res[0][i][..., 1:].tobytes() == res[1][i][..., 1:].tobytes()
        assert res[0][2 + i][2:].tobytes() == res[1][2 + i][2:].tobytes()
        assert np.all(np.isfinite(res[0][2 + i])) and not np.any(np.isfinite(dec(res[1][i][..., 0])))
