"""Streams whose results are written through to memory (8 MB and more to a tensor that starts on a 128-byte line): the call over the
whole tensor against calls over pieces of it that are below that size, which take the other form.  The bytes are the same.
Values include the ones that a rounding or a clamp would treat apart."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LINE = 1 << 21          # fp32 values of 8 MB


@pytest.fixture(scope="module")
def br():
    import ane_amd.bridge as b
    b.init()
    return b


def values(rng, n, dtype):
    x = rng.standard_normal(n, dtype=np.float32)
    x[:8] = [0.0, -0.0, np.inf, -np.inf, np.nan, 3e38, -1e-42, -200.0]
    x[-3:] = [1e-45, -3e38, 88.8]
    if dtype == np.uint16:
        return (x.view(np.uint32) >> 16).astype(np.uint16)
    with np.errstate(over="ignore"):
        return x.astype(dtype)


def pieces(n, step):
    return [(a, min(step, n - a)) for a in range(0, n, step)]


def both(br, call, n, ins, outs, step, off=0):
    """call(out addresses, in addresses, count) over [off, n) at once, then piece by piece into other buffers"""
    got = []
    for parts in ([(off, n - off)], [(off + a, k) for a, k in pieces(n - off, step)]):
        o = [br.DevArray.from_numpy(np.full(n, 7, d)) for d in outs]
        for a, k in parts:
            br.check(call([b.ptr + a * b.dtype.itemsize for b in o], [b.ptr + a * b.dtype.itemsize for b in ins], k))
        got.append([b.numpy() for b in o])
    for a, b in zip(*got):
        assert a.tobytes() == b.tobytes(), np.flatnonzero(a.view(np.uint8) != b.view(np.uint8))[:8]


# (fp32 values, first value: 32 starts on a line, 4 does not)
SIZES = [(LINE - 4, 0), (LINE, 0), (LINE + 7, 0), (LINE + 36, 32), (LINE + 40, 4), (2 * LINE + 252, 0)]


@pytest.mark.parametrize("n,off", SIZES)
def test_fp32_elementwise(br, n, off):
    rng = np.random.default_rng(n + off)
    a, b, c = (br.DevArray.from_numpy(values(rng, n, np.float32)) for _ in range(3))
    f4 = np.float32
    both(br, lambda o, i, k: br.lib.mi355_swiglu_fwd_dev(o[0], i[0], i[1], k), n, [a, b], [f4], LINE // 2, off)
    both(br, lambda o, i, k: br.lib.mi355_swiglu_bwd_dev(o[0], o[1], i[0], i[1], i[2], k), n, [a, b, c], [f4, f4], LINE // 2, off)
    for mode in range(3):
        both(br, lambda o, i, k: br.lib.mi355_axpby_dev(o[0], i[0], i[1], 0.3, k, mode), n, [a, b], [f4], LINE // 2, off)
        both(br, lambda o, i, k: br.lib.mi355_axpby_dev(o[0], o[0], i[1], 0.3, k, mode), n, [a, b], [f4], LINE // 2, off)
    q, s = br.DevArray.from_numpy(rng.integers(-128, 128, n).astype(np.int8)), br.DevArray.from_numpy(np.array([0.037], f4))
    both(br, lambda o, i, k: br.lib.mi355_int8_dequant_dev(o[0], i[0], s.ptr, k), n, [q], [f4], LINE // 2, off)


@pytest.mark.parametrize("n,off", [(2 * n, 2 * off) for n, off in SIZES])
def test_bf16_elementwise(br, n, off):
    rng = np.random.default_rng(n + off)
    a, b, c = (br.DevArray.from_numpy(values(rng, n, np.uint16)) for _ in range(3))
    u2 = np.uint16
    both(br, lambda o, i, k: br.lib.mi355_swiglu_fwd_bf16_dev(o[0], i[0], i[1], k), n, [a, b], [u2], LINE, off)
    both(br, lambda o, i, k: br.lib.mi355_swiglu_bwd_bf16_dev(o[0], o[1], i[0], i[1], i[2], k), n, [a, b, c], [u2, u2], LINE, off)
    for mode in range(3):
        both(br, lambda o, i, k: br.lib.mi355_axpby_bf16_dev(o[0], i[0], i[1], 0.3, k, mode), n, [a, b], [u2], LINE, off)


@pytest.mark.parametrize("zero", [0, 1])
@pytest.mark.parametrize("n,off", SIZES + [(8 * LINE - 1, 0), (8 * LINE + 36, 32), (8 * LINE + 11, 8)])
def test_adam(br, n, off, zero):
    """one tensor as a whole, one tensor in pieces, and the many-tensor launch over the pieces, which is written through from 16 M
    parameters (8 * LINE) on where all pieces start on a line"""
    import ctypes
    rng = np.random.default_rng(n + off)
    host = [rng.standard_normal(n, dtype=np.float32) for _ in range(4)]
    host[3] = host[3] ** 2
    rest = (3, 1e-3, 0.9, 0.95, 1e-8)
    got = []
    for way in range(3):
        d = [br.DevArray.from_numpy(h) for h in host]
        parts = [(off, n - off)] if way == 0 else [(off + a, k) for a, k in pieces(n - off, LINE // 2 + 64)]
        if way < 2:
            for a, k in parts:
                br.check(br.lib.mi355_adam_update_dev(*[b.ptr + 4 * a for b in d], k, *rest, 0.1, 0.5, None, zero))
        else:
            arrays = [(ctypes.c_void_p * len(parts))(*[b.ptr + 4 * a for a, _ in parts]) for b in d]
            ns = (ctypes.c_size_t * len(parts))(*[k for _, k in parts])
            wd = (ctypes.c_float * len(parts))(*[0.1] * len(parts))
            br.check(br.lib.mi355_adam_update_multi_dev(*arrays, ns, wd, len(parts), *rest, 0.5, None, zero))
        got.append([b.numpy().tobytes() for b in d])
    assert got[0] == got[1] == got[2]


# row lengths and pitches that are whole lines of the result or not, rows, first element of the surface
@pytest.mark.parametrize("cols,ld,rows,off", [(256, 256, 16384, 0), (256, 1280, 16384, 0), (192, 256, 21846, 64), (256, 264, 16384, 0),
                                              (250, 256, 16800, 0), (256, 1280, 16384, 8), (LINE * 2 + 64, LINE * 2 + 64, 1, 0)])
def test_fp16_rectangles(br, cols, ld, rows, off):
    rng = np.random.default_rng(cols + ld)
    n = rows * ld + off
    for to16 in (True, False):
        src_t, dst_t = (np.float32, np.float16) if to16 else (np.float16, np.float32)
        fn = br.lib.mi355_cvt_f32_f16_dev if to16 else br.lib.mi355_cvt_f16_f32_dev
        src = br.DevArray.from_numpy(values(rng, rows * cols, src_t))
        got = []
        for step in (rows, max(rows // 3, 1)) if rows > 1 else (1,):
            dst = br.DevArray.from_numpy(np.full(n, 7, dst_t))
            for r, k in pieces(rows, step):
                br.check(fn(dst.ptr + dst.dtype.itemsize * (off + r * ld), ld, src.ptr + src.dtype.itemsize * r * cols, cols, k, cols))
            got.append(dst.numpy())
        want = np.full(n, 7, dst_t)
        with np.errstate(over="ignore"):
            want[off:].reshape(rows, ld)[:, :cols] = src.numpy().reshape(rows, cols).astype(dst_t)
        for g in got:
            assert np.array_equal(g, want, equal_nan=True)
        assert got[0].tobytes() == got[-1].tobytes()


@pytest.mark.parametrize("in_f16", [0, 1])
@pytest.mark.parametrize("table", [True, False])
@pytest.mark.parametrize("S,heads,kvh,off", [(256, 16, 8, 0), (768, 6, 2, 0), (256, 16, 16, 4), (256, 12, 12, 0), (256, 16, 4, 0)])
def test_attention_gradients(br, in_f16, S, heads, kvh, off, table):
    """a batch at once against one sequence after the other; off: results that do not start on a line"""
    hd, rng = 64, np.random.default_rng(S + heads)
    B = -(-LINE // (heads * hd * S)) + 1
    full, kv = heads * hd * S, kvh * hd * S
    t = np.float16 if in_f16 else np.float32
    ins = [br.DevArray.from_numpy(rng.standard_normal(B * full, dtype=np.float32).astype(t)) for _ in range(3)]
    cos, sin = br.rope_tables_dev(S, hd, 1e4) if table else (None, None)
    got = []
    for step in (B, 1):
        outs = [br.DevArray.from_numpy(np.full(B * k + off, 7, np.float32)) for k in (full, kv, kv)]
        for b, k in pieces(B, step):
            br.check(br.lib.mi355_attn_grads_finish_dev(*[o.ptr + 4 * (off + b * m) for o, m in zip(outs, (full, kv, kv))],
                                                        *[i.ptr + i.dtype.itemsize * b * full for i in ins], in_f16, 0, 0, 0,
                                                        heads, kvh, hd, S, k, cos, sin))
        got.append([o.numpy().tobytes() for o in outs])
    assert got[0] == got[1]
