"""The hand-over kernels at the lines between their forms: values at and around half a step of the INT8 grid, where the product with the
reciprocal gives way to the division, and scales whose reciprocal is not a normal number; attention gradients on
rows of whole waves of columns and others, with one to five query heads to a KV head."""
import numpy as np
import pytest

import oracle as O
import test_gpu_parity as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def br():
    import ane_amd.bridge as b
    b.init()
    return b


def around_halves(scale):
    """(k + 1/2) * scale, a few floats to either side, and whole multiples, for every k of the grid and some beyond"""
    k = np.arange(-132, 133, dtype=np.float64)
    v = np.concatenate([k + 0.5, k]) * np.float64(scale)
    with np.errstate(over="ignore", invalid="ignore"):
        v = v.astype(np.float32)
        steps = [v]
        up = down = v
        for _ in range(4):
            up, down = np.nextafter(up, np.float32(np.inf)), np.nextafter(down, np.float32(-np.inf))
            steps += [up, down]
    return np.concatenate(steps)


@pytest.mark.parametrize("rounding", [0, 1])
@pytest.mark.parametrize("scale", [1.0, 0.0371, 1 / 3, 3.7e-5, 1e-30, 1.1e-38, 3e-42, 7e35, 2.1e38, -0.25])
def test_quantize_by_a_given_scale(br, scale, rounding):
    x = around_halves(scale)
    x = np.concatenate([x, np.array([0.0, -0.0, 3e38, -3e38, 1e-45], np.float32)])
    x = np.resize(x, (x.size + 3) // 4 * 4 + 3)
    xd, sd, q = br.DevArray.from_numpy(x), br.DevArray.from_numpy(np.array([scale], np.float32)), br.DevArray(x.size, np.int8)
    br.check(br.lib.mi355_int8_quant_dev(q.ptr, xd.ptr, sd.ptr, x.size, rounding))
    want = O.int8_quant(x, float(np.float32(scale)), rounding)
    assert np.array_equal(q.numpy(), want), np.flatnonzero(q.numpy() != want)[:10]


@pytest.mark.parametrize("rounding", [0, 1])
@pytest.mark.parametrize("top", [127.0, 1.0, 4.7e-6, 3.3e38, 1e-44, 0.0])
@pytest.mark.parametrize("n", [4, 5003, 300000])
def test_quantize_by_its_own_scale(br, n, top, rounding):
    x = np.resize(np.clip(around_halves(top / 127), -top, top), n).astype(np.float32)
    x[n // 2] = top
    scale = O.int8_scale(x)
    xd, sd, q = br.DevArray.from_numpy(x), br.DevArray(1), br.DevArray(n, np.int8)
    br.check(br.lib.mi355_int8_quantize_dynamic_dev(q.ptr, sd.ptr, xd.ptr, n, rounding))
    assert sd.numpy()[0] == np.float32(scale)
    assert np.array_equal(q.numpy(), O.int8_quant(x, scale, rounding))


@pytest.mark.parametrize("in_f16", [0, 1])
@pytest.mark.parametrize("B,heads,kvh,hd,S", [(1, 1, 1, 2, 256), (2, 6, 3, 6, 512), (1, 6, 2, 4, 768), (3, 5, 1, 10, 256), (2, 4, 4, 6, 252), (1, 10, 2, 2, 260),
                                              (2, 3, 1, 4, 9)])
def test_attention_gradients(br, B, heads, kvh, hd, S, in_f16):
    P.test_attn_grads_finish_equals_separate_steps(br, B, heads, kvh, hd, S, in_f16)


@pytest.mark.parametrize("rotate", [False, True])
@pytest.mark.parametrize("in_f16", [0, 1])
@pytest.mark.parametrize("ratio", [1, 2, 3, 4])
@pytest.mark.parametrize("S", [256, 260, 9, 3])
def test_heads_to_a_kv_head(br, S, ratio, in_f16, rotate):
    """one head and more, with and without the tables, zeros of either sign and infinities among the gradients; dQ, and for one head
    dK and dV, over their inputs where these are fp32"""
    B, kvh, hd, theta = 2, 3, 4, 1e4
    shape = (B, kvh * ratio * hd, S)
    src = [P.H.normal(1010 + i, shape) for i in range(3)]
    for k, a in enumerate(src):
        a.ravel()[k::7] = 0.0
        a.ravel()[k + 1::7] = -0.0
        a.ravel()[k + 5::97] = np.inf
    ins = [O.cvt_f32_f16(a) for a in src] if in_f16 else src
    cos, sin = br.rope_tables_dev(S, hd, theta) if rotate else (None, None)
    with np.errstate(invalid="ignore"):
        want = P._finish_reference(*ins, kvh * ratio, kvh, hd, theta, in_f16, rotate=rotate)
    for in_place in (False, True)[:1 if in_f16 else 2]:
        ind = [br.DevArray.from_numpy(a) for a in ins]
        outs = [br.DevArray(shape)] + [br.DevArray((B, kvh * hd, S)) for _ in range(2)]
        if in_place:
            outs = [ind[0]] + (ind[1:] if ratio == 1 else outs[1:])
        br.check(br.lib.mi355_attn_grads_finish_dev(*[o.ptr for o in outs], *[i.ptr for i in ind], in_f16, 0, 0, 0, kvh * ratio, kvh, hd, S, B, cos, sin))
        for got, ref in zip(outs, want):
            got = got.numpy().reshape(ref.shape)
            bits = got.view(np.uint32) == ref.astype(np.float32).view(np.uint32)
            assert np.all(bits | (np.isnan(got) & np.isnan(ref)))
