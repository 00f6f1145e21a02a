"""RoPE on rows whose last group of columns is short, in both storages: out of place and in place; rows of less than a group; tensors at any element.  The same products and sums as the oracle's, so the same bits."""
import numpy as np
import pytest
import torch

import helpers as H
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def br():
    import ane_amd.bridge as b
    b.init()
    return b


def to_bf(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(torch.bfloat16).view(torch.int16).numpy().view(np.uint16)


def of_bf(a):
    return (a.astype(np.uint32) << 16).view(np.float32)


@pytest.mark.parametrize("storage", ["f32", "bf16"])
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("B,heads,kvh,hd,S", [(1, 1, 0, 2, 1), (2, 3, 1, 6, 3), (1, 2, 2, 4, 5), (2, 3, 2, 6, 7), (1, 2, 1, 4, 8), (3, 2, 1, 6, 9), (1, 0, 3, 8, 15),
                                              (5, 3, 3, 10, 54), (2, 4, 2, 64, 197), (3, 1, 1, 16, 259)])
def test_rope_tails(br, B, heads, kvh, hd, S, off, storage):
    print("[case] rope tails B=%d heads=%d/%d hd=%d S=%d off=%d %s" % (B, heads, kvh, hd, S, off, storage), flush=True)
    bf = storage == "bf16"
    fn = br.lib.mi355_rope_bf16_dev if bf else br.lib.mi355_rope_dev
    enc = to_bf if bf else (lambda a: a)
    dec = of_bf if bf else (lambda a: a)
    dtype, size = (np.uint16, 2) if bf else (np.float32, 4)
    q, k = enc(H.normal(810, (B, heads * hd, S))), enc(H.normal(811, (B, kvh * hd, S)))
    cos, sin = br.rope_tables_dev(S, hd, 1e4)
    put = lambda a: br.DevArray.from_numpy(np.concatenate([np.full(off, 7, dtype), a.ravel(), np.full(9, 7, dtype)]))

    def check(d, want):
        got = d.numpy()
        assert got[off:off + want.size].tobytes() == want.tobytes()
        assert np.all(got[:off] == 7) and np.all(got[off + want.size:] == 7)

    def rotated(a, n, direction):
        if n == 0:
            return a
        # the oracle takes [heads*hd][S]; sequences are independent
        return enc(np.stack([O.rope(np.ascontiguousarray(dec(s)), hd, 1e4, direction) for s in a]))

    for direction in (1, -1):
        want_q, want_k = rotated(q, heads, direction), rotated(k, kvh, direction)
        for in_place in (False, True):
            qi, ki = put(q), put(k)
            qo, ko = (qi, ki) if in_place else (put(np.zeros_like(q)), put(np.zeros_like(k)))
            at = lambda d, n: d.ptr + size * off if n else None
            br.check(fn(at(qo, heads), at(ko, kvh), at(qi, heads), at(ki, kvh), heads, kvh, hd, S, B, cos, sin, direction))
            check(qo, want_q)
            check(ko, want_k)
