"""The multi-tensor norm and update at the edges of their block tables: 64 tensors to a launch, 1024 elements to a block of the
update and 8192 to one of the norm, tensors of a few elements, ends within a 128-bit group."""
import ctypes as C

import numpy as np
import pytest

import helpers as H
import oracle as O

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 3, 4, 5, 1023, 1024, 1025, 1027, 8188, 8191, 8192, 8193, 8196, 40961]


@pytest.mark.parametrize("sizes", [[1], [3], [8192], [8193, 7], EDGES, [5] * 63, [5] * 64, [1029] * 65, EDGES * 9 + [300001]],
                         ids=lambda s: "%dx%d" % (len(s), sum(s)))
def test_every_element_belongs_to_one_block(br, sizes):
    print("[case] optimizer blocks", len(sizes), "tensors,", sum(sizes), "elements", flush=True)
    k, pre = len(sizes), np.float32(0.5)
    at = np.concatenate([[0], np.cumsum([(n + 3) // 4 * 4 + 4 for n in sizes])])        # a gap of 4 or more behind each
    w, g, m, v = (H.normal(700 + i, int(at[-1])) for i in range(4))
    v = np.abs(v)
    wd = [0.1 * (i % 3) for i in range(k)]
    bufs = [br.DevArray.from_numpy(a) for a in (w, g, m, v)]
    arrs = [(C.c_void_p * k)(*[b.ptr + 4 * int(a) for a in at[:-1]]) for b in bufs]
    ns, wds = (C.c_size_t * k)(*sizes), (C.c_float * k)(*wd)
    ss = br.DevArray.from_numpy(np.full(1, 2.0, np.float32))
    br.check(br.lib.mi355_sumsq_accum_multi_dev(ss.ptr, arrs[1], ns, k, pre))
    want = 2.0 + sum(float(np.sum((g[a:a + n] * pre).astype(np.float64) ** 2)) for a, n in zip(at, sizes))
    # a lane adds 8 terms to each of 4 sums, then two, 6 + 2 levels of a tree, up to 14 partials, 10 levels: all positive
    assert abs(float(ss.numpy()[0]) - want) <= 44 * 2.0 ** -24 * want
    br.check(br.lib.mi355_adam_update_multi_dev(*arrs, ns, wds, k, 3, 1e-3, 0.9, 0.95, 1e-8, pre, None, 1))
    got = [b.numpy() for b in bufs]
    for i, (a, n) in enumerate(zip(at, sizes)):
        one = [br.DevArray.from_numpy(x[a:a + n].copy()) for x in (w, g, m, v)]
        br.check(br.lib.mi355_adam_update_dev(*[o.ptr for o in one], n, 3, 1e-3, 0.9, 0.95, 1e-8, wd[i], pre, None, 1))
        for x, o in zip(got, one):
            assert x[a:a + n].tobytes() == o.numpy().tobytes(), (i, n)
    gap = np.ones(int(at[-1]), bool)
    for a, n in zip(at, sizes):
        gap[a:a + n] = False
    for x, x0 in zip(got, (w, g, m, v)):
        assert x[gap].tobytes() == x0[gap].tobytes()
    rw, rm, rv = O.adam_update(w[:sizes[0]], g[:sizes[0]] * pre, m[:sizes[0]], v[:sizes[0]], 3, 1e-3, 0.9, 0.95, 1e-8, wd[0])
    assert H.rel_err(got[0][:sizes[0]], rw) <= 1e-5
