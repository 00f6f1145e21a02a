"""mi355_sgemm_dev at the edges of its tiles (64 and 128 rows and columns, steps of 16 along K) and K slices, every transpose
case, operands at any element of a row."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (3, 5, 15), (64, 64, 16), (65, 63, 17), (127, 129, 33), (130, 66, 31), (64, 1024, 256),
                                   (1037, 259, 48), (5, 700, 2049), (256, 33, 4096)])
def test_sgemm_tile_edges(br, M, N, K, ta, tb):
    print("[case] sgemm tiles M=%d N=%d K=%d ta=%d tb=%d" % (M, N, K, ta, tb), flush=True)
    off = 1                                                   # the matrices start one float behind an aligned address
    A = H.normal(500, (K, M) if ta else (M, K)); B = H.normal(501, (N, K) if tb else (K, N)); C0 = H.normal(502, (M, N))
    put = lambda a: br.DevArray.from_numpy(np.concatenate([np.zeros(off, np.float32), a.ravel()]))
    ad, bd = put(A), put(B)
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    ref = (A64.T if ta else A64) @ (B64.T if tb else B64)
    mag = np.abs(A64.T if ta else A64) @ np.abs(B64.T if tb else B64)
    for alpha, beta in ((1.0, 0.0), (-0.75, 1.5)):
        cd = put(C0)
        br.check(br.lib.mi355_sgemm_dev(ta, tb, M, N, K, alpha, ad.ptr + 4 * off, A.shape[1], bd.ptr + 4 * off, B.shape[1],
                                        beta, cd.ptr + 4 * off, N))
        got = cd.numpy()[off:].reshape(M, N).astype(np.float64)
        want = alpha * ref + beta * C0
        # K products and sums, each rounded to 24 bits, and three more operations on the result
        bound = ((K + 1) * 2.0 ** -24) * abs(alpha) * mag + 3 * 2.0 ** -24 * (np.abs(want) + abs(beta) * np.abs(C0))
        assert np.all(np.abs(got - want) <= bound + 1e-30)
        assert cd.numpy()[0] == 0.0
