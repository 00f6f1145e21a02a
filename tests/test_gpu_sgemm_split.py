"""mi355_sgemm_dev through the bfloat16 matrix instruction, fp32 values as sums of three: tile edges in every transpose case,
every bit of an operand, and the values that such a sum cannot hold, which have to give what the fp32 instruction gives."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu


def product(br, knob, A, B, ta, tb, alpha=1.0, beta=0.0, C0=None, off=0, splitk=0):
    """(M, N, K of the operands as stored) -> C; every matrix starts `off` floats behind an aligned address."""
    M, K = A.shape[::-1] if ta else A.shape
    N = B.shape[0] if tb else B.shape[1]
    put = lambda a: br.DevArray.from_numpy(np.concatenate([np.zeros(off, np.float32), a.ravel()]))
    ad, bd, cd = put(A), put(B), put(np.full((M, N), np.nan, np.float32) if C0 is None else C0)
    br.tune("gemm_split", knob)
    br.tune("gemm_splitk", splitk)
    try:
        br.check(br.lib.mi355_sgemm_dev(ta, tb, M, N, K, alpha, ad.ptr + 4 * off, A.shape[1], bd.ptr + 4 * off, B.shape[1],
                                        beta, cd.ptr + 4 * off, N))
        return cd.numpy()[off:].reshape(M, N)
    finally:
        br.tune("gemm_split", 0)
        br.tune("gemm_splitk", 0)


@pytest.mark.parametrize("knob", [1, 2, 3, 4])
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (127, 257, 31), (129, 255, 33), (256, 256, 64), (300, 130, 97), (70, 3, 700)])
def test_split_tile_edges(br, M, N, K, ta, tb, knob):
    print("[case] sgemm split M=%d N=%d K=%d ta=%d tb=%d knob=%d" % (M, N, K, ta, tb, knob), flush=True)
    A = H.normal(600, (K, M) if ta else (M, K)); B = H.normal(601, (N, K) if tb else (K, N)); C0 = H.normal(602, (M, N))
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    ref = (A64.T if ta else A64) @ (B64.T if tb else B64)
    mag = np.abs(A64.T if ta else A64) @ np.abs(B64.T if tb else B64)
    for alpha, beta in ((1.0, 0.0), (-0.75, 1.5)):
        got = product(br, knob, A, B, ta, tb, alpha, beta, None if beta == 0.0 else C0, off=1).astype(np.float64)
        want = alpha * ref + beta * C0
        # six instructions per 32 values of k, each within 2^-23 of the sum of magnitudes (rounded or cut off), slices added
        # the same way; what is left out of a product is below 2^-24 of it; three more operations on the result.  (K = 1 and a
        # few hundred terms of one size would not notice a missing third: test_split_holds_every_bit.)
        bound = (6 * (K // 32 + 2) + 1) * 2.0 ** -23 * abs(alpha) * mag + 3 * 2.0 ** -24 * (np.abs(want) + abs(beta) * np.abs(C0))
        assert np.all(np.abs(got - want) <= bound)


# one slice; three of 96, 96 and 8 values of k (128 and 72 in two groups)
SLICED = [(70, 0), (200, 3)]


@pytest.mark.parametrize("scale", [1.0, 2.0 ** -95, 2.0 ** -108, 2.0 ** -109, 2.0 ** -113, 2.0 ** -120])
@pytest.mark.parametrize("K,splitk", SLICED)
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_split_holds_every_bit(br, ta, tb, K, splitk, scale):
    """One operand has a single power of two per row or column, so every element of the result is an element of the other
    times that power and every partial sum of its thirds is an fp32 value: nothing is rounded in any order and the bits must
    agree.  A missing third is an error of up to 2^-16.  The smaller scales make the last third a subnormal bfloat16 value and
    then none at all (all of 24 bits down to 2^-109, 2^-110 and below not), which only some tiles are computed again for."""
    M, N = 130, 200
    rng = np.random.default_rng(620)
    full = lambda shape: ((1 + rng.random(shape)) * rng.choice([-1.0, 1.0], shape)).astype(np.float32)
    pick = np.zeros((K, N), np.float32)
    pick[rng.integers(0, K, N), np.arange(N)] = 2.0 ** rng.integers(-3, 20, N)
    pick[:, 0] = 0; pick[K - 1, 0] = 1.0                                 # the last value of the last slice
    A = full((M, K)) * np.float32(scale)
    if scale < 1:
        A[64:] = full((M - 64, K))                                       # tiles without small values beside tiles with them
    for swap in (False, True):
        X, Y = (pick.T, A.T) if swap else (A, pick)
        want = (X.astype(np.float64) @ Y.astype(np.float64)).astype(np.float32)
        Xs, Ys = np.ascontiguousarray(X.T if ta else X), np.ascontiguousarray(Y.T if tb else Y)
        for knob in (1, 2, 3, 4):
            got = product(br, knob, Xs, Ys, ta, tb, splitk=splitk)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), knob


@pytest.mark.parametrize("beta", [0.0, 1.5])
@pytest.mark.parametrize("K,splitk", SLICED)
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_split_gives_infinities_and_nans_of_fp32(br, ta, tb, K, splitk, beta):
    M, N = 300, 300
    A = H.normal(610, (M, K)); B = H.normal(611, (K, N)); C0 = H.normal(612, (M, N))
    mid = K // 2                                # in the second of three slices
    A[3, 5] = np.inf; A[140, K - 1] = -np.inf; A[141, 0] = np.nan; A[75, mid] = np.inf; A[299, K - 1] = np.nan
    A[7, 1] = np.finfo(np.float32).max          # rounds to an infinity in 8 bits
    A[200, mid] = np.finfo(np.float32).max
    B[64, 260] = np.inf; B[mid, 130] = -np.inf; B[K - 2, 70] = np.nan; B[1, 17] = 0.0; B[5, 4] = 0.0
    As, Bs = np.ascontiguousarray(A.T if ta else A), np.ascontiguousarray(B.T if tb else B)
    c = C0 if beta else None
    want = product(br, -1, As, Bs, ta, tb, 1.0, beta, c, splitk=splitk)
    for knob in (1, 2, 3, 4):
        got = product(br, knob, As, Bs, ta, tb, 1.0, beta, c, splitk=splitk)
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
        assert np.array_equal(np.sign(got[np.isinf(got)]), np.sign(want[np.isinf(want)]))
        ok = np.isfinite(want)
        with np.errstate(invalid="ignore"):
            mag = np.abs(A.astype(np.float64)) @ np.abs(B.astype(np.float64)) + abs(beta) * np.abs(C0)
        assert np.all(np.abs(got[ok].astype(np.float64) - want[ok]) <= (K + 20) * 2.0 ** -23 * mag[ok])


def test_alpha_zero_reads_no_operand(br):
    A = np.full((40, 300), np.nan, np.float32); B = np.full((300, 50), np.inf, np.float32); C0 = H.normal(630, (40, 50))
    for knob in (-1, 1, 3, 4):
        assert np.array_equal(product(br, knob, A, B, 0, 0, alpha=0.0, beta=2.0, C0=C0), 2.0 * C0)
        assert not np.any(product(br, knob, A, B, 0, 0, alpha=0.0))


@pytest.fixture(scope="module")
def br():
    import ane_amd.bridge as b
    b.init()
    return b
