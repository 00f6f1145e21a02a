"""mi355_sgemm_dev with B split by a launch of its own: edges of the tiles (96 and 64 rows, 256 columns, 32 columns of a wave,
steps of 64 k, two groups of 32), ranges of columns, every bit of an operand, special values of either operand, and a tile's
pitch.  The knobs are those of the kernels: 5 and 6 tiles of 96 x 256 and 64 x 256, 7 and 8 whole rows of A (K <= 256, 384)."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu
KNOBS = [5, 6, 7, 8]
TRANS = [(0, 0), (1, 0), (0, 1), (1, 1)]


@pytest.fixture(scope="module")
def br():
    import ane_amd.bridge as b
    b.init()
    return b


def product(br, knob, A, B, ta, tb, alpha=1.0, beta=0.0, C0=None, off=0, splitk=0, pad=0):
    """Operands as stored -> C; every matrix starts `off` floats behind an aligned address, C's rows are `pad` floats apart."""
    M, K = A.shape[::-1] if ta else A.shape
    N = B.shape[0] if tb else B.shape[1]
    put = lambda a: br.DevArray.from_numpy(np.concatenate([np.zeros(off, np.float32), a.ravel()]))
    full = np.full((M, N + pad), 7.0 if pad else np.nan, np.float32)
    if C0 is not None:
        full[:, :N] = C0
    ad, bd, cd = put(A), put(B), put(full)
    br.tune("gemm_split", knob)
    br.tune("gemm_splitk", splitk)
    try:
        br.check(br.lib.mi355_sgemm_dev(ta, tb, M, N, K, alpha, ad.ptr + 4 * off, A.shape[1], bd.ptr + 4 * off, B.shape[1],
                                        beta, cd.ptr + 4 * off, N + pad))
        out = cd.numpy()[off:].reshape(M, N + pad)
    finally:
        br.tune("gemm_split", 0)
        br.tune("gemm_splitk", 0)
    assert np.all(out[:, N:] == 7.0)                     # what lies between the rows is not touched
    return out[:, :N]


@pytest.mark.parametrize("knob", KNOBS)
@pytest.mark.parametrize("ta,tb", TRANS)
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (95, 33, 31), (97, 255, 65), (64, 256, 64), (193, 513, 127), (300, 31, 256), (65, 1057, 200)])
def test_planes_edges(br, M, N, K, ta, tb, knob):
    print("[case] sgemm planes M=%d N=%d K=%d ta=%d tb=%d knob=%d" % (M, N, K, ta, tb, knob), flush=True)
    A = H.normal(700, (K, M) if ta else (M, K)); B = H.normal(701, (N, K) if tb else (K, N)); C0 = H.normal(702, (M, N))
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    ref = (A64.T if ta else A64) @ (B64.T if tb else B64)
    mag = np.abs(A64.T if ta else A64) @ np.abs(B64.T if tb else B64)
    for alpha, beta, pad in ((1.0, 0.0, 0), (-0.75, 1.5, 3)):
        got = product(br, knob, A, B, ta, tb, alpha, beta, None if beta == 0.0 else C0, off=1, pad=pad).astype(np.float64)
        want = alpha * ref + beta * C0
        # per 32 values of k six instructions within 2^-23 of the sum of magnitudes and one addition; the sum of the groups; what
        # is left out of a product is below 2^-24 of it; three more operations on the result
        bound = (7 * (K // 32 + 2) + 2) * 2.0 ** -23 * abs(alpha) * mag + 3 * 2.0 ** -24 * (np.abs(want) + abs(beta) * np.abs(C0))
        assert np.all(np.abs(got - want) <= bound)


@pytest.mark.parametrize("knob,K,splitk", [(5, 1000, 1), (5, 1000, 3), (6, 1000, 4), (6, 64, 1), (7, 256, 1), (8, 384, 1), (8, 300, 1)])
def test_planes_are_as_accurate_as_the_other_split(br, knob, K, splitk):
    """Against 64 bits, normal operands: no further off than the tiles of 64 x 64 that split both operands, in the same number
    of slices (2-norms)."""
    M, N = 700, 600
    A = H.normal(710, (M, K)); B = H.normal(711, (K, N))
    ref = A.astype(np.float64) @ B.astype(np.float64)
    err = lambda k, s: np.linalg.norm(product(br, k, A, B, 0, 0, splitk=s) - ref) / np.linalg.norm(ref)
    # (at 64 k and fewer both are one rounding or two of the result; a twentieth for that)
    assert err(knob, splitk) <= 1.05 * err(3, splitk)


@pytest.mark.parametrize("scale", [1.0, 2.0 ** -108, 2.0 ** -109, 2.0 ** -120])
@pytest.mark.parametrize("K,splitk", [(70, 0), (200, 3)])
@pytest.mark.parametrize("ta,tb", TRANS)
def test_planes_hold_every_bit(br, ta, tb, K, splitk, scale):
    """One operand has a single power of two per row or column, so nothing is rounded in any order and the bits must agree (as
    in test_gpu_sgemm_split.py); the smaller scales leave bits out of a split, of A in one block of rows, of B in a few units
    of columns."""
    M, N = 130, 200
    rng = np.random.default_rng(720)
    full = lambda shape: ((1 + rng.random(shape)) * rng.choice([-1.0, 1.0], shape)).astype(np.float32)
    pick = np.zeros((K, N), np.float32)
    pick[rng.integers(0, K, N), np.arange(N)] = 2.0 ** rng.integers(-3, 20, N)
    pick[:, 0] = 0; pick[K - 1, 0] = 1.0                                 # the last value of the last slice
    A = full((M, K)) * np.float32(scale)
    if scale < 1:
        A[70:] = full((M - 70, K))
    for swap in (False, True):
        X, Y = (pick.T, A.T) if swap else (A, pick)
        want = (X.astype(np.float64) @ Y.astype(np.float64)).astype(np.float32)
        Xs, Ys = np.ascontiguousarray(X.T if ta else X), np.ascontiguousarray(Y.T if tb else Y)
        for knob in KNOBS:
            got = product(br, knob, Xs, Ys, ta, tb, splitk=splitk)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), knob


@pytest.mark.parametrize("beta", [0.0, 1.5])
@pytest.mark.parametrize("K,splitk", [(70, 0), (200, 3)])
@pytest.mark.parametrize("ta,tb", TRANS)
def test_planes_give_infinities_and_nans_of_fp32(br, ta, tb, K, splitk, beta):
    M, N = 300, 300
    A = H.normal(730, (M, K)); B = H.normal(731, (K, N)); C0 = H.normal(732, (M, N))
    mid = K // 2
    A[3, 5] = np.inf; A[140, K - 1] = -np.inf; A[141, 0] = np.nan; A[75, mid] = np.inf; A[299, K - 1] = np.nan
    A[7, 1] = np.finfo(np.float32).max          # rounds to an infinity in 8 bits
    B[64, 260] = np.inf; B[mid, 130] = -np.inf; B[K - 2, 70] = np.nan; B[2, 33] = np.finfo(np.float32).max
    B[1, 17] = 0.0; B[5, 4] = 0.0
    As, Bs = np.ascontiguousarray(A.T if ta else A), np.ascontiguousarray(B.T if tb else B)
    c = C0 if beta else None
    want = product(br, -1, As, Bs, ta, tb, 1.0, beta, c, splitk=splitk)
    for knob in KNOBS:
        got = product(br, knob, As, Bs, ta, tb, 1.0, beta, c, splitk=splitk)
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
        assert np.array_equal(np.sign(got[np.isinf(got)]), np.sign(want[np.isinf(want)]))
        ok = np.isfinite(want)
        with np.errstate(invalid="ignore"):
            mag = np.abs(A.astype(np.float64)) @ np.abs(B.astype(np.float64)) + abs(beta) * np.abs(C0)
        assert np.all(np.abs(got[ok].astype(np.float64) - want[ok]) <= (K + 20) * 2.0 ** -23 * mag[ok])


def test_planes_alpha_zero_reads_no_operand(br):
    A = np.full((40, 100), np.nan, np.float32); B = np.full((100, 50), np.inf, np.float32); C0 = H.normal(740, (40, 50))
    for knob in KNOBS:
        assert np.array_equal(product(br, knob, A, B, 0, 0, alpha=0.0, beta=2.0, C0=C0), 2.0 * C0)
        assert not np.any(product(br, knob, A, B, 0, 0, alpha=0.0))


def test_many_columns_in_ranges(br):
    """Few rows and more units of 32 columns than a workgroup's waves take in one turn: several turns, several ranges."""
    M, N, K = 70, 3001, 96
    A = H.normal(750, (M, K)); B = H.normal(751, (K, N)); C0 = H.normal(752, (M, N))
    want = A.astype(np.float64) @ B.astype(np.float64) + 0.5 * C0
    mag = np.abs(A.astype(np.float64)) @ np.abs(B.astype(np.float64))
    for knob in (7, 8):
        got = product(br, knob, A, B, 0, 0, 1.0, 0.5, C0)
        assert np.all(np.abs(got - want) <= 7 * 5 * 2.0 ** -23 * mag + 3 * 2.0 ** -24 * (np.abs(want) + np.abs(C0)))


@pytest.mark.parametrize("knob", KNOBS)
@pytest.mark.parametrize("M", [1, 2, 65, 66, 97, 98, 127, 191])
def test_planes_write_nothing_outside_c(br, M, knob):
    """Last blocks of 1, 2, 63 and 95 rows: a whole block of rows in front of C and one behind its last row keep their values, and
    what lies there is not read either (it would make a NaN of a sum)."""
    for N, beta, pad in ((70, 0.0, 0), (70, 1.5, 3), (33, 1.5, 0), (300, 0.0, 5)):
        K, ldc, guard = 100, N + pad, 96 * (N + pad)
        print("[case] sgemm planes guards M=%d N=%d knob=%d beta=%g pad=%d" % (M, N, knob, beta, pad), flush=True)
        A = H.normal(760, (M, K)); B = H.normal(761, (K, N)); C0 = H.normal(762, (M, N))
        inside = np.full((M, ldc), np.nan, np.float32)
        inside[:, :N] = C0 if beta else np.nan
        fence = np.full(guard, np.nan, np.float32)
        buf = br.DevArray.from_numpy(np.concatenate([fence, inside.ravel(), fence]))
        ad, bd = br.DevArray.from_numpy(A), br.DevArray.from_numpy(B)
        br.tune("gemm_split", knob)
        try:
            br.check(br.lib.mi355_sgemm_dev(0, 0, M, N, K, 1.0, ad.ptr, K, bd.ptr, N, beta, buf.ptr + 4 * guard, ldc))
            got = buf.numpy()
        finally:
            br.tune("gemm_split", 0)
        same = lambda a: np.array_equal(a.view(np.uint32), np.full(a.size, fence[:1].view(np.uint32)[0]))
        out = got[guard:guard + M * ldc].reshape(M, ldc)
        assert same(got[:guard]) and same(got[guard + M * ldc:]) and same(np.ascontiguousarray(out[:, N:]).ravel())
        mag = np.abs(A.astype(np.float64)) @ np.abs(B.astype(np.float64))
        want = A.astype(np.float64) @ B.astype(np.float64) + beta * C0
        bound = (7 * (K // 32 + 2) + 2) * 2.0 ** -23 * mag + 3 * 2.0 ** -24 * (np.abs(want) + beta * np.abs(C0))
        assert np.all(np.abs(out[:, :N] - want) <= bound)


@pytest.mark.parametrize("M,N,K,knob", [(4096, 4096, 4096, 1), (256, 256, 4096, -1), (24573, 256, 1024, 5)])
def test_the_quickest_kernel_is_chosen(br, M, N, K, knob):
    """Planes of a large operand that every tile reads again, many slices of a small output, and the classifier's logits: the choice
    is seen by the bits, which differ between the kernels."""
    print("[case] sgemm choice M=%d N=%d K=%d knob=%d" % (M, N, K, knob), flush=True)
    A, B = H.normal(770, (M, K)), H.normal(771, (K, N))
    got = {k: product(br, k, A, B, 0, 0).tobytes() for k in (0, -1, 1, 4, 5)}
    assert got[0] == got[knob] and all(got[0] != got[k] for k in (-1, 1, 4, 5) if k != knob)
