"""mi355_sgemm_dev where rows, columns or k come near 2^31: more workgroups than one launch numbers, and indices whose next
tile or step would leave 32 bits.  The operands are zero but for a few entries, so the results are exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BIG = 2 ** 31 - 1


class Sparse:
    """n floats on the device, zero but for the given entries."""

    def __init__(self, br, n, entries=()):
        self.br, self.n = br, n
        self.handle = br.lib.mi355_buf_alloc(4 * n)
        assert self.handle, br.last_error()
        self.ptr = br.lib.mi355_buf_devptr(self.handle)
        br.check(br.lib.mi355_buf_zero(self.handle))
        for i, v in entries:
            v = np.full(1, v, np.float32)
            br.lib.mi355_buf_write(self.handle, 4 * i, v.ctypes.data, 4)

    def at(self, i, n=1):
        out = np.empty(n, np.float32)
        self.br.lib.mi355_buf_read(self.handle, 4 * i, out.ctypes.data, 4 * n)
        return out

    def free(self):
        self.br.lib.mi355_buf_free(self.handle)


@pytest.mark.parametrize("knob", [-1, 1, 4])
@pytest.mark.parametrize("K", [BIG, 2 ** 30 + 5])
def test_k(br, K, knob):
    print("[case] sgemm K=%d knob=%d" % (K, knob), flush=True)
    at = [0, 1, 2 ** 30 - 1, 2 ** 30, 2 ** 30 + 1, K - 1]
    a, b = Sparse(br, K, [(i, 1 + j) for j, i in enumerate(at)]), Sparse(br, K, [(i, 2.0 ** j) for j, i in enumerate(at)])
    c = Sparse(br, 1, [(0, 3.0)])
    br.tune("gemm_split", knob)
    try:
        # (leading dimensions of 2^22 and more go through the fp32 instruction whatever the knob says)
        ta, ld = (1, 1) if knob > 0 else (0, K)
        br.check(br.lib.mi355_sgemm_dev(ta, 1 - ta, 1, 1, K, 2.0, a.ptr, ld, b.ptr, ld, 0.5, c.ptr, 1))
        assert c.at(0)[0] == 1.5 + 2 * sum((1 + j) * 2.0 ** j for j in range(len(at)))
        br.check(br.lib.mi355_sgemm_dev(1, 0, 1, 1, K, 0.0, a.ptr, 1, b.ptr, 1, 2.0, c.ptr, 1))
        assert c.at(0)[0] == 3.0 + 4 * sum((1 + j) * 2.0 ** j for j in range(len(at)))
    finally:
        br.tune("gemm_split", 0)
        for t in (a, b, c): t.free()


@pytest.mark.parametrize("knob", [-1, 1, 4])
@pytest.mark.parametrize("rows", [True, False])
def test_rows_and_columns(br, rows, knob):
    print("[case] sgemm %s=%d knob=%d" % ("M" if rows else "N", BIG, knob), flush=True)
    at = [0, 63, 64, 2 ** 26 - 1, 2 ** 26, 2 ** 29, 2 ** 30, BIG - 64, BIG - 1]
    a, c = Sparse(br, BIG, [(i, 1 + j) for j, i in enumerate(at)]), Sparse(br, BIG, [(i, 10) for i in at])
    b = Sparse(br, 1, [(0, 2.0)])
    br.tune("gemm_split", knob)
    try:
        if rows: br.check(br.lib.mi355_sgemm_dev(0, 0, BIG, 1, 1, 1.0, a.ptr, 1, b.ptr, 1, 1.0, c.ptr, 1))
        else: br.check(br.lib.mi355_sgemm_dev(0, 0, 1, BIG, 1, 1.0, b.ptr, 1, a.ptr, BIG, 1.0, c.ptr, BIG))
        for j, i in enumerate(at):
            assert c.at(i)[0] == 10 + 2 * (1 + j), i
        assert not np.any(c.at(65, 1000)) and not np.any(c.at(2 ** 26 + 1, 1000)) and not np.any(c.at(BIG - 63, 62))
    finally:
        br.tune("gemm_split", 0)
        for t in (a, b, c): t.free()
