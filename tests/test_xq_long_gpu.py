"""mx_xq on long matrices (operands made once per workgroup, waves streaming
tiles): bit for bit the CPU oracle's, at the first size that takes this form,
at ragged last tiles, with more tiles than waves, and with scale rows that no
vector load may read."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

K = 2048
LONG = 16385  # rows from which this form runs


@pytest.mark.parametrize("n,bits,m,shift", [
    (LONG - 1, 8, 8, 0), (LONG, 4, 8, 0), (LONG, 6, 3, 0), (LONG, 8, 8, 0),
    (LONG + 1, 8, 1, 0), (LONG + 31, 4, 5, 0), (LONG + 17, 6, 8, 0),
    (LONG + 15, 4, 4, 1), (LONG + 9, 8, 7, 1), (LONG + 3, 6, 2, 1),
    (65536 + 16 * 40 + 5, 8, 6, 0)])  # 4096 waves: a second round, the last of them partial
def test_xq_long_bit_exact(mx, orc, n, bits, m, shift):
    seed = n + bits + m
    codes, s, b = orc.random_qweight(n, K, bits, 64, seed)
    x = orc.fill_bf16(m * K, seed + 7, 1, 1.0, 0.0).reshape(m, K)
    pad = np.zeros(shift, np.uint16)
    dc = mx.DeviceArray.from_numpy(codes)
    ds, db = (mx.DeviceArray.from_numpy(np.concatenate([pad, np.ravel(v)])) for v in (s, b))
    dx = mx.DeviceArray.from_numpy(x)
    dy = mx.DeviceArray.from_numpy(np.full((m + 1, n), 0x7FC0, np.uint16))
    qc = mx.QWeightC(dc.ptr, ds.ptr + 2 * shift, db.ptr + 2 * shift, n, K, bits, 64)
    mx.check(mx.lib.mx_xq(C.byref(qc), dx.ptr, m, dy.ptr, None))
    out = dy.numpy()
    assert (out[m] == 0x7FC0).all()  # nothing past the last row
    assert (out[:m] == orc.f32_to_bf16(orc.xq(codes, s, b, K, bits, x))).all()
