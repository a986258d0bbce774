"""mx_qmm beyond 16 rows: every form of the GEMM that it takes without room for
partial sums (the tiles of 64 weight rows x 64, 96, 128 and 256 activation
rows; the split of k over a workgroup's waves with each of its tile shapes), at
row and column remainders, one and odd numbers of groups, one and several
stages for a wave, against the float64 closed form.  (The split of k over
workgroups: test_prefill_layers_gpu.py.)"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bf(h):
    return (np.asarray(h, np.uint16).astype(np.uint32) << 16).view(np.float32)


@pytest.mark.parametrize("bits", [4, 5, 6, 8])
@pytest.mark.parametrize("m,n,k", [
    (38, 31, 64), (67, 12139, 64), (100, 16387, 64), (386, 12559, 64),  # tiles, one group
    (38, 22, 512), (34, 2197, 384), (17, 4259, 384), (38, 4131, 448), (51, 4366, 640),  # k split
    (17, 65, 320), (512, 70, 192), (129, 6001, 192)])
def test_gemm_forms(mx, orc, m, n, k, bits):
    check(mx, orc, m, n, k, bits)


# k over a workgroup's waves with several stages for each of them, a number of
# stages that the waves do not divide, and an odd last group; tiles over
# several groups
@pytest.mark.parametrize("bits", [4, 5, 6, 8])
@pytest.mark.parametrize("form,m,n,k", [
    ("D1.2", 17, 40, 2112), ("D1.2", 90, 264, 8128), ("D1.3", 33, 2049, 2112),
    ("D1.3", 512, 264, 4096), ("D2.2", 49, 2049, 2176), ("D2.2", 128, 2048, 4160),
    ("D2.3", 100, 2049, 2112), ("D2.3", 160, 2048, 4160), ("D2.4", 512, 1000, 2112),
    ("D2.4", 200, 1999, 2112), ("T2.1", 77, 5001, 192), ("T3.1", 77, 12001, 192),
    ("T4.1", 385, 8001, 192), ("T8.1", 385, 16001, 192)])
def test_gemm_forms_by_name(mx, orc, gemm_plan, form, m, n, k, bits):
    assert gemm_plan(m, n, k, bits) == form
    check(mx, orc, m, n, k, bits)


def check(mx, orc, m, n, k, bits):
    seed = 4100 + m + n + bits
    w = mx.QWeight.random(n, k, bits, 64, seed)
    codes, s, b = orc.random_qweight(n, k, bits, 64, seed)
    x = orc.fill_bf16(m * k, seed + 7, 1, 1.0, 0.0).reshape(m, k)
    dx = mx.DeviceArray.from_numpy(x)
    dy = mx.DeviceArray.from_numpy(np.full((m + 1, n), 0x7FC0, np.uint16))
    qc = w.c()
    mx.check(mx.lib.mx_qmm(C.byref(qc), dx.ptr, m, dy.ptr, None))
    out = dy.numpy()
    assert (out[m] == 0x7FC0).all()  # nothing past the last row
    got = bf(out[:m]).astype(np.float64)
    y64 = orc.qmv_f64(codes, s, b, k, bits, 64, x)
    # one bf16 rounding, and fp32 sums of weights kept to 2^-17
    mag = np.abs(bf(x)).astype(np.float64).sum(axis=1, keepdims=True) * (2.0 ** bits * 0.03 + 0.2)
    assert np.all(np.abs(got - y64) <= 2.0 ** -8 * np.abs(y64) + 2.0 ** -16 * mag + 1e-6)
