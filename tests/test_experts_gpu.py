"""The chunk experts whose activation rows lie in LDS whole (depths that are
multiples of 512, up to 2048, with scales on 16 bytes): output rows that leave part of a workgroup, a wave or a tile idle,
depths of one to four pairs of units, every code width, items of one to
sixteen routes, against the exact kernels eight rows at a time.  And the
general forms, which keep the other depths and unaligned scales."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bf(h):
    return (np.asarray(h, np.uint16).astype(np.uint32) << 16).view(np.float32)


@pytest.mark.parametrize("gbits,dbits,H,I,rows", [
    (4, 5, 1536, 576, 33), (5, 4, 512, 1024, 9), (6, 6, 1024, 512, 50), (8, 8, 2048, 64, 17),
    (4, 8, 512, 512, 21), (4, 6, 2048, 1536, 12)])
def test_chunk_experts_in_lds(mx, orc, gbits, dbits, H, I, rows):
    from test_layers_gpu import Moe
    from test_qmm_gpu import _experts_mfma

    E, top_k = 24, 5
    m = Moe(mx, orc, E, I, H, seed=300 + gbits * 10 + dbits, gbits=gbits, dbits=dbits)
    m.ws = mx.DeviceArray((mx.lib.mx_moe_workspace_bytes(rows, top_k, I),), np.uint8)
    rng = np.random.default_rng(H + rows)
    ids = np.stack([rng.choice(E, top_k, replace=False) for _ in range(rows)]).astype(np.uint32)
    scores = orc.f32_to_bf16(rng.uniform(0.05, 0.5, (rows, top_k)).astype(np.float32))
    x = orc.fill_bf16(rows * H, 310 + rows, 1, 1.0, 0.0).reshape(rows, H)
    got = bf(_experts_mfma(mx, m, x, ids, scores, top_k)).astype(np.float64)
    ws = m.ws
    m.ws = mx.DeviceArray((mx.lib.mx_moe_workspace_bytes(8, top_k, I),), np.uint8)
    want = np.concatenate([m.run(mx, x[r:r + 8], ids[r:r + 8], scores[r:r + 8], top_k)
                           for r in range(0, rows, 8)])
    m.ws = ws
    want = bf(want).astype(np.float64)
    # the bound of the other matrix-core expert tests: h and the output are
    # rounded to bf16, so a sum in another order may round either way
    scale = np.abs(want).max(axis=2, keepdims=True)
    assert np.all(np.abs(got - want) <= 2e-2 * np.abs(want) + 1e-2 * scale)
    assert np.mean(got == want) > 0.5


def _general(mx, orc, m, rows, top_k, E, seed):
    from test_qmm_gpu import _experts_mfma

    m.ws = mx.DeviceArray((mx.lib.mx_moe_workspace_bytes(rows, top_k, m.I),), np.uint8)
    rng = np.random.default_rng(seed)
    ids = np.stack([rng.choice(E, top_k, replace=False) for _ in range(rows)]).astype(np.uint32)
    scores = orc.f32_to_bf16(rng.uniform(0.05, 0.5, (rows, top_k)).astype(np.float32))
    x = orc.fill_bf16(rows * m.H, seed + 1, 1, 1.0, 0.0).reshape(rows, m.H)
    got = bf(_experts_mfma(mx, m, x, ids, scores, top_k)).astype(np.float64)
    want = bf(np.concatenate([m.oracle(orc, x[r:r + 8], ids[r:r + 8], scores[r:r + 8], top_k)
                              for r in range(0, rows, 8)])).astype(np.float64)
    scale = np.abs(want).max(axis=2, keepdims=True)  # the bound of the tests above
    assert np.all(np.abs(got - want) <= 2e-2 * np.abs(want) + 1e-2 * scale)
    assert np.mean(got == want) > 0.5


# whole batches of four groups (4 and 8 bits: 32-row tiles), rows that do not
# fit LDS, and depths of an odd number of groups
@pytest.mark.parametrize("bits", [4, 5, 6, 8])
@pytest.mark.parametrize("H,I", [(768, 256), (2304, 320), (448, 768)])
def test_chunk_experts_other_depths(mx, orc, bits, H, I):
    from test_layers_gpu import Moe

    E, top_k, rows = 16, 4, 37
    m = Moe(mx, orc, E, I, H, seed=900 + bits * 10, gbits=bits, dbits=bits)
    _general(mx, orc, m, rows, top_k, E, H + bits)


@pytest.mark.parametrize("bits", [4, 5, 6, 8])
def test_chunk_experts_scales_off_16_bytes(mx, orc, bits):
    """Depths that fit LDS, but scales and biases one value past an aligned
    address: no vector load may read them."""
    from test_layers_gpu import Moe

    E, top_k, rows, H, I = 16, 4, 29, 1024, 512
    m = Moe(mx, orc, E, I, H, seed=950 + bits, gbits=bits, dbits=bits)
    keep = []

    def shift(w, host, make):
        c = w.c()
        keep.append(w)  # its codes are used where they are
        arrays = []
        for v in host[1:]:
            a = mx.DeviceArray.from_numpy(np.concatenate([np.zeros(1, np.uint16), np.ravel(v)]))
            keep.append(a)
            arrays.append(a.ptr + 2)
        return make(c, *arrays)

    def bank(c, s, b):
        return mx.QBankC(c.codes, s, b, c.experts, c.n, c.k, c.bits, c.group_size)

    def weight(c, s, b):
        return mx.QWeightC(c.codes, s, b, c.n, c.k, c.bits, c.group_size)

    class Shifted:
        def __init__(self, c):
            self.c = lambda: c

    m.gate, m.up, m.down = (Shifted(shift(w, h, bank))
                            for w, h in zip((m.gate, m.up, m.down), m.h_host))
    m.sg, m.su, m.sd = (Shifted(shift(w, h, weight))
                        for w, h in zip((m.sg, m.su, m.sd), m.s_host))
    _general(mx, orc, m, rows, top_k, E, 970 + bits)
