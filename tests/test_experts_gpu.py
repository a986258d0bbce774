"""The chunk experts whose activation rows lie in LDS whole (depths of 512 to
2048): output rows that leave part of a workgroup, a wave or a tile idle,
depths of one to four pairs of units, every code width, items of one to
sixteen routes, against the exact kernels eight rows at a time."""
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
