"""The chunked GatedDeltaNet scan where its slices take another place: heads
that do and do not divide among eight XCDs (over groups too), a last chunk of
one token, an odd number of chunks, value heads sharing a key head, and a value
stride wider than its heads; against the float64 delta rule."""
import numpy as np
import pytest

from test_gdn_prefill_gpu import bf, inputs, run_chunked

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hk,hv,groups,t", [(1, 3, 1, 65), (2, 4, 2, 130), (4, 8, 1, 1),
                                            (8, 16, 1, 321), (3, 3, 3, 64)])
def test_scan_slices(mx, orc, hk, hv, groups, t):
    rows = groups * t
    q, k, v, g, beta = inputs(orc, rows, hk, hv, 40 + t, zero_decay_at=(rows // 2, 0))
    rng = np.random.default_rng(t)
    state = (rng.standard_normal((groups + 1, hv, 128, 128)) * 0.1).astype(np.float32)
    slots = np.arange(groups, 0, -1).astype(np.int32)
    y, st = run_chunked(mx, q, k, v, g, beta, hk, hv, groups, t, slots, state)
    assert (st[0] == state[0]).all()  # a slot not named
    rep = hv // hk
    q64, k64 = (np.repeat(bf(a).astype(np.float64), rep, axis=1) for a in (q, k))
    v64, b64, g64 = bf(v).astype(np.float64), bf(beta).astype(np.float64), g.astype(np.float64)
    for gi in range(groups):
        S = state[slots[gi]].astype(np.float64)
        out = np.empty((t, hv, 128))
        for i in range(t):
            r = gi * t + i
            S = S * g64[r][:, None, None]
            d = (v64[r] - np.einsum("hk,hkv->hv", k64[r], S)) * b64[r][:, None]
            S = S + k64[r][:, :, None] * d[:, None, :]
            out[i] = np.einsum("hk,hkv->hv", q64[r], S)
        # fp32 sums of at most 128 + 64 products a chunk: 2^-24 per sum, grown by
        # the inverse's few steps; the north star's bound is 1e-4
        assert np.abs(st[slots[gi]] - S).max() <= 1e-5 * np.abs(S).max()
        got = bf(y).astype(np.float64)[gi * t:(gi + 1) * t]
        assert np.all(np.abs(got - out) <= 2.0 ** -8 * np.abs(out) + 1e-5 * np.abs(out).max())
