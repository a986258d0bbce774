"""One layer of a prompt chunk (the GEMM's epilogues in place: the low-rank
hyper-connection projections and the output projections that write the four
residual streams) against the same prompt eight tokens at a time, output by
output, at row counts and widths that leave tiles, slices and groups partial."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bf(h):
    return (np.asarray(h, np.uint16).astype(np.uint32) << 16).view(np.float32)


# attention (attn_every 1) or GatedDeltaNet (2) output projections 4096 or 1024
# deep; hidden 1600: 100 groups of the streams, which 16 slices
# do not divide (the last is empty)
MODELS = {
    "attn4": dict(hidden=2048, attn_every=1, heads=16, kv_heads=2, head_dim=256, bits=4),
    "gdn4": dict(hidden=2048, attn_every=2, gdn_hk=16, gdn_hv=32, bits=4),
    "gdn5": dict(hidden=1600, attn_every=2, gdn_hk=4, gdn_hv=8, bits=5),
    "attn5": dict(hidden=1600, attn_every=1, heads=8, kv_heads=4, head_dim=128, bits=5),
    "gdn6": dict(hidden=1600, attn_every=2, gdn_hk=4, gdn_hv=8, bits=6),
}


@pytest.fixture(scope="module", params=sorted(MODELS))
def engine(request, mx):
    cfg = dict(mx.TINY, layers=1, hc_rank=256, moe_inter=256, shared_inter=256, max_slots=2,
               rotary_dim=64, seed=31, **MODELS[request.param])
    eng = mx.Engine(cfg)
    eng.set_flags(exact=False)
    yield eng, cfg
    eng.close()


def blocks(eng, cfg, prompt):
    """The layer's streams and routes, eight tokens at a time."""
    n, H, K = len(prompt), cfg["hc"] * cfg["hidden"], cfg["top_k"]
    h, ids = np.empty((n, H)), np.empty((n, K), np.uint32)
    eng.reset(1)
    for a in range(0, n, 8):
        b = min(a + 8, n)
        eng.prefill(1, prompt[a:b])
        h[a:b] = bf(eng.read("act.h", np.uint16, (b - a, H)))
        ids[a:b] = np.sort(eng.read("act.ids", np.uint32, (b - a, K)), axis=1)
    return h, ids


@pytest.mark.parametrize("n", [17, 77, 200, 301, 512])
def test_chunk_layer_matches_blocks(engine, gemm_plan, n):
    eng, cfg = engine
    # both sides of a layer that split k over workgroups: the low-rank
    # projection always, the output projection where it is deep and has rows
    bits, H = cfg["bits"], cfg["hidden"]
    assert gemm_plan(n, 260, 4 * H, bits, False, 4 << 20) in ("T2.16", "T3.16")
    deep = cfg["heads"] * cfg["head_dim"] if cfg["attn_every"] == 1 else 128 * cfg["gdn_hv"]
    out = gemm_plan(n, H, deep, bits, True, 4 << 20)
    assert (out[0] == "T" and out[-2:] != ".1") == (deep == 4096 and n > 17)
    prompt = np.random.default_rng(n).integers(0, cfg["vocab"], n)
    want, wids = blocks(eng, cfg, prompt)
    eng.reset(0)
    eng.prefill(0, prompt, chunked=True)
    got = bf(eng.read("act.h", np.uint16, want.shape)).astype(np.float64)
    ids = np.sort(eng.read("act.ids", np.uint32, wids.shape), axis=1)
    # a near tie in the router may go either way: those rows took other experts
    same = (ids == wids).all(axis=1)
    assert same.mean() >= 0.8
    # sixteen columns of a row at a time.  Sums in another order and the bf16
    # roundings between a layer's kernels, through the router and the experts:
    # up to 0.29 of the row's root mean square measured (0.17 below 6 bits); a
    # value from a wrong place, or left out, differs by about one
    d, w = (got - want)[same], want[same]
    rms = np.sqrt((w * w).mean(axis=1, keepdims=True))
    err = np.sqrt((d * d).reshape(len(d), -1, 16).mean(axis=2)) / rms
    print(f"{n} rows, {int((~same).sum())} routed differently: {err.max():.3f}", flush=True)
    assert err.max() <= 0.5
