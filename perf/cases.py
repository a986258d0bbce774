"""Performance cases: what a user of the library has it do, through its public entry points.

`listed()` names the cases, `draw()` gives more of the same ranges, `prepare()` makes a
case's inputs from a seed, `run()` is one pass, `work()` the bytes and operations that a pass
cannot do without, `tolerance()` how far another correct implementation may be off, and
`exact()` the result in 64 bits, in plain torch, where that is practical.

The geometry is the library's benchmark model (CONFIG3): hidden 2048, 512 experts top-10 with
512-wide MLPs (4-bit, 5-bit down), 16 key / 32 value GatedDeltaNet heads of 128, 16 query and
2 key/value heads of 256, vocabulary 151936, four hyper-connection streams.

Kinds of case:
  decode    `steps` greedy steps of the whole engine in exact mode, for `rows` requests that
            start from a cached prefix (cloned slots), each step's tokens fed to the next
  proj      one quantised projection: exact-integer (mx_xq) or matrix-core (mx_qmm)
  moe       the MoE sublayer after its router projection: routing, experts, slot sum and
            hyper-connection write, on the matrix cores
  scan      the chunked GatedDeltaNet prefill scan
  gdn       a GatedDeltaNet step: causal conv and recurrence with its gated norm
  attn      gated attention of decode rows over their own contexts, or of a prompt chunk
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    """The package (its folder's name has a hyphen)."""
    if "rust_mlx_amd" not in sys.modules:
        path = os.path.join(_ROOT, "rust-mlx_amd", "__init__.py")
        spec = importlib.util.spec_from_file_location("rust_mlx_amd", path)
        mod = importlib.util.module_from_spec(spec)
        sys.modules["rust_mlx_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["rust_mlx_amd"]


mx = _package()
BF16 = torch.bfloat16
GROUP = 64
HIDDEN, EXPERTS, TOP_K, INTER, STREAMS = 2048, 512, 10, 512, 4
HEADS, KV_HEADS, HEAD_DIM, MAX_CTX = 16, 2, 256, 4096
GDN_DIM, CONV_K = 128, 4


# ---- the cases ----------------------------------------------------------------------------
def listed():
    return [
        # continuous batching at full batch: eight users of the 48-layer model, 1000 tokens in
        {"name": "decode_8_users", "kind": "decode", "layers": 48, "rows": 8, "context": 1000, "steps": 4},
        # one interactive user with a long context: launches and latency count
        {"name": "decode_1_user", "kind": "decode", "layers": 48, "rows": 1, "context": 3001, "steps": 4},
        # the smallest call: one row through one 4-bit projection
        {"name": "proj_1_row", "kind": "proj", "exact": True, "rows": 1, "n": 4096, "k": 2048, "bits": 4},
        # the vocabulary head's logits for a full batch: the largest exact projection, 8-bit
        {"name": "head_8_rows", "kind": "proj", "exact": True, "rows": 8, "n": 151936, "k": 2048, "bits": 8},
        # the GatedDeltaNet input projection of a whole prompt chunk
        {"name": "proj_512_rows", "kind": "proj", "exact": False, "rows": 512, "n": 12352, "k": 2048, "bits": 4},
        # the GatedDeltaNet output projection of a prompt's short last chunk: few rows, few columns
        {"name": "proj_77_rows", "kind": "proj", "exact": False, "rows": 77, "n": 2048, "k": 4096, "bits": 4},
        # the MoE sublayer of a full decode batch
        {"name": "moe_8_rows", "kind": "moe", "rows": 8, "bits": 4, "down_bits": 5},
        # the MoE sublayer of a prompt's last, shorter chunk
        {"name": "moe_301_rows", "kind": "moe", "rows": 301, "bits": 4, "down_bits": 5},
        # a 2048-token prompt through one GatedDeltaNet layer's scan
        {"name": "scan_2048", "kind": "scan", "groups": 1, "tokens": 2048, "hk": 16, "hv": 32},
        # one GatedDeltaNet decode step of a full batch, in exact mode
        {"name": "gdn_8_rows", "kind": "gdn", "exact": True, "groups": 8, "tokens": 1},
        # attention of a full decode batch whose longest context is 4000 tokens, in exact mode
        {"name": "attn_8_rows", "kind": "attn", "form": "exact", "rows": 8, "context": 4000},
        # attention of a prompt chunk (not a whole number of query blocks) 1500 tokens in
        {"name": "attn_chunk", "kind": "attn", "form": "chunk", "rows": 509, "context": 1500},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "proj", "proj", "moe", "scan", "gdn", "attn"])
    if kind == "decode":
        return {"kind": kind, "layers": 4 * rng.randint(1, 12), "rows": rng.randint(1, 8),
                "context": _log(rng, 16, 4000), "steps": rng.randint(1, 4)}
    if kind == "proj":
        exact = rng.random() < 0.4
        n = _log(rng, 64, 20000)
        if exact:  # the depths the exact kernels take
            k, rows = rng.choice([256, 512, 1024, 2048, 4096, 8192]), rng.randint(1, 8)
        else:
            k, rows = GROUP * _log(rng, 4, 128), _log(rng, 1, 512)
        return {"kind": kind, "exact": exact, "rows": rows, "n": n, "k": k, "bits": rng.choice([4, 4, 5, 6, 8])}
    if kind == "moe":
        bits = rng.choice([4, 4, 4, 5, 6, 8])
        return {"kind": kind, "rows": _log(rng, 1, 512), "bits": bits, "down_bits": rng.choice([4, 5, 5, 6, 8])}
    if kind == "scan":
        hk = rng.choice([4, 8, 16])
        return {"kind": kind, "groups": rng.randint(1, 2), "tokens": _log(rng, 16, 1500), "hk": hk, "hv": 2 * hk}
    if kind == "gdn":
        groups = rng.randint(1, 8)
        return {"kind": kind, "exact": rng.random() < 0.5, "groups": groups, "tokens": 1 if groups > 1 else rng.randint(1, 8)}
    form = rng.choice(["exact", "fast", "chunk"])
    rows = _log(rng, 9, 512) if form == "chunk" else rng.randint(1, 8)
    return {"kind": kind, "form": form, "rows": rows, "context": _log(rng, 16, 3500)}


# ---- inputs -------------------------------------------------------------------------------
def _gen(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFFFFFF)
    return g


def _normal(g, shape, scale=1.0, dtype=BF16):
    return (torch.randn(shape, generator=g, device="cuda") * scale).to(dtype)


def _uniform(g, shape, lo, hi, dtype=torch.float32):
    return (torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo).to(dtype)


def _quantised(g, n, k, bits, experts=None):
    """Random affine-quantised weights of about unit gain: uniform codes, biases near -s (2^bits - 1) / 2."""
    lead = (n,) if experts is None else (experts, n)
    codes = torch.randint(-(1 << 31), 1 << 31, lead + (k * bits // 32,), generator=g, device="cuda",
                          dtype=torch.int64).to(torch.int32)
    step = math.sqrt(12.0) / (1 << bits) / math.sqrt(k)
    scales = _uniform(g, lead + (k // GROUP,), 0.6 * step, 1.4 * step, BF16)
    biases = (scales.float() * (-((1 << bits) - 1) / 2) + _normal(g, scales.shape, 0.1 * step, torch.float32)).to(BF16)
    return {"codes": codes, "scales": scales, "biases": biases, "n": n, "k": k, "bits": bits, "experts": experts}


def _c(w):
    """The C descriptor of a weight matrix or bank."""
    p = [w[x].data_ptr() for x in ("codes", "scales", "biases")]
    if w["experts"] is None:
        return mx.QWeightC(*p, w["n"], w["k"], w["bits"], GROUP)
    return mx.QBankC(*p, w["experts"], w["n"], w["k"], w["bits"], GROUP)


def _empty(shape, dtype=BF16):
    return torch.empty(shape, dtype=dtype, device="cuda")


def _bytes(n):
    return torch.empty(int(n), dtype=torch.uint8, device="cuda")


def _stream():
    return torch.cuda.current_stream().cuda_stream


def prepare(case, seed):
    return {"decode": _prepare_decode, "proj": _prepare_proj, "moe": _prepare_moe,
            "scan": _prepare_scan, "gdn": _prepare_gdn, "attn": _prepare_attn}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


# ---- the engine -----------------------------------------------------------------------------
def _tokens(g, n):
    return torch.randint(0, mx.CONFIG3["vocab"], (n,), generator=g, device="cuda").cpu().numpy().astype(np.uint32)


def _prepare_decode(case, seed):
    rows = case["rows"]
    e = mx.Engine(dict(mx.CONFIG3, layers=case["layers"], max_slots=2 * rows, max_context=MAX_CTX, seed=20250 + seed % 100003))
    e.set_flags(exact=True)
    for r in range(rows):  # the cached prefixes, in slots rows .. 2 rows - 1
        e.fill_slot(rows + r, case["context"], seed=1 + seed + 1000 * r)
    v = mx.CONFIG3["vocab"]
    return {"run": _run_decode, "engine": e, "rows": rows, "steps": case["steps"], "tokens": _tokens(_gen(seed), rows),
            "slots": np.arange(rows, dtype=np.int32), "logits": _empty((rows, v)),
            "hidden": _empty((rows, STREAMS * HIDDEN))}


def _step(e, slots, tokens, logits, hidden):
    out = np.empty(len(slots), np.uint32)
    mx.check(mx.lib.mx_engine_decode_batch_outputs(e.h, slots.ctypes.data, tokens.ctypes.data, len(slots), out.ctypes.data,
                                                   logits.data_ptr(), hidden.data_ptr()))
    return out


def _run_decode(s):
    e, rows, tok = s["engine"], s["rows"], s["tokens"]
    for r in range(rows):  # each request starts from its cached prefix
        e.clone(rows + r, r)
    ids = []
    for _ in range(s["steps"]):
        tok = _step(e, s["slots"], tok, s["logits"], s["hidden"])
        ids.append(tok)
    return {"tokens": np.stack(ids).astype(np.int64), "logits": s["logits"], "hidden": s["hidden"]}


# ---- projections ----------------------------------------------------------------------------
def _prepare_proj(case, seed):
    g = _gen(seed, 1)
    w = _quantised(g, case["n"], case["k"], case["bits"])
    return {"run": _run_proj, "w": w, "c": _c(w), "x": _normal(g, (case["rows"], case["k"])), "rows": case["rows"],
            "y": _empty((case["rows"], case["n"])), "call": mx.lib.mx_xq if case["exact"] else mx.lib.mx_qmm}


def _run_proj(s):
    mx.check(s["call"](ctypes.byref(s["c"]), s["x"].data_ptr(), s["rows"], s["y"].data_ptr(), _stream()))
    return s["y"]


# ---- the MoE sublayer -------------------------------------------------------------------------
def _prepare_moe(case, seed):
    g, rows, b, d = _gen(seed, 2), case["rows"], case["bits"], case["down_bits"]
    w = {"gate": _quantised(g, INTER, HIDDEN, b, EXPERTS), "up": _quantised(g, INTER, HIDDEN, b, EXPERTS),
         "down": _quantised(g, HIDDEN, INTER, d, EXPERTS), "sgate": _quantised(g, INTER, HIDDEN, b),
         "sup": _quantised(g, INTER, HIDDEN, b), "sdown": _quantised(g, HIDDEN, INTER, d)}
    return {"run": _run_moe, "rows": rows, "w": w, "c": {n: _c(v) for n, v in w.items()},
            "x": _normal(g, (rows, HIDDEN)), "logits": _normal(g, (rows, EXPERTS + 1), 1.5),
            "streams": _normal(g, (rows, STREAMS, HIDDEN), 2.0), "gate": _uniform(g, (rows, STREAMS), 0.0, 2.0, BF16),
            "ids": _empty((rows, TOP_K), torch.int32), "scores": _empty((rows, TOP_K)), "factor": _empty((rows,)),
            "partial": _empty((rows, TOP_K + 1, HIDDEN)),
            "ws": _bytes(mx.lib.mx_moe_workspace_bytes(rows, TOP_K, INTER))}


def _run_moe(s):
    ref = ctypes.byref
    rows, st, c = s["rows"], _stream(), s["c"]
    lg, xp, ws = s["logits"].data_ptr(), s["x"].data_ptr(), s["ws"].data_ptr()
    ids, scores, factor = s["ids"].data_ptr(), s["scores"].data_ptr(), s["factor"].data_ptr()
    banks = [ref(c[n]) for n in ("gate", "up", "down", "sgate", "sup", "sdown")]
    if rows <= 8:  # a decode batch: the whole sublayer in one call, the streams written in place
        mx.check(mx.lib.mx_moe_routed_experts_hc_mfma(
            lg, EXPERTS + 1, lg + 2 * EXPERTS, EXPERTS + 1, EXPERTS, xp, rows, TOP_K, STREAMS, *banks, ws, ids, scores,
            factor, s["gate"].data_ptr(), s["streams"].data_ptr(), st))
    else:  # a prompt chunk: routing, experts, then the slot sum and stream write
        part, h = s["partial"].data_ptr(), s["streams"].data_ptr()
        mx.check(mx.lib.mx_moe_route(lg, EXPERTS + 1, lg + 2 * EXPERTS, EXPERTS + 1, rows, EXPERTS, TOP_K, ids, scores,
                                     factor, st))
        mx.check(mx.lib.mx_moe_experts_mfma(xp, ids, scores, rows, TOP_K, *banks, ws, part, st))
        mx.check(mx.lib.mx_moe_reduce_hc_epilogue(part, factor, h, s["gate"].data_ptr(), rows, TOP_K, STREAMS, HIDDEN, h,
                                                  st))
    return {"ids": s["ids"], "scores": s["scores"], "factor": s["factor"], "streams": s["streams"]}


# ---- GatedDeltaNet ------------------------------------------------------------------------------
def _unit(g, shape):
    v = torch.randn(shape, generator=g, device="cuda")
    return (v / v.norm(dim=-1, keepdim=True)).to(BF16)


def _prepare_scan(case, seed):
    g, hk, hv, t, groups = _gen(seed, 3), case["hk"], case["hv"], case["tokens"], case["groups"]
    rows = t * groups
    rate = _uniform(g, (hv,), 0.0, 16.0)
    decay = torch.exp(-torch.nn.functional.softplus(torch.randn((rows, hv), generator=g, device="cuda")) * rate)
    return {"run": _run_scan, "dims": mx.GdnDimsC(hk, hv, GDN_DIM, GDN_DIM, CONV_K), "groups": groups, "t": t,
            "q": _unit(g, (rows, hk, GDN_DIM)), "k": _unit(g, (rows, hk, GDN_DIM)),
            "v": _normal(g, (rows, hv, GDN_DIM)), "g": decay.contiguous(),
            "beta": torch.sigmoid(torch.randn((rows, hv), generator=g, device="cuda")).to(BF16),
            "slots": torch.arange(groups, device="cuda", dtype=torch.int32),
            "state": _normal(g, (groups, hv, GDN_DIM, GDN_DIM), 0.1, torch.float32),
            "y": _empty((rows, hv, GDN_DIM)), "ws": _bytes(mx.lib.mx_gdn_prefill_workspace_bytes(groups, hv, t))}


def _run_scan(s):
    p = {n: s[n].data_ptr() for n in ("q", "k", "v", "g", "beta", "slots", "state", "y", "ws")}
    mx.check(mx.lib.mx_gdn_prefill_chunked(p["q"], p["k"], p["v"], p["g"], p["beta"], ctypes.byref(s["dims"]), s["groups"],
                                           s["t"], p["slots"], p["state"], p["y"], p["ws"], _stream()))
    return {"y": s["y"], "state": s["state"]}


HK, HV = 16, 32
CHANNELS = (2 * HK + HV) * GDN_DIM


def _prepare_gdn(case, seed):
    g, groups, t = _gen(seed, 4), case["groups"], case["tokens"]
    rows = groups * t
    slots = torch.randperm(9, generator=g, device="cuda")[:groups].to(torch.int32)
    return {"run": _run_gdn, "exact": case["exact"], "groups": groups, "t": t,
            "dims": mx.GdnDimsC(HK, HV, GDN_DIM, GDN_DIM, CONV_K),
            # the input projection's rows: qkv | z | a | b
            "proj": _normal(g, (rows, CHANNELS + HV * GDN_DIM + 2 * HV)),
            "conv_w": _uniform(g, (CONV_K, CHANNELS), -0.6, 0.6), "window": _normal(g, (9, CONV_K - 1, CHANNELS)),
            "a_log": torch.log(_uniform(g, (HV,), 0.01, 16.0)), "dt": _uniform(g, (HV,), -1.0, 1.0, BF16),
            "norm": _uniform(g, (GDN_DIM,), 0.5, 1.5, BF16), "slots": slots,
            "state": _normal(g, (9, HV, GDN_DIM, GDN_DIM), 0.05, torch.float32),
            "conv": _empty((rows, CHANNELS)), "y": _empty((rows, HV * GDN_DIM))}


def _run_gdn(s):
    st, p = _stream(), s["proj"].data_ptr()
    width = s["proj"].shape[1]
    zp = p + 2 * CHANNELS
    ap = zp + 2 * HV * GDN_DIM
    mx.check(mx.lib.mx_gdn_conv(p, width, s["groups"], s["t"], s["slots"].data_ptr(), s["window"].data_ptr(),
                                s["conv_w"].data_ptr(), CHANNELS, CONV_K, s["conv"].data_ptr(), CHANNELS, None, st))
    call = mx.lib.mx_gdn_recurrence if s["exact"] else mx.lib.mx_gdn_recurrence_fast
    mx.check(call(s["conv"].data_ptr(), CHANNELS, zp, ap, ap + 2 * HV, width, s["a_log"].data_ptr(), s["dt"].data_ptr(),
                  s["norm"].data_ptr(), 1e-6, ctypes.byref(s["dims"]), s["groups"], s["t"], s["slots"].data_ptr(),
                  s["state"].data_ptr(), None, s["y"].data_ptr(), st))
    return {"y": s["y"], "state": s["state"], "window": s["window"]}


# ---- attention ------------------------------------------------------------------------------------
def _prepare_attn(case, seed):
    g, rows, ctx = _gen(seed, 5), case["rows"], case["context"]
    if case["form"] == "chunk":  # a chunk of one slot's prompt at positions ctx ..
        nslots = 1
        pos = torch.arange(ctx, ctx + rows, device="cuda", dtype=torch.int32)
        slots = torch.zeros(rows, device="cuda", dtype=torch.int32)
    else:  # requests at their own offsets, the longest at ctx
        nslots = 8
        pos = (torch.rand(rows, generator=g, device="cuda") * ctx).to(torch.int32)
        pos[0] = ctx - 1
        slots = torch.randperm(8, generator=g, device="cuda")[:rows].to(torch.int32)
    shape = (nslots, KV_HEADS, MAX_CTX, HEAD_DIM)
    return {"run": _run_attn, "rows": rows, "flags": {"exact": 0, "fast": 1, "chunk": 3}[case["form"]],
            "dims": mx.AttnDimsC(HEADS, KV_HEADS, HEAD_DIM, MAX_CTX, KV_HEADS * MAX_CTX * HEAD_DIM),
            "q": _normal(g, (rows, HEADS, HEAD_DIM)), "qkv": _normal(g, (rows, (2 * HEADS + 2 * KV_HEADS) * HEAD_DIM)),
            "slots": slots, "pos": pos, "k": _normal(g, shape), "v": _normal(g, shape),
            "out": _empty((rows, HEADS, HEAD_DIM)),
            "ws": _bytes(mx.lib.mx_attn_workspace_bytes(rows, HEADS, HEAD_DIM, MAX_CTX))}


def _run_attn(s):
    p = {n: s[n].data_ptr() for n in ("q", "qkv", "slots", "pos", "k", "v", "ws", "out")}
    mx.check(mx.lib.mx_attn_decode(p["q"], p["qkv"], s["qkv"].shape[1], s["rows"], p["slots"], p["pos"], p["k"], p["v"],
                                   ctypes.byref(s["dims"]), s["flags"], p["ws"], p["out"], _stream()))
    return s["out"]


# ---- what a pass cannot do without ------------------------------------------------------------------
def _q(n, k, bits):
    return n * k * bits / 8 + 4 * n * k / GROUP


def _distinct(rows):
    """Expected number of experts that `rows` rows name."""
    return EXPERTS * (1 - (1 - TOP_K / EXPERTS) ** rows)


def _moe_work(rows, bits, down_bits):
    expert = 2 * _q(INTER, HIDDEN, bits) + _q(HIDDEN, INTER, down_bits)
    return (_distinct(rows) + 1) * expert, 2.0 * rows * (TOP_K + 1) * 3 * INTER * HIDDEN


def _model_work(layers, rows, positions, new):
    """One pass over `layers` layers with `rows` tokens: every weight that is used once, the caches read and written."""
    c = mx.CONFIG3
    rank, vd = c["hc_rank"], HV * GDN_DIM
    hc = 2 * (_q(rank + STREAMS, STREAMS * HIDDEN, 4) + _q(STREAMS * HIDDEN, rank, 4))
    gdn = _q(CHANNELS + vd + 2 * HV, HIDDEN, 4) + _q(HIDDEN, vd, 4)
    att = _q((2 * HEADS + 2 * KV_HEADS) * HEAD_DIM, HIDDEN, 4) + _q(HIDDEN, HEADS * HEAD_DIM, 4)
    eb, ef = _moe_work(rows, 4, 5)
    n_att = layers // 4
    b = layers * (hc + _q(EXPERTS + 1, HIDDEN, 4) + eb) + (layers - n_att) * gdn + n_att * att
    f = layers * ef + 2.0 * rows * (layers * (2 * (2 * rank + STREAMS) * STREAMS * HIDDEN + (EXPERTS + 1) * HIDDEN)
                                    + (layers - n_att) * HIDDEN * (CHANNELS + 2 * vd + 2 * HV)
                                    + n_att * HIDDEN * (3 * HEADS + 2 * KV_HEADS) * HEAD_DIM)
    state = (layers - n_att) * new * (2 * HV * GDN_DIM * GDN_DIM * 4 + 4 * (CONV_K - 1) * CHANNELS)
    kv = n_att * positions * KV_HEADS * HEAD_DIM * 4
    f += (layers - n_att) * rows * HV * GDN_DIM * GDN_DIM * 6.0
    return b + state + kv, f


def work(case):
    kind, rows = case["kind"], case.get("rows", 0)
    head = _q(mx.CONFIG3["vocab"], HIDDEN, 8)
    if kind == "decode":
        b, f = _model_work(case["layers"], rows, rows * (case["context"] + 1), rows)
        f += rows * case["layers"] // 4 * 4.0 * (case["context"] + 1) * HEADS * HEAD_DIM
        return {"bytes": case["steps"] * (b + head), "flops": case["steps"] * (f + 2.0 * rows * mx.CONFIG3["vocab"] * HIDDEN)}
    if kind == "proj":
        return {"bytes": _q(case["n"], case["k"], case["bits"]) + 2 * rows * (case["n"] + case["k"]),
                "flops": 2.0 * rows * case["n"] * case["k"]}
    if kind == "moe":
        b, f = _moe_work(rows, case["bits"], case["down_bits"])
        return {"bytes": b + rows * 2 * (HIDDEN + EXPERTS + 2 * STREAMS * HIDDEN), "flops": f}
    if kind == "scan":
        n = case["groups"] * case["tokens"]
        return {"bytes": n * 2 * GDN_DIM * (2 * case["hk"] + 2 * case["hv"]) + 6 * n * case["hv"]
                + 8 * case["groups"] * case["hv"] * GDN_DIM ** 2, "flops": 6.0 * n * case["hv"] * GDN_DIM ** 2}
    if kind == "gdn":
        n = case["groups"] * case["tokens"]
        return {"bytes": case["groups"] * (8 * HV * GDN_DIM ** 2 + 4 * (CONV_K - 1) * CHANNELS)
                + n * 2 * (CHANNELS + 2 * HV * GDN_DIM) + 4 * CONV_K * CHANNELS, "flops": 6.0 * n * HV * GDN_DIM ** 2}
    if case["form"] == "chunk":
        keys = sum(case["context"] + r + 1 for r in range(rows))
        read = case["context"] + rows
    else:
        keys = read = case["context"] * (rows + 1) / 2
    return {"bytes": read * KV_HEADS * HEAD_DIM * 4 + rows * HEADS * HEAD_DIM * 6, "flops": 4.0 * keys * HEADS * HEAD_DIM}


def tolerance(case):
    kind = case["kind"]
    if kind == "decode" or case.get("exact") or case.get("form") == "exact":
        return "exact"  # the exact mode's arithmetic has one fixed order
    if kind == "proj":  # equal sums but for their order: now and then another bf16 value
        return {"rel": 2e-3, "max": 0.01}
    if kind == "moe":
        return {"rel": 7e-3, "max": 0.05, "differ": 0.0}
    if kind in ("scan", "gdn"):
        return {"rel": 3e-3, "max": 0.02}
    return {"rel": 1e-2, "max": 0.06}


# ---- the results in 64 bits -------------------------------------------------------------------------
def _dequant(codes, scales, biases, bits):
    """float64 weights [n, k] of one matrix (value v of a row at bit v * bits of its little-endian words)."""
    n, words = codes.shape
    k = words * 32 // bits
    w = codes.to(torch.int64) & 0xFFFFFFFF
    w = torch.cat([w, w.new_zeros(n, 1)], 1)
    bit = torch.arange(k, device=codes.device) * bits
    lo, sh = bit >> 5, bit & 31
    q = ((w[:, lo] | (w[:, lo + 1] << 32)) >> sh) & ((1 << bits) - 1)
    return q.double() * scales.double().repeat_interleave(GROUP, 1) + biases.double().repeat_interleave(GROUP, 1)


def _matrix(w, expert=None):
    pick = (lambda t: t) if expert is None else (lambda t: t[expert])
    return _dequant(pick(w["codes"]), pick(w["scales"]), pick(w["biases"]), w["bits"])


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        return None
    s = prepare(case, seed)
    return {"proj": _exact_proj, "moe": _exact_moe, "scan": _exact_scan, "gdn": _exact_gdn, "attn": _exact_attn}[kind](s)


def _exact_proj(s):
    w, x = s["w"], s["x"].double()
    out = [x @ _dequant(w["codes"][a:a + 4096], w["scales"][a:a + 4096], w["biases"][a:a + 4096], w["bits"]).T
           for a in range(0, w["n"], 4096)]
    return torch.cat(out, 1)


def _exact_moe(s):
    w, x, rows = s["w"], s["x"].double(), s["rows"]
    logits = s["logits"].double()
    # the contract ranks bf16 gates, the larger expert id first among equals, ascending by key
    gates = torch.softmax(logits[:, :EXPERTS], 1).to(BF16).double()
    order = torch.argsort(gates, dim=1, stable=True)[:, -TOP_K:]
    picked = gates.gather(1, order)
    scores = picked / picked.sum(1, keepdim=True)
    factor = torch.sigmoid(logits[:, EXPERTS])

    def mlp(xi, e, shared=False):
        gw, uw, dw = (_matrix(w["s" + n]) if shared else _matrix(w[n], e) for n in ("gate", "up", "down"))
        return (torch.nn.functional.silu(xi @ gw.T) * (xi @ uw.T)) @ dw.T

    y = mlp(x, None, True) * factor[:, None]
    for e in torch.unique(order).tolist():
        r, j = torch.nonzero(order == e, as_tuple=True)
        y.index_add_(0, r, mlp(x[r], e) * scores[r, j][:, None])
    streams = s["streams"].double() + y[:, None, :] * s["gate"].double()[:, :, None]
    return {"ids": None, "scores": scores, "factor": factor, "streams": streams}


def _delta_rule(state, q, k, v, g, beta):
    """One token of the delta rule for [groups, heads]: state [.., dk, dv] -> (new state, output [.., dv])."""
    state = state * g[..., None, None]
    delta = (v - torch.einsum("ghk,ghkv->ghv", k, state)) * beta[..., None]
    state = state + k[..., :, None] * delta[..., None, :]
    return state, torch.einsum("ghk,ghkv->ghv", q, state)


def _exact_scan(s):
    groups, t, hv = s["groups"], s["t"], s["v"].shape[1]
    rep = hv // s["q"].shape[1]

    def rows(x):
        return x.double().reshape((groups, t) + tuple(x.shape[1:]))

    q, k = (rows(s[n]).repeat_interleave(rep, 2) for n in ("q", "k"))
    v, g, beta = (rows(s[n]) for n in ("v", "g", "beta"))
    state, out = s["state"].double(), []
    for i in range(t):
        state, y = _delta_rule(state, q[:, i], k[:, i], v[:, i], g[:, i], beta[:, i])
        out.append(y)
    return {"y": torch.stack(out, 1).reshape(groups * t, hv, GDN_DIM), "state": state}


def _exact_gdn(s):
    groups, t, slots = s["groups"], s["t"], s["slots"].long()
    p = s["proj"].double().reshape(groups, t, -1)
    window = s["window"].double()
    run_ = torch.cat([window[slots], p[..., :CHANNELS]], 1)
    cw = s["conv_w"].double()
    conv = sum(run_[:, j:j + t] * cw[j] for j in range(CONV_K))
    conv = torch.nn.functional.silu(conv)
    window[slots] = run_[:, t:]
    kd = HK * GDN_DIM

    def heads(x, n):
        return x.reshape(groups, t, n, GDN_DIM)

    def unit(x):
        return x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)

    q = unit(heads(conv[..., :kd], HK)).repeat_interleave(HV // HK, 2) * GDN_DIM ** -0.5
    k = unit(heads(conv[..., kd:2 * kd], HK)).repeat_interleave(HV // HK, 2)
    v = heads(conv[..., 2 * kd:], HV)
    z = heads(p[..., CHANNELS:CHANNELS + HV * GDN_DIM], HV)
    a, b = p[..., -2 * HV:-HV], p[..., -HV:]
    g = torch.exp(-torch.exp(s["a_log"].double()) * torch.nn.functional.softplus(a + s["dt"].double()))
    state, out = s["state"].double(), []
    cur = state[slots]
    for i in range(t):
        cur, y = _delta_rule(cur, q[:, i], k[:, i], v[:, i], g[:, i], torch.sigmoid(b[:, i]))
        y = y * torch.rsqrt((y * y).mean(-1, keepdim=True) + 1e-6) * s["norm"].double()
        out.append(y * torch.sigmoid(z[:, i]))
    state[slots] = cur
    return {"y": torch.stack(out, 1).reshape(groups * t, HV * GDN_DIM), "state": state, "window": window}


def _exact_attn(s):
    per, out = HEADS // KV_HEADS, []
    gate = s["qkv"].double()[:, :2 * HEADS * HEAD_DIM].reshape(-1, HEADS, 2, HEAD_DIM)[:, :, 1]
    k, v = (s[n].double() for n in ("k", "v"))
    slots, pos = s["slots"].tolist(), s["pos"].tolist()
    for r in range(s["rows"]):
        n = pos[r] + 1
        q = s["q"][r].double().reshape(KV_HEADS, per, HEAD_DIM)
        p = torch.softmax(q @ k[slots[r], :, :n].transpose(1, 2) / math.sqrt(HEAD_DIM), 2)
        out.append((p @ v[slots[r], :, :n]).reshape(HEADS, HEAD_DIM))
    return torch.stack(out) * torch.sigmoid(gate)
