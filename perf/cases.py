"""The attention library's work as its users call it, case by case: decode steps,
prefill chunks and the projections behind them, through the Python mirror of the
C ABI.  A case is a dict of plain values; `prepare` makes what a caller holds
before the call, `run` is one pass, `exact` the same result in 64 bits.

Kinds (the "kind" of a case):
  decode   attention of one token over `layers` caches of `seq` positions: one
           eager call (layers 0) or the captured graph of n layers
  step     `steps` replays of the captured decode step (norm + RoPE + cache
           append, attention, and with `wo` the output projection) from
           position `ctx` on
  layer    one layer of a prefill chunk through the chunk driver (norm + RoPE,
           cache append, int8 K copy, attention, Q8_1) and its output projection
  attn     the prefill attention alone, int8 or fp16 scores, into fp32 rows
  linear   fp32 rows quantised to Q8_1, then a Q4_0 matrix product
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "lfm2-ampere_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import lk_attn as lk  # noqa: E402

H, KV, D = 32, 8, 64
HID, KROW = H * D, KV * D
LOG2E = 1.4426950408889634

_decode_stream = None


def listed():
    return [
        # a single attention call of a short chat, issued eagerly: launch latency
        {"name": "decode_389", "kind": "decode", "seq": 389, "layers": 0},
        # the attention of a whole step as the engine captures it, at a long and
        # at the longest context it is configured for
        {"name": "decode_32k_x10", "kind": "decode", "seq": 32768, "layers": 10},
        {"name": "decode_131k_x10", "kind": "decode", "seq": 131072, "layers": 10},
        # tokens generated in a chat of ordinary length, output projection included
        {"name": "step_2500_x10", "kind": "step", "ctx": 2500, "layers": 10, "steps": 4, "wo": True},
        # a short prompt, the default-size first chunk, a chat turn deep in a
        # conversation (with rows that decode has appended since), and the first
        # chunk of a context with smoothed keys
        {"name": "layer_m201", "kind": "layer", "m": 201, "P": 0, "int8": True, "smooth": False, "stale": 0,
         "near": 1024, "sink": 1},
        {"name": "layer_m4096", "kind": "layer", "m": 4096, "P": 0, "int8": True, "smooth": False, "stale": 0,
         "near": 1024, "sink": 1},
        {"name": "layer_m77_at_30011", "kind": "layer", "m": 77, "P": 30011, "int8": True, "smooth": False,
         "stale": 190, "near": 1024, "sink": 1},
        {"name": "layer_m2999_smooth", "kind": "layer", "m": 2999, "P": 0, "int8": True, "smooth": True, "stale": 0,
         "near": 1024, "sink": 1},
        # the last chunk of a 131072-token prompt
        {"name": "attn8_m4096_at_126976", "kind": "attn", "m": 4096, "P": 126976, "int8": True, "near": 1024,
         "sink": 1},
        # the fp16 kernel on a ragged chunk in the middle of a prompt
        {"name": "attn16_m1100_at_3333", "kind": "attn", "m": 1100, "P": 3333, "int8": False, "near": 0, "sink": 0},
        # the projection of a short prompt's rows into the residual, and of a chunk's
        {"name": "linear_333", "kind": "linear", "ntok": 333, "n": 2048, "k": 2048, "add": True},
        {"name": "linear_4096", "kind": "linear", "ntok": 4096, "n": 2048, "k": 2048, "add": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _chunk(rng):
    """(m, P) over all chunk lengths and depths that cost no more than the
    last 4096-row chunk of a 131072-token prompt."""
    while True:
        m = _log(rng, 1, 8192)
        P = 0 if rng.random() < 0.4 else _log(rng, 16, 126976)
        if m * (P + m / 2) <= 0.9 * 4096 * (126976 + 2048) and P + m <= 131072:
            return m, P


def draw(rng):
    kind = rng.choice(["decode", "step", "layer", "layer", "attn", "linear"])
    if kind == "decode":
        layers = rng.choice([0, 0, 4, 10])
        return {"kind": kind, "seq": _log(rng, 1, 131072), "layers": layers}
    if kind == "step":
        return {"kind": kind, "ctx": _log(rng, 1, 100000), "layers": rng.choice([2, 6, 10]),
                "steps": rng.choice([1, 3, 8]), "wo": rng.random() < 0.7}
    if kind == "layer":
        m, P = _chunk(rng)
        int8 = rng.random() < 0.8
        return {"kind": kind, "m": m, "P": P, "int8": int8, "smooth": int8 and P == 0 and rng.random() < 0.4,
                "stale": min(P, _log(rng, 1, 600)) if int8 and rng.random() < 0.5 else 0,
                "near": rng.choice([256, 1024, 1024, 2048]), "sink": rng.choice([0, 1, 1])}
    if kind == "attn":
        m, P = _chunk(rng)
        int8 = rng.random() < 0.6
        return {"kind": kind, "m": m, "P": P, "int8": int8, "near": rng.choice([256, 1024, 2048]) if int8 else 0,
                "sink": rng.choice([0, 1]) if int8 else 0}
    return {"kind": kind, "ntok": _log(rng, 1, 8192), "n": 128 * rng.choice([1, 3, 16, 24]),
            "k": 256 * rng.choice([1, 8, 8, 9, 16]), "add": rng.random() < 0.5}


# ---- inputs -----------------------------------------------------------------------
def _gen(seed, tag):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + tag) & 0x7FFFFFFFFFFF)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _rand(g, lo, hi, *shape):
    return lo + (hi - lo) * torch.rand(*shape, generator=g, device="cuda", dtype=torch.float32)


def _unit(x):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True))


def _cache(seed, tag, rows):
    """K and V rows as the model's own layers leave them in the cache: K of unit
    RMS per head times a per-channel gain, V about N(0, 1), both fp16."""
    g = _gen(seed, tag)
    k = _unit(_randn(g, rows, KV, D)) * _rand(g, 0.5, 2.0, KV, D)
    return k.half().contiguous(), _randn(g, rows, KV, D).half().contiguous()


def _weights(seed, tag, n, bpr):
    g = _gen(seed, tag)
    qs = torch.randint(0, 256, (n, bpr, 16), generator=g, device="cuda", dtype=torch.uint8)
    return qs, _rand(g, 0.002, 0.02, n, bpr).half()


def _norms(seed):
    g = _gen(seed, 900)
    return _rand(g, 0.5, 1.5, D), _rand(g, 0.5, 1.5, D)


def _stream():
    global _decode_stream
    if _decode_stream is None:
        _decode_stream = torch.cuda.Stream()
    return _decode_stream


def _decode_inputs(case, seed):
    n = max(1, case["layers"])
    qs = [_unit(_randn(_gen(seed, 10 + i), H, D)) for i in range(n)]
    kvs = [_cache(seed, 100 + i, case["seq"]) for i in range(n)]
    return qs, [k for k, _ in kvs], [v for _, v in kvs]


def _step_inputs(case, seed):
    rows = case["ctx"] + case["steps"]
    layers = []
    for i in range(case["layers"]):
        g = _gen(seed, 200 + i)
        kc, vc = _cache(seed, 300 + i, rows)
        L = {"q_src": 3 * _randn(g, H, D), "k_src": 3 * _randn(g, KV, D), "v_src": _randn(g, KV, D),
             "q_norm": _rand(g, 0.5, 1.5, D), "k_norm": _rand(g, 0.5, 1.5, D), "kc": kc, "vc": vc}
        if case["wo"]:
            L["wo_qs"], L["wo_d"] = _weights(seed, 400 + i, HID, HID // 32)
        layers.append(L)
    return layers, _randn(_gen(seed, 500), HID)


def _layer_inputs(case, seed):
    m, P = case["m"], case["P"]
    kc, vc = _cache(seed, 600, P + m)
    Y = _randn(_gen(seed, 601), m, HID + 2 * KROW) * 3
    return Y, kc, vc, _norms(seed), _weights(seed, 602, HID, HID // 32)


def _attn_inputs(case, seed):
    kc, vc = _cache(seed, 700, case["P"] + case["m"])
    qh = (_unit(_randn(_gen(seed, 701), case["m"], H, D)) * 1.5 * 0.125).half().reshape(case["m"], HID)
    return qh.contiguous(), kc, vc


def _linear_inputs(case, seed):
    g = _gen(seed, 800)
    X = _randn(g, case["ntok"], case["k"]) * _rand(g, 0.5, 2.0, case["k"])
    return X, _weights(seed, 801, case["n"], case["k"] // 32), _randn(g, case["ntok"], case["n"])


# ---- what a caller keeps, and one pass ---------------------------------------------
def prepare(case, seed):
    s = {"case": case}
    kind = case["kind"]
    if kind == "decode":
        qs, kcs, vcs = _decode_inputs(case, seed)
        s["pos"] = torch.tensor([case["seq"] - 1], dtype=torch.int32, device="cuda")
        s["part"] = torch.empty(lk.part_bytes() // 4, device="cuda")
        s["out"] = [torch.empty(H, D, device="cuda") for _ in qs]
        s["yq8"] = [torch.zeros(2 * H, lk.Q8_1_BYTES, dtype=torch.uint8, device="cuda") for _ in qs]
        s["in"] = (qs, kcs, vcs)
        if case["layers"]:
            torch.cuda.synchronize()
            s["graph"] = lk.DecodeGraph(qs, kcs, vcs, s["pos"], s["part"], s["out"], s["yq8"], stream=_stream())
    elif kind == "step":
        layers, x0 = _step_inputs(case, seed)
        s["x0"], s["x"] = x0, x0.clone()
        s["pos0"] = torch.tensor([case["ctx"]], dtype=torch.int32, device="cuda")
        s["pos"] = s["pos0"].clone()
        s["part"] = torch.empty(lk.part_bytes() // 4, device="cuda")
        for L in layers:
            L.update(q=torch.empty(H, D, device="cuda"), k=torch.empty(KV, D, device="cuda"),
                     out=torch.empty(H, D, device="cuda"),
                     yq8=torch.zeros(2 * H, lk.Q8_1_BYTES, dtype=torch.uint8, device="cuda"))
            if case["wo"]:
                L["x"] = s["x"]
        s["layers"] = layers
        torch.cuda.synchronize()
        s["graph"] = lk.DecodeStepGraph(layers, s["pos"], s["part"], stream=_stream())
    elif kind == "layer":
        m, P = case["m"], case["P"]
        Y, kc, vc, norms, w = _layer_inputs(case, seed)
        ctx = lk.PrefillCtx(1, m, P + m, attn8=case["int8"], ksmooth=case["smooth"], near=case["near"],
                            sink=case["sink"])
        s.update(Y=Y, kc=kc, vc=vc, norms=norms, w=w, ctx=ctx,
                 aqs=torch.empty(m, HID, dtype=torch.int8, device="cuda"),
                 asc=torch.empty(m, HID // 32, 2, device="cuda"), x=torch.empty(m, HID, device="cuda"))
        if P and case["int8"]:
            # the earlier chunks of the prompt: their int8 keys are in the context
            ctx.chunk_attn(0, Y, norms[0], norms[1], m, P, kc, vc, None, s["aqs"], s["asc"])
            ctx.chunk_done(P - case["stale"])
    elif kind == "attn":
        m, P = case["m"], case["P"]
        qh, kc, vc = _attn_inputs(case, seed)
        s.update(qh=qh, kc=kc, vc=vc, o=torch.empty(m, HID, device="cuda"),
                 work=torch.empty(lk.pf_part_bytes() // 4, device="cuda"))
        if case["int8"]:
            s["ks"] = lk.kstride_for(P + m)
            s["k8"] = torch.empty((P + m) * KROW, dtype=torch.int8, device="cuda")
            s["ksc"] = torch.empty(KV * s["ks"] + 4, device="cuda")
            lk.pf_k8(kc, 0, P + m, None, s["ks"], s["k8"], s["ksc"])
    else:
        X, w, res = _linear_inputs(case, seed)
        s.update(X=X, w=w, res=res, out=torch.empty_like(res),
                 qs=torch.empty(case["ntok"], case["k"], dtype=torch.int8, device="cuda"),
                 sc=torch.empty(case["ntok"], case["k"] // 32, 2, device="cuda"))
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        if case["layers"]:
            s["graph"].launch()
        else:
            qs, kcs, vcs = s["in"]
            lk.attn_decode(qs[0], kcs[0], vcs[0], s["pos"], s["part"], s["out"][0], s["yq8"][0])
        return {"out": s["out"], "yq8": s["yq8"]}
    if kind == "step":
        # a new request: its position and residual row, then its tokens
        with torch.cuda.stream(_stream()):
            s["pos"].copy_(s["pos0"])
            s["x"].copy_(s["x0"])
        s["graph"].run(case["steps"])
        new = slice(case["ctx"], case["ctx"] + case["steps"])
        return {"out": [L["out"] for L in s["layers"]], "k": [L["kc"][new] for L in s["layers"]],
                "v": [L["vc"][new] for L in s["layers"]], "x": s["x"] if case["wo"] else None}
    if kind == "layer":
        m, P = case["m"], case["P"]
        s["ctx"].chunk_attn(0, s["Y"], s["norms"][0], s["norms"][1], m, P, s["kc"], s["vc"], None, s["aqs"],
                            s["asc"])
        lk.pf_gemm_q4_0(s["w"][0], s["w"][1], HID, HID // 32, s["aqs"], s["asc"], m, s["x"])
        return {"aqs": s["aqs"], "asc": s["asc"], "x": s["x"], "k": s["kc"][P:], "v": s["vc"][P:]}
    if kind == "attn":
        if case["int8"]:
            lk.pf_attn8_ws(None, None, None, s["qh"], case["m"], case["P"], s["k8"], s["ksc"], s["ks"], s["kc"],
                           s["vc"], case["near"], case["sink"], s["o"], None, None, s["work"])
        else:
            lk.pf_attn_ws(s["qh"], case["m"], case["P"], s["kc"], s["vc"], s["o"], None, None, s["work"])
        return {"o": s["o"]}
    n, k, t = case["n"], case["k"], case["ntok"]
    if case["add"]:
        s["out"].copy_(s["res"])                    # the residual rows that the product is added to
    lk.pf_quant_rows(s["X"], t, k, k // 32, s["qs"], s["sc"])
    lk.pf_gemm_q4_0(s["w"][0], s["w"][1], n, k // 32, s["qs"], s["sc"], t, s["out"], n, case["add"])
    return {"qs": s["qs"], "sc": s["sc"], "out": s["out"]}


# ---- what a pass cannot do without ---------------------------------------------------
_W_BYTES = HID * HID // 32 * 18


def work(case):
    kind = case["kind"]
    if kind == "decode":
        n = max(1, case["layers"])
        return {"bytes": n * (case["seq"] * 2 * KROW * 2 + 2 * HID * 4 + 2 * H * 36),
                "flops": n * case["seq"] * H * D * 4}
    if kind == "step":
        n = case["layers"] * case["steps"]
        seq = case["ctx"] + (case["steps"] + 1) / 2
        wo = 1 if case["wo"] else 0
        return {"bytes": n * (seq * 2 * KROW * 2 + (HID + 2 * KROW) * 4 + 2 * HID * 4 + wo * (_W_BYTES + 2 * HID * 4)),
                "flops": n * (seq * H * D * 4 + wo * 2 * HID * HID)}
    if kind in ("layer", "attn"):
        m, P = case["m"], case["P"]
        pairs = m * P + m * (m + 1) / 2
        # the earlier rows: fp16 V, and K as int8 (fp16 when every tile is exact)
        cache = P * KROW * (3 if case["int8"] else 4)
        flops = pairs * H * D * 4
        if kind == "attn":
            return {"bytes": cache + m * KROW * 4 + m * HID * 2 + m * HID * 4, "flops": flops}
        return {"bytes": cache + m * (HID + 2 * KROW) * 4 + m * KROW * 4 + m * HID * 4 + _W_BYTES,
                "flops": flops + 2 * m * HID * HID}
    n, k, t = case["n"], case["k"], case["ntok"]
    return {"bytes": t * k * 4 + n * k // 32 * 18 + t * n * 4 * (2 if case["add"] else 1), "flops": 2 * t * n * k}


def tolerance(case):
    """About four times what a pass differs by from `exact`: the rounding of fp16
    probabilities in the prefill attention, of 32-bit sums elsewhere.  A Q8_1
    quant moves by one where its value lies near a tie, and the projection
    behind it (rel 3e-3 to 4e-3) with it; the Q4_0 product's block offset is
    rounded once per block (rel 2e-4)."""
    kind = case["kind"]
    if kind == "decode":
        return {"rel": 2e-6, "max": 4e-5, "differ": 0.002}
    if kind == "step":
        return {"rel": 4e-4, "max": 1e-2, "differ": 0.002}
    if kind == "attn":
        return {"rel": 2e-3 if case["int8"] else 8e-4}
    if kind == "layer":
        return {"rel": 1.2e-2, "max": 0.3, "differ": 0.01}
    return {"rel": 8e-4, "differ": 1e-4}


# ---- the same in 64 bits -------------------------------------------------------------
def _q8_1(x):
    """Q8_1 of rows of 32-value blocks, x float64 [..., 32]: quants, d and the sum of the block."""
    am = x.abs().amax(-1, keepdim=True)
    d = am / 127
    q = torch.where(am == 0, torch.zeros_like(x), (x / d).abs().add(0.5).floor() * x.sign())
    return q, d.half().double(), x.sum(-1, keepdim=True).half().double()


def _gemm(q, d, sm, w):
    """Q4_0 weights against Q8_1 rows: the weights' offset comes in through the blocks' sums."""
    qs, wd = w
    nib = torch.cat([qs & 15, qs >> 4], -1).double()
    a = (q * d).flatten(1) @ (nib * wd.double().unsqueeze(-1)).flatten(1).t()
    return a - 8 * (sm.squeeze(-1) @ wd.double().t())


def _rope(v, w, pos):
    """Norm and rotation of rows v float64 [n, heads, 64] at positions pos [n]."""
    y = v / torch.sqrt((v * v).mean(-1, keepdim=True) + float(torch.tensor(1e-5))) * w.double()
    f = (10000000.0 ** (-torch.arange(32, device=v.device, dtype=torch.float64) / 32)).float()
    a = (pos.float().unsqueeze(-1) * f).double().unsqueeze(1)       # the angle is an fp32 product
    c, s = torch.cos(a), torch.sin(a)
    return torch.cat([y[..., :32] * c - y[..., 32:] * s, y[..., :32] * s + y[..., 32:] * c], -1)


def _int8(x):
    """The int8 rows of fp32 rows x [..., 64] and their scales, as the quantiser's formula defines them."""
    am = x.abs().amax(-1, keepdim=True)
    return torch.round(x * torch.where(am > 0, 127 / am, torch.zeros_like(am))).double(), (am / 127).double()


def _prefill(qh, kc, vc, m, P, int8, near, sink, cm=None):
    """The chunk's attention rows [m][H*D] in float64: int8 scores outside the exact tiles."""
    S = P + m
    out = torch.empty(m, H, D, dtype=torch.float64, device="cuda")
    qh = qh.view(m, H, D)
    step = max(64, min(m, (1 << 26) // S // 64 * 64))
    kpos = torch.arange(S, device="cuda")
    for h in range(H):
        k, v = kc[:S, h // 4].double(), vc[:S, h // 4].double()
        c = cm[h // 4] if cm is not None else torch.zeros(D, device="cuda")
        if int8:
            k8, ksc = _int8(kc[:S, h // 4].float() - c)
            q8, qsc = _int8(qh[:, h].float())
            k8t = (k8 * ksc).t().contiguous()
            q8 = q8 * qsc
        kt = k.t().contiguous()
        for a in range(0, m, step):
            b = min(m, a + step)
            hi = P + b
            q = qh[a:b, h].double()
            sc = q @ kt[:, :hi]
            if int8:
                row = torch.arange(a, b, device="cuda").unsqueeze(1)
                tile = kpos[:hi].unsqueeze(0) // 64
                exact = tile * 64 + 64 > P + row // 32 * 32 - near
                if sink:
                    exact |= tile == 0
                # smoothed keys: the rows' common part of the scores is taken off the exact ones too
                sc = torch.where(exact, sc - (q @ c.double()).unsqueeze(1), q8[a:b] @ k8t[:, :hi])
            sc.masked_fill_(kpos[:hi].unsqueeze(0) > P + torch.arange(a, b, device="cuda").unsqueeze(1), -math.inf)
            sc -= sc.amax(-1, keepdim=True)
            sc.exp_()
            out[a:b, h] = (sc @ v[:hi]) / sc.sum(-1, keepdim=True)
    return out.view(m, HID)


def _decode_one(q, k, v):
    out = torch.empty(H, D, dtype=torch.float64, device="cuda")
    for h in range(KV):
        s = q[4 * h:4 * h + 4].double() @ k[:, h].double().t().contiguous() / 8
        out[4 * h:4 * h + 4] = torch.softmax(s, -1) @ v[:, h].double().contiguous()
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        qs, kcs, vcs = _decode_inputs(case, seed)
        return {"out": [_decode_one(q, k, v) for q, k, v in zip(qs, kcs, vcs)], "yq8": [None for _ in qs]}
    if kind == "step":
        layers, x = _step_inputs(case, seed)
        x, outs = x.double(), [None] * len(layers)
        for t in range(case["steps"]):
            pos = case["ctx"] + t
            at = torch.tensor([pos], device="cuda")
            for i, L in enumerate(layers):
                L["kc"][pos] = _rope(L["k_src"].double().unsqueeze(0), L["k_norm"], at)[0].half()
                L["vc"][pos] = L["v_src"].half()
                q = _rope(L["q_src"].double().unsqueeze(0), L["q_norm"], at)[0]
                outs[i] = _decode_one(q, L["kc"][:pos + 1], L["vc"][:pos + 1])
                if case["wo"]:
                    b = _q8_1(outs[i].view(1, -1, 32))
                    x = x + _gemm(b[0], b[1], b[2], (L["wo_qs"], L["wo_d"]))[0]
        new = slice(case["ctx"], case["ctx"] + case["steps"])
        return {"out": outs, "k": [L["kc"][new].double() for L in layers],
                "v": [L["vc"][new].double() for L in layers], "x": x if case["wo"] else None}
    if kind == "layer":
        m, P = case["m"], case["P"]
        Y, kc, vc, norms, w = _layer_inputs(case, seed)
        Yd = Y.double()
        pos = torch.arange(P, P + m, device="cuda")
        qh = (_rope(Yd[:, :HID].view(m, H, D), norms[0], pos) / 8).half()
        kc[P:] = _rope(Yd[:, HID:HID + KROW].view(m, KV, D), norms[1], pos).half()
        vc[P:] = Y[:, HID + KROW:].view(m, KV, D).half()
        cm = kc.double().mean(0).float() if case["smooth"] else None
        o = _prefill(qh, kc, vc, m, P, case["int8"], case["near"], case["sink"], cm)
        q, d, sm = _q8_1(o.view(m, -1, 32))
        return {"aqs": None, "asc": torch.cat([d, 8 * sm], -1), "x": _gemm(q, d, sm, w), "k": kc[P:].double(),
                "v": vc[P:].double()}
    if kind == "attn":
        qh, kc, vc = _attn_inputs(case, seed)
        return {"o": _prefill(qh, kc, vc, case["m"], case["P"], case["int8"], case["near"], case["sink"])}
    X, w, res = _linear_inputs(case, seed)
    q, d, sm = _q8_1(X.double().view(case["ntok"], -1, 32))
    out = _gemm(q, d, sm, w)
    return {"qs": None, "sc": torch.cat([d, 8 * sm], -1), "out": out + res.double() if case["add"] else out}
