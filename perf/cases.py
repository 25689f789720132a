"""The calls this framework is measured on, over the ranges its users have: the quantized MUL_MAT from one token to a
512-token prompt, a Llama-3-8B layer at prompt and decode, a decode step of a short stack with the output head, prompt
and decode attention (f16 and quantized caches), and BitNet's batched I2_S product and token step.

listed() names the cases, draw() gives more of the same ranges, prepare() makes what a program holds before the call,
run() is one call through the public entry points, work() what it cannot do without, tolerance() and exact() what it is
compared with. Weights are made here, as ggml blocks, in plain torch; exact() follows ggml's arithmetic (activations
rounded to 8 bits per block, the rest as real numbers) in 64 bits.
"""
import math

import numpy as np
import torch

DEV = "cuda"
Q4_0, Q8_0, Q4_K, Q6_K = 2, 8, 12, 14
TYPES = {"q4_0": Q4_0, "q8_0": Q8_0, "q4_K": Q4_K, "q6_K": Q6_K}
BLOCK = {Q4_0: (32, 18), Q8_0: (32, 34), Q4_K: (256, 144), Q6_K: (256, 210)}
H, N_HEAD, N_KV_HEAD, D, FF = 4096, 32, 8, 128, 14336  # the Llama-3-8B layer
VOCAB, MODEL_LAYERS, CTX = 128256, 2, 4096
BN_E, BN_F, BN_HEAD, BN_KV, BN_LAYERS, BN_VOCAB = 2560, 6912, 20, 5, 3, 65536  # BitNet b1.58 2B layers, a cut stack
BN_CTX, BN_EPS, BN_THETA = 4096, 1e-5, 500000.0
BN_SCALES = dict(scale_wq=1.2, scale_wk=1.1, scale_wv=0.9, scale_wo=0.03, scale_w_gate=0.8, scale_w_up=0.7,
                 scale_w_down=0.01)


# --------------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # one projection of one token, called by itself: a scripted check or a small model's decode without a graph
        {"name": "mul_mat_q4_0_m1", "kind": "mul_mat", "type": "q4_0", "n": 4096, "k": 4096, "m": 1},
        # a few sequences decoded together (an odd number of them) through the down projection
        {"name": "mul_mat_q6_K_m19", "kind": "mul_mat", "type": "q6_K", "n": 4096, "k": 14336, "m": 19},
        # a server's decode batch, or a short prompt, through gate / up
        {"name": "mul_mat_q4_K_m48", "kind": "mul_mat", "type": "q4_K", "n": 14336, "k": 4096, "m": 48},
        # a prompt chunk of 512 tokens through gate / up in the commonest weight type
        {"name": "mul_mat_q4_K_m512", "kind": "mul_mat", "type": "q4_K", "n": 14336, "k": 4096, "m": 512},
        # a prompt whose length is no multiple of anything through the down projection
        {"name": "mul_mat_q8_0_m331", "kind": "mul_mat", "type": "q8_0", "n": 4096, "k": 14336, "m": 331},
        # prompt processing: a whole decoder layer on 512 tokens
        {"name": "layer_prefill_q4_0", "kind": "layer_prefill", "type": "q4_0", "n_tok": 512, "pos0": 0},
        # single-stream decode with a long context: one layer's step as a program replays it from its graph
        {"name": "layer_decode_q4_0", "kind": "layer_decode", "type": "q4_0", "n_kv": 4096},
        # a decode step of a Q4_K_M model (layers, Q6_K output head, greedy sample) after a 512-token prompt
        {"name": "model_decode_q4_K", "kind": "model_decode", "n_kv": 513},
        # causal attention of a long prompt
        {"name": "attn_prefill", "kind": "attn_prefill", "n_tok": 2048, "pos0": 0, "masked": False},
        # the attention of a decode step over quantized caches at a long context, several layers' caches in one graph
        {"name": "attn_decode_q8_0", "kind": "attn_decode", "type": "q8_0", "n_kv": 8192, "layers": 8},
        # BitNet's FFN projection on a batch of 128 tokens
        {"name": "i2s_m128", "kind": "i2s", "n": 6912, "k": 2560, "m": 128},
        # one BitNet token through the engine, logits back to the host
        {"name": "bitnet_token", "kind": "bitnet_token", "pos": 100, "logits": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mul_mat"] * 6 + ["layer_prefill"] * 2 + ["attn_prefill"] * 2 + ["attn_decode"] * 2 +
                      ["layer_decode", "i2s", "i2s", "bitnet_token", "model_decode"])
    if kind == "mul_mat":
        t = rng.choice(list(TYPES))
        # the layer's own projections, or any: rows as they come, k in whole blocks
        n, k = rng.choice([(4096, 4096), (6144, 4096), (28672, 4096), (14336, 4096), (4096, 14336), (0, 0), (0, 0)])
        if n == 0:
            n, k = 2 * _log(rng, 512, 7168), 256 * _log(rng, 4, 56)
        return {"kind": kind, "type": t, "n": n, "k": k, "m": _log(rng, 1, 512)}
    if kind == "layer_prefill":
        n = _log(rng, 8, 512)
        return {"kind": kind, "type": rng.choice(["q4_0", "q4_K"]), "n_tok": n, "pos0": rng.choice([0, 0, rng.randrange(512)])}
    if kind == "layer_decode":
        return {"kind": kind, "type": rng.choice(["q4_0", "q4_K"]), "n_kv": _log(rng, 1, 4096)}
    if kind == "model_decode":
        return {"kind": kind, "n_kv": _log(rng, 2, 1024)}
    if kind == "attn_prefill":
        n = _log(rng, 16, 2048)
        return {"kind": kind, "n_tok": n, "pos0": rng.choice([0, rng.randrange(2048)]) if n <= 1024 else 0,
                "masked": rng.random() < 0.25}
    if kind == "attn_decode":
        return {"kind": kind, "type": rng.choice(["f16", "q8_0", "q4_0"]), "n_kv": _log(rng, 64, 16384), "layers": 8}
    if kind == "i2s":
        n, k = rng.choice([(2560, 2560), (2560, 6912), (6912, 2560), (640, 2560)])
        return {"kind": kind, "n": n, "k": k, "m": _log(rng, 1, 256)}
    return {"kind": kind, "pos": _log(rng, 1, 1024), "logits": rng.random() < 0.5}


# --------------------------------------------------------------------------------------------------- ggml blocks
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * int(seed) + 17)
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _bytes(t):
    return t.contiguous().view(torch.uint8)


def _signed_max(x):
    return x.gather(-1, x.abs().argmax(-1, keepdim=True))


def _blocks(t, x):
    """f32 rows [n, k] -> the bytes [n, row bytes] of ggml blocks of type t that hold them."""
    n, k = x.shape
    if t == Q4_0:
        x = x.view(n, k // 32, 32)
        d = _signed_max(x) / -8
        q = (x / torch.where(d == 0, 1.0, d) + 8.5).clamp(0, 15).to(torch.uint8)
        b = torch.cat([_bytes(d.half()), q[..., :16] | q[..., 16:] << 4], -1)
    elif t == Q8_0:
        x = x.view(n, k // 32, 32)
        d = x.abs().amax(-1, keepdim=True) / 127
        q = (x / torch.where(d == 0, 1.0, d)).round().to(torch.int8)
        b = torch.cat([_bytes(d.half()), _bytes(q)], -1)
    elif t == Q4_K:
        x = x.view(n, k // 256, 8, 32)
        low = (-x.amin(-1)).clamp(min=0)
        step = (x.amax(-1) + low) / 15
        d, dm = (v.amax(-1, keepdim=True).clamp(min=1e-8) / 63 for v in (step, low))
        sc, mn = (step / d).round(), (low / dm).round()
        d, dm = d.half(), dm.half()
        q = ((x + (dm.float() * mn)[..., None]) / (d.float() * sc)[..., None].clamp(min=1e-8)).round().clamp(0, 15)
        q, sc, mn = q.to(torch.uint8), sc.to(torch.uint8), mn.to(torch.uint8)
        head = torch.cat([sc[..., :4] | sc[..., 4:] >> 4 << 6, mn[..., :4] | mn[..., 4:] >> 4 << 6,
                          (sc[..., 4:] & 15) | (mn[..., 4:] & 15) << 4], -1)
        q = q.view(n, k // 256, 4, 2, 32)
        b = torch.cat([_bytes(d), _bytes(dm), head, (q[..., 0, :] | q[..., 1, :] << 4).flatten(-2)], -1)
    else:
        x = x.view(n, k // 256, 16, 16)
        step = _signed_max(x)[..., 0] / -32
        d = step.abs().amax(-1, keepdim=True).clamp(min=1e-8) / 127
        sc = (step / d).round()
        d = d.half()
        s = (d.float() * sc)[..., None]
        q = (x / torch.where(s == 0, 1.0, s)).round().clamp(-32, 31).to(torch.int8) + 32
        q = q.view(torch.uint8).view(n, k // 256, 2, 4, 32)
        ql = torch.cat([(q[..., 0:2, :] & 15) | (q[..., 2:4, :] & 15) << 4], -2).flatten(-3)
        qh = (q[..., 0, :] >> 4 | q[..., 1, :] >> 4 << 2 | q[..., 2, :] >> 4 << 4 | q[..., 3, :] >> 4 << 6).flatten(-2)
        b = torch.cat([ql, qh, _bytes(sc.to(torch.int8)), _bytes(d)], -1)
    return b.reshape(n, -1).contiguous()


def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _values(t, b, k):
    """The numbers that blocks of type t hold, in 64 bits: [n, k]."""
    n = b.shape[0]
    b = b.view(n, k // BLOCK[t][0], BLOCK[t][1])
    if t == Q4_0:
        q = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], -1).double() - 8
        v = q * _f16(b[..., :2])
    elif t == Q8_0:
        v = b[..., 2:].contiguous().view(torch.int8).double() * _f16(b[..., :2])
    elif t == Q4_K:
        h = b[..., 4:16]
        sc = torch.cat([h[..., :4] & 63, (h[..., 8:] & 15) | h[..., :4] >> 6 << 4], -1).double()
        mn = torch.cat([h[..., 4:8] & 63, h[..., 8:] >> 4 | h[..., 4:8] >> 6 << 4], -1).double()
        q = b[..., 16:].reshape(n, -1, 4, 32)
        q = torch.stack([q & 15, q >> 4], -2).view(n, -1, 8, 32).double()
        v = q * (_f16(b[..., :2]) * sc)[..., None] - (_f16(b[..., 2:4]) * mn)[..., None]
    else:
        ql, qh = b[..., :128].reshape(n, -1, 2, 2, 32), b[..., 128:192].reshape(n, -1, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], -2)
        hi = torch.cat([qh & 3, qh >> 2 & 3, qh >> 4 & 3, qh >> 6], -2)
        q = (lo | hi << 4).view(n, -1, 16, 16).double() - 32
        sc = b[..., 192:208].contiguous().view(torch.int8).double()
        v = q * (_f16(b[..., 208:]) * sc)[..., None]
    return v.reshape(n, k)


def _weight(t, g, n, k, scale=0.02):
    return torch.cat([_blocks(t, _randn(g, min(16384, n - r), k) * scale) for r in range(0, n, 16384)])


def _over(a, b):
    """a / b of 32-bit numbers, rounded once (a quotient in 64 bits first does not change it)."""
    a, b = (v.double() if isinstance(v, torch.Tensor) else v for v in (a, b))
    return (a / b).float()


def _rounded(x, t):
    """The activations as a weight of type t meets them: Q8_0 (per 32) or Q8_K (per 256) blocks of f32 rows."""
    x = x.float()
    if t in (Q4_0, Q8_0):
        b = x.reshape(*x.shape[:-1], -1, 32)
        a = b.abs().amax(-1, keepdim=True)
        q = (b * torch.where(a == 0, 0.0, _over(127.0, a))).round()
        v = q.double() * _over(a, 127.0).half().double()
    else:
        b = x.reshape(*x.shape[:-1], -1, 256)
        m = _signed_max(b)
        s = _over(-127.0, torch.where(m == 0, 1.0, m))
        q = (b * s).round().clamp(max=127)
        v = torch.where(m == 0, 0.0, q.double() * _over(1.0, s).double())
    return v.reshape(x.shape)


def _product(x, t, blocks):
    k = x.shape[-1]
    a = _rounded(x, t)
    return torch.cat([a @ _values(t, blocks[r:r + 16384], k).T for r in range(0, blocks.shape[0], 16384)], -1)


# --------------------------------------------------------------------------------------------------- layers
def _norm(x, w, eps=1e-5):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * w.double()


def _rope(x, pos):
    """x [n, heads, D] rotated in pairs (2 j, 2 j + 1) by pos [n]: the angle by repeated f32 products, as ggml does."""
    step = np.float32(np.float32(500000.0) ** np.float32(-2.0 / D))
    th = [pos.float()]
    for _ in range(D // 2 - 1):
        th.append(th[-1] * float(step))
    th = torch.stack(th, -1).double()[:, None, :]
    a, b, c, s = x[..., 0::2], x[..., 1::2], th.cos(), th.sin()
    return torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)


def _attention(q, k, v, limit=None, bias=None):
    """q [n, heads, D] over k, v [kv heads, keys, D]: query i sees the keys below limit[i] (None: all), bias [n, keys]."""
    n, heads, _ = q.shape
    out = torch.empty_like(q)
    g = heads // k.shape[0]
    hide = None if limit is None else torch.arange(k.shape[1], device=q.device)[None, :] >= limit[:, None]
    for h in range(heads):
        s = q[:, h] @ k[h // g].T / D ** 0.5
        if bias is not None:
            s = s + bias
        if hide is not None:
            s = s.masked_fill(hide, -math.inf)
        out[:, h] = s.softmax(-1) @ v[h // g]
    return out


def _layer_blocks(t, g):
    kv = N_KV_HEAD * D
    return {"qkv": _weight(t, g, H + 2 * kv, H), "o": _weight(t, g, H, H), "gu": _weight(t, g, 2 * FF, H),
            "down": _weight(t, g, H, FF), "an": 1 + 0.1 * _randn(g, H), "fn": 1 + 0.1 * _randn(g, H)}


def _cache(g, rows):
    return (_randn(g, rows, N_KV_HEAD * D).half(), _randn(g, rows, N_KV_HEAD * D).half())


def _layer(t, b, kc, vc):
    from ameva_compute_amd import llama, ops
    kv = N_KV_HEAD * D
    w = ops.QWeight.from_ggml
    lay = llama.LlamaLayer(w(t, b["qkv"], H + 2 * kv, H), w(t, b["o"], H, H), w(t, b["gu"], 2 * FF, H),
                           w(t, b["down"], H, FF), b["an"], b["fn"], N_HEAD, N_KV_HEAD, D, CTX)
    lay.k_cache[:kc.shape[0]].copy_(kc)
    lay.v_cache[:vc.shape[0]].copy_(vc)
    return lay


def _layer_exact(t, b, x, kc, vc, pos0):
    """x [n, H] in 64 bits through the layer at positions pos0 ..; kc, vc [CTX, kv] f16 get the new rows."""
    n, kv = x.shape[0], N_KV_HEAD * D
    pos = torch.arange(pos0, pos0 + n, device=x.device)
    qkv = _product(_norm(x, b["an"]), t, b["qkv"])
    q = _rope(qkv[:, :H].reshape(n, N_HEAD, D), pos)
    kc[pos0:pos0 + n] = _rope(qkv[:, H:H + kv].reshape(n, N_KV_HEAD, D), pos).reshape(n, kv).half()
    vc[pos0:pos0 + n] = qkv[:, H + kv:].half()
    kk, vv = (c[:pos0 + n].double().view(-1, N_KV_HEAD, D).transpose(0, 1) for c in (kc, vc))
    a = _attention(q.half().double(), kk, vv, pos + 1).reshape(n, H)
    x = x + _product(a, t, b["o"])
    gu = _product(_norm(x, b["fn"]), t, b["gu"])
    h = torch.nn.functional.silu(gu[:, :FF]) * gu[:, FF:]
    return x + _product(h, t, b["down"])


def _captured(fn):
    """fn's launches as a graph, as a decode loop keeps them."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fn()
    return graph


# --------------------------------------------------------------------------------------------------- per kind
def _inputs(case, seed):
    """The case's inputs from its seed alone, shared by prepare() and exact()."""
    g, kind = _gen(seed), case["kind"]
    t = TYPES.get(case.get("type"))
    s = {"g": g, "t": t}
    if kind == "mul_mat":
        s["w"] = _weight(t, g, case["n"], case["k"])
        s["x"] = _randn(g, case["m"], case["k"])
    elif kind in ("layer_prefill", "layer_decode"):
        n = case.get("n_tok", 1)
        past = case["pos0"] if kind == "layer_prefill" else case["n_kv"] - 1
        s.update(b=_layer_blocks(t, g), kv=_cache(g, past), x=_randn(g, n, H), past=past)
    elif kind == "model_decode":
        s["emb"], s["head"] = _weight(Q4_K, g, VOCAB, H), _weight(Q6_K, g, VOCAB, H)
        s["layers"] = [(_layer_blocks(Q4_K, g), _cache(g, case["n_kv"] - 1)) for _ in range(MODEL_LAYERS)]
        s["on"] = 1 + 0.1 * _randn(g, H)
        s["token"] = int(torch.randint(VOCAB, (1,), generator=g, device=DEV))
    elif kind == "attn_prefill":
        n, keys = case["n_tok"], case["pos0"] + case["n_tok"]
        s["q"], (s["k"], s["v"]) = _randn(g, n, N_HEAD, D), _cache(g, keys)
        if case["masked"]:  # ggml's KQ mask: the causal limit as 0 / -inf
            see = torch.arange(keys, device=DEV)[None, :] <= case["pos0"] + torch.arange(n, device=DEV)[:, None]
            s["mask"] = torch.zeros((n, keys), dtype=torch.float16, device=DEV).masked_fill_(~see, -math.inf)
    elif kind == "attn_decode":
        s["layers"] = []
        for _ in range(case["layers"]):
            k, v = _randn(g, case["n_kv"] * N_KV_HEAD, D), _randn(g, case["n_kv"] * N_KV_HEAD, D)
            k, v = (k.half(), v.half()) if t is None else (_blocks(t, k), _blocks(t, v))
            s["layers"].append((_randn(g, N_HEAD, D), *(c.view(case["n_kv"], N_KV_HEAD, -1) for c in (k, v))))
    elif kind == "i2s":
        s["w"] = _ternary(g, case["n"], case["k"])
        s["x"] = _randn(g, case["m"], case["k"])
    else:
        kv = BN_KV * D
        rows = {"wq": (BN_E, BN_E), "wk": (kv, BN_E), "wv": (kv, BN_E), "wo": (BN_E, BN_E), "w_gate": (BN_F, BN_E),
                "w_up": (BN_F, BN_E), "w_down": (BN_E, BN_F)}
        norms = {"attn_norm": BN_E, "attn_sub_norm": BN_E, "ffn_norm": BN_E, "ffn_sub_norm": BN_F}
        s["layers"] = [{**{n: _ternary(g, *r).cpu().numpy() for n, r in rows.items()},
                        **{n: (1 + 0.1 * _randn(g, r)).cpu().numpy() for n, r in norms.items()}, **BN_SCALES}
                       for _ in range(BN_LAYERS)]
        s["on"] = (1 + 0.1 * _randn(g, BN_E)).cpu().numpy()
        s["head"] = (0.02 * _randn(g, BN_VOCAB, BN_E)).half().cpu().numpy()
        s["x"] = (0.5 * _randn(g, BN_E)).cpu().numpy()
    return s


def _ternary(g, n, k):
    """I2_S rows: codes 0, 1, 2 with probability 1/3, four to a byte, 128 weights in 32 bytes."""
    c = torch.randint(3, (4, n, k // 4), generator=g, device=DEV, dtype=torch.uint8)
    return (c[0] << 6 | c[1] << 4 | c[2] << 2 | c[3]).contiguous()


def prepare(case, seed):
    from ameva_compute_amd import model, ops
    from ameva_compute_amd.bitnet_engine import BitNetEngine
    kind = case["kind"]
    i = _inputs(case, seed)
    t = i["t"]
    s = {"case": case}
    if kind == "mul_mat":
        s.update(w=ops.QWeight.from_ggml(t, i["w"], case["n"], case["k"]), x=i["x"])
    elif kind == "layer_prefill":
        s.update(layer=_layer(t, i["b"], *i["kv"]), x=i["x"], out=torch.empty_like(i["x"]))
        s["layer"].set_prefill_position(case["pos0"], case["n_tok"])
    elif kind == "layer_decode":
        lay, x, out = _layer(t, i["b"], *i["kv"]), i["x"][0].contiguous(), torch.empty(H, device=DEV)
        lay.set_position(i["past"])
        s.update(layer=lay, x=x, out=out, graph=_captured(lambda: lay.decode(x, out)))
    elif kind == "model_decode":
        layers = [_layer(Q4_K, b, *kv) for b, kv in i["layers"]]
        m = model.LlamaModel(i["emb"], Q4_K, layers, i["on"], ops.QWeight.from_ggml(Q6_K, i["head"], VOCAB, H))
        m.set_position(case["n_kv"] - 1)
        s.update(model=m, token=i["token"], graph=_captured(m.decode_step))
    elif kind == "attn_prefill":
        # llama.cpp's cache: a token's heads side by side
        s.update(q=i["q"], mask=i.get("mask"), **{n: i[n].view(-1, N_KV_HEAD, D).permute(1, 0, 2) for n in "kv"})
    elif kind == "attn_decode":
        need = ops.lib().amv_flash_attn_workspace_bytes(N_HEAD, N_KV_HEAD, case["n_kv"], D)
        ws = torch.empty(need, dtype=torch.uint8, device=DEV)
        ins = [(q, k.permute(1, 0, 2), v.permute(1, 0, 2)) for q, k, v in i["layers"]]

        def step():
            s["outs"] = [ops.flash_attn_decode_kv(q, k, v, 1 if t is None else t, 1 / D ** 0.5, workspace=ws)
                         for q, k, v in ins]
        s.update(ins=ins, ws=ws, graph=_captured(step))
    elif kind == "i2s":
        s.update(w=i["w"], x=i["x"])
    else:
        e = BitNetEngine()
        e.configure(BN_E, BN_F, BN_HEAD, BN_KV, D, BN_CTX, BN_LAYERS, BN_EPS, BN_THETA, True)
        for n, lay in enumerate(i["layers"]):
            e.upload_layer(n, lay)
        e.upload_output(i["on"], i["head"])
        x, xo = i["x"], np.empty(BN_E, np.float32)
        # the tokens before this one: a few rows of history, the rest of the cache as the engine clears it
        for p in range(min(8, case["pos"])):
            e.eval_token(case["pos"] - 1 - p, np.roll(x, p + 1), xo)
        s.update(engine=e, x=x, xo=xo, logits=np.empty(BN_VOCAB, np.float32) if case["logits"] else None)
    return s


def run(s):
    from ameva_compute_amd import ops
    case = s["case"]
    kind = case["kind"]
    if kind == "mul_mat":
        return ops.mul_mat(s["w"], s["x"])
    if kind == "layer_prefill":
        s["layer"].prefill(s["x"], s["out"])
        return [s["out"], s["layer"].k_cache, s["layer"].v_cache]
    if kind == "layer_decode":
        s["graph"].replay()
        return [s["out"], s["layer"].k_cache, s["layer"].v_cache]
    if kind == "model_decode":
        m = s["model"]
        m.set_position(case["n_kv"] - 1)
        m.token.fill_(s["token"])
        s["graph"].replay()
        return [m.logits] + [c for lay in m.layers for c in (lay.k_cache, lay.v_cache)]
    if kind == "attn_prefill":
        return ops.flash_attn_prefill(s["q"], s["k"], s["v"], 1 / D ** 0.5, mask=s["mask"],
                                      causal_pos0=-1 if case["masked"] else case["pos0"])
    if kind == "attn_decode":
        s["graph"].replay()
        return s["outs"]
    if kind == "i2s":
        act = ops.i2s_quantize_act(s["x"])
        return ops.i2s_gemv(s["w"], case["n"], case["k"], act, case["m"], 1.25)
    s["engine"].eval_token(case["pos"], s["x"], s["xo"], s["logits"])
    return [s["xo"]] + ([s["logits"]] if case["logits"] else [])


# --------------------------------------------------------------------------------------------------- work
def _size(t, n, k):
    return n * k // BLOCK[t][0] * BLOCK[t][1]


def work(case):
    kind, t = case["kind"], TYPES.get(case.get("type"))
    kv = N_KV_HEAD * D
    weights = [(H + 2 * kv, H), (H, H), (2 * FF, H), (H, FF)]
    per_tok = 2 * sum(n * k for n, k in weights)
    if kind == "mul_mat":
        n, k, m = case["n"], case["k"], case["m"]
        return {"bytes": _size(t, n, k) + 4 * m * (n + k), "flops": 2 * m * n * k}
    if kind in ("layer_prefill", "layer_decode"):
        n = case.get("n_tok", 1)
        past = case["pos0"] if kind == "layer_prefill" else case["n_kv"] - 1
        pairs = n * past + n * (n + 1) // 2
        return {"bytes": sum(_size(t, *w) for w in weights) + 8 * n * H + 4 * kv * (past + 2 * n),
                "flops": n * per_tok + 4 * N_HEAD * D * pairs}
    if kind == "model_decode":
        nb = MODEL_LAYERS * (sum(_size(Q4_K, *w) for w in weights) + 4 * kv * case["n_kv"])
        return {"bytes": nb + _size(Q6_K, VOCAB, H) + 4 * VOCAB,
                "flops": MODEL_LAYERS * (per_tok + 4 * N_HEAD * D * case["n_kv"]) + 2 * VOCAB * H}
    if kind == "attn_prefill":
        n, p = case["n_tok"], case["pos0"]
        return {"bytes": 8 * n * N_HEAD * D + 4 * kv * (n + p) + (2 * n * (n + p) if case["masked"] else 0),
                "flops": 4 * N_HEAD * D * (n * p + n * (n + 1) // 2)}
    if kind == "attn_decode":
        row = 2 * D if t is None else _size(t, 1, D)
        return {"bytes": case["layers"] * (2 * case["n_kv"] * N_KV_HEAD * row + 8 * N_HEAD * D),
                "flops": case["layers"] * 4 * N_HEAD * D * case["n_kv"]}
    if kind == "i2s":
        n, k, m = case["n"], case["k"], case["m"]
        return {"bytes": n * k // 4 + 4 * m * (n + k), "flops": 2 * m * n * k}
    w = 2 * BN_E * BN_E + 2 * BN_KV * D * BN_E + 3 * BN_E * BN_F
    head = BN_E * BN_VOCAB if case["logits"] else 0
    keys = BN_LAYERS * (case["pos"] + 1)
    return {"bytes": BN_LAYERS * w // 4 + 2 * head + 8 * keys * BN_KV * D,
            "flops": 2 * BN_LAYERS * w + 2 * head + 4 * keys * BN_HEAD * D}


# --------------------------------------------------------------------------------------------------- the outputs
def tolerance(case):
    """About four times what two orders of the same sums differ by (exact() against the kernels, measured)."""
    kind = case["kind"]
    if kind in ("mul_mat", "i2s", "attn_decode"):  # exact integers or f16 products, sums in 32 bits
        return {"rel": 2e-6, "max": 1e-4}
    if kind == "attn_prefill":  # probabilities rounded to 16 bits: 1.5e-4
        return {"rel": 6e-4, "max": 5e-2}
    # layers: an 8-bit rounding that falls the other way moves what follows by a step, 0.3 to 1.2 % in all
    return {"rel": 3e-2, "max": 5e-1}


def exact(case, seed):
    kind = case["kind"]
    i = _inputs(case, seed)
    t = i["t"]
    if kind == "mul_mat":
        return _product(i["x"], t, i["w"])
    if kind in ("layer_prefill", "layer_decode"):
        kc, vc = _filled(i["kv"])
        return [_row(_layer_exact(t, i["b"], i["x"].double(), kc, vc, i["past"]), kind), kc.double(), vc.double()]
    if kind == "model_decode":
        x = _values(Q4_K, i["emb"][i["token"]:i["token"] + 1], H)
        caches = []
        for b, kv in i["layers"]:
            kc, vc = _filled(kv)
            x = _layer_exact(Q4_K, b, x, kc, vc, case["n_kv"] - 1)
            caches += [kc.double(), vc.double()]
        return [_product(_norm(x, i["on"]), Q6_K, i["head"])[0]] + caches
    if kind == "attn_prefill":
        n = case["n_tok"]
        kk, vv = (i[c].double().view(-1, N_KV_HEAD, D).transpose(0, 1) for c in "kv")
        return _attention(i["q"].half().double(), kk, vv, case["pos0"] + 1 + torch.arange(n, device=DEV))
    if kind == "attn_decode":
        outs = []
        for q, k, v in i["layers"]:
            if t is None:
                q, k, v = q.half().double(), k.double(), v.double()
            else:  # a quantized K meets q in 8 bits
                q = _rounded(q, Q8_0)
                k, v = (_values(t, c.reshape(-1, c.shape[-1]), D).view(-1, N_KV_HEAD, D) for c in (k, v))
            outs.append(_attention(q[None], k.transpose(0, 1), v.transpose(0, 1))[0])
        return outs
    if kind == "i2s":
        a, scale = _bn_rounded(i["x"])
        return (a @ _bn_values(i["w"], case["k"]).T) * (scale * 1.25)
    return _bn_exact(case, i)


def _filled(kv):
    full = [torch.zeros((CTX, N_KV_HEAD * D), dtype=torch.float16, device=DEV) for _ in kv]
    for c, p in zip(full, kv):
        c[:p.shape[0]] = p
    return full


def _row(x, kind):
    return x[0] if kind == "layer_decode" else x


def _bn_rounded(x):
    """BitNet's activation rows: int8 by the row's largest magnitude (halves away from zero), and the step."""
    x = x.float()
    s = _over(127.0, x.abs().amax(-1, keepdim=True).clamp(min=1e-7))
    y = x * s
    q = torch.where((y.abs() - y.abs().floor()) == 0.5, y.sign() * (y.abs() + 0.5).floor(), y.round())
    return q.clamp(-127, 127).double(), _over(1.0, s).double()


def _bn_values(w, k):
    w = w.view(w.shape[0], k // 128, 1, 32)
    c = torch.cat([w >> 6 & 3, w >> 4 & 3, w >> 2 & 3, w & 3], -2)
    return c.reshape(w.shape[0], k).double() - 1


def _bn_exact(case, i):
    layers = [{n: torch.from_numpy(v).to(DEV) if isinstance(v, np.ndarray) else v for n, v in lay.items()}
              for lay in i["layers"]]
    on, head, x0 = (torch.from_numpy(i[n]).to(DEV).double() for n in ("on", "head", "x"))
    caches = [[torch.zeros((case["pos"] + 1, BN_KV, D), dtype=torch.float64, device=DEV) for _ in "kv"] for _ in layers]

    def project(x, lay, name):
        a, step = _bn_rounded(x)
        return (_bn_values(lay[name], x.shape[-1]) @ a) * (step * lay["scale_" + name])

    def rope(v, pos):
        f = torch.arange(D // 2, device=DEV).float() * 2 / D
        th = (torch.tensor(float(pos), device=DEV) / torch.pow(torch.tensor(BN_THETA, device=DEV), f)).double()
        a, b = v[..., :D // 2], v[..., D // 2:]
        return torch.cat([a * th.cos() - b * th.sin(), b * th.cos() + a * th.sin()], -1)

    def token(x, pos):
        for lay, (kc, vc) in zip(layers, caches):
            n = _norm(x, lay["attn_norm"], BN_EPS)
            q = rope(project(n, lay, "wq").view(BN_HEAD, D), pos)
            kc[pos] = rope(project(n, lay, "wk").view(BN_KV, D), pos)
            vc[pos] = project(n, lay, "wv").view(BN_KV, D)
            a = _attention(q[None], kc[:pos + 1].transpose(0, 1), vc[:pos + 1].transpose(0, 1)).reshape(BN_E)
            x = x + project(_norm(a, lay["attn_sub_norm"], BN_EPS), lay, "wo")
            n = _norm(x, lay["ffn_norm"], BN_EPS)
            h = project(n, lay, "w_gate").clamp(min=0).square() * project(n, lay, "w_up")
            x = x + project(_norm(h, lay["ffn_sub_norm"], BN_EPS), lay, "w_down")
        return x

    for p in range(min(8, case["pos"])):
        token(x0.roll(p + 1), case["pos"] - 1 - p)
    x = token(x0, case["pos"])
    return [x] + ([head @ _norm(x, on, BN_EPS)] if case["logits"] else [])
