"""The work that a program on this framework has it do, as cases that can be timed and compared.

Four families, each through the public entry points that a program calls:

* ``attention`` -- :func:`lucid_amd.lucid_attention`: a training step's forward and backward, or
  the forward alone as a prefill calls it (O and the V' rows that fill the cache);
* ``decode``    -- :func:`lucid_amd.lucid.lucid_decode`: new tokens against a (K, V') cache;
* ``path``      -- the LUCID-Path layer (:func:`lucid_amd.lucid_path.lucid_path_layer_attention`:
  the key-key solve, then PaTH softmax attention on its V') or one of its two halves;
* ``block``     -- one decoder layer (:class:`lucid_amd.modeling_lucid.LlamaDecoderLayer`):
  norms, stacked projections, rotary embedding, attention, MLP, forward and backward.

Inputs have the values these paths meet in a model: queries, keys and values of unit variance
(projections of normalised activations), stored as the ``[B, T, H, d]`` projections they are
views of; ``shared`` is the share of the kv heads whose keys lie along a common direction, as
those of trained heads often do (they run the split-precision chains).  ``exact`` evaluates the
definitions densely in float64 torch.
"""
import math

import torch

DEV = "cuda:0"
EPS = 1e-5
_DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # one token of an interactive session just begun: the smallest call, latency alone
        {"name": "decode_short", "op": "decode", "B": 1, "Hq": 16, "Hkv": 16, "d": 64, "cache": 300, "new": 1},
        # one token at the end of a 128K context, grouped heads: the cache is read once
        {"name": "decode_long", "op": "decode", "B": 1, "Hq": 32, "Hkv": 8, "d": 128, "cache": 131072, "new": 1},
        # a batch of chats of the reference model's heads (head dim 68), several new tokens each
        {"name": "decode_batch", "op": "decode", "B": 8, "Hq": 32, "Hkv": 4, "d": 68, "cache": 2900, "new": 5},
        # a small ragged training batch, as fine-tuning on short examples makes it
        {"name": "train_short", "op": "attention", "B": 2, "Hq": 8, "Hkv": 8, "T": 333, "d": 64, "dtype": "bf16",
         "grad": True, "shared": 0.0},
        # the attention of a pre-training step at an ordinary context
        {"name": "train_4k", "op": "attention", "B": 4, "Hq": 16, "Hkv": 16, "T": 4096, "d": 64, "dtype": "bf16",
         "grad": True, "shared": 0.0},
        # the attention of a long-context training step: the largest
        {"name": "train_32k", "op": "attention", "B": 1, "Hq": 16, "Hkv": 16, "T": 32768, "d": 64, "dtype": "bf16",
         "grad": True, "shared": 0.0},
        # long-context fine-tuning at the reference model's grouping, half of the heads trained
        # to a common key direction
        {"name": "finetune_gqa", "op": "attention", "B": 1, "Hq": 32, "Hkv": 4, "T": 16000, "d": 64, "dtype": "bf16",
         "grad": True, "shared": 0.5},
        # the reference model's attention as it is shipped: fp32, head dim 68, 32 / 4 heads
        {"name": "train_f32", "op": "attention", "B": 8, "Hq": 32, "Hkv": 4, "T": 2048, "d": 68, "dtype": "f32",
         "grad": True, "shared": 0.0},
        # the prefill of a long prompt whose length is what it is, wide grouped heads
        {"name": "prefill_128", "op": "attention", "B": 1, "Hq": 32, "Hkv": 8, "T": 30011, "d": 128, "dtype": "bf16",
         "grad": False, "shared": 0.0},
        # training with the same wide grouped heads
        {"name": "train_128", "op": "attention", "B": 1, "Hq": 32, "Hkv": 8, "T": 8192, "d": 128, "dtype": "bf16",
         "grad": True, "shared": 0.0},
        # one LUCID-Path layer of a training step: the solve and the PaTH softmax, both directions
        {"name": "path_layer", "op": "path", "kind": "layer", "B": 1, "HQ": 16, "H": 16, "T": 8192, "K": 64,
         "dtype": "bf16", "grad": True},
        # one decoder layer of a training step, with its norms, projections, rotation and MLP
        {"name": "decoder_layer", "op": "block", "B": 1, "T": 4096, "hidden": 2048, "inter": 5632, "heads": 32,
         "kv": 32, "rope": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# a drawn case's bound: score products of the largest listed case, B (Hq + Hkv) T^2 d of train_32k
_MOST = 32 * 32768 ** 2 * 64


def draw(rng):
    op = rng.choice(["attention", "attention", "attention", "decode", "path", "block"])
    if op == "attention":
        hq, hkv = rng.choice([(8, 8), (16, 16), (32, 32), (32, 8), (32, 4), (12, 4), (4, 1)])
        c = {"op": op, "B": rng.choice([1, 1, 2, 3, 4, 8]), "Hq": hq, "Hkv": hkv, "T": _log(rng, 64, 32768),
             "d": rng.choice([64, 64, 64, 68, 80, 96, 128, 128]), "dtype": rng.choice(["bf16", "bf16", "bf16", "f32"]),
             "grad": rng.random() < 0.7, "shared": rng.choice([0.0, 0.0, 0.5])}
        # the split-precision products of fp32 and of shared keys cost up to four times as much
        weight = (4 if c["dtype"] == "f32" else 2 if c["shared"] else 1) * c["B"] * (hq + hkv) * (64 if c["d"] == 64 else 128)
        c["T"] = max(64, min(c["T"], int((0.6 * _MOST / weight) ** 0.5)))
        return c
    if op == "decode":
        hq, hkv = rng.choice([(16, 16), (32, 8), (32, 4), (12, 4)])
        c = {"op": op, "B": rng.choice([1, 1, 2, 4, 8]), "Hq": hq, "Hkv": hkv, "d": rng.choice([64, 68, 128]),
             "cache": _log(rng, 100, 131072), "new": rng.choice([1, 1, 1, 2, 5, 8])}
        c["cache"] = min(c["cache"], 2 ** 20 // (c["B"] * hkv))
        return c
    if op == "path":
        hq, h = rng.choice([(8, 8), (16, 16), (32, 4), (8, 2)])
        c = {"op": op, "kind": rng.choice(["solve", "softmax", "layer"]), "B": rng.choice([1, 1, 2]), "HQ": hq, "H": h,
             "T": _log(rng, 64, 8192), "K": rng.choice([64, 64, 128]), "dtype": "bf16", "grad": rng.random() < 0.7}
        if c["K"] == 64 and rng.random() < 0.3:
            c["dtype"] = "f32"
        return c
    heads = rng.choice([8, 16, 32])
    return {"op": op, "B": rng.choice([1, 2]), "T": _log(rng, 64, 2048), "hidden": 64 * heads, "inter": 176 * heads,
            "heads": heads, "kv": rng.choice([heads, heads // 4]), "rope": rng.random() < 0.7}


# --------------------------------------------------------------------------------------------
# inputs, from the seed alone
# --------------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _keys(g, case, B, T, Hkv, d):
    """Keys [B, T, Hkv, d] of unit variance; the first ``shared`` of the heads a common direction
    with half as much of their own beside it."""
    k = _randn(g, B, T, Hkv, d)
    n = int(round(case.get("shared", 0.0) * Hkv))
    if n:
        k[:, :, :n] = (_randn(g, B, 1, n, d) + 0.5 * k[:, :, :n]) / 1.25 ** 0.5
    return k


def _inputs(case, seed):
    """The tensors of a case in its dtype, in the order its entry point takes them."""
    g = _gen(seed)
    op = case["op"]
    if op == "attention":
        B, Hq, Hkv, T, d = (case[n] for n in ("B", "Hq", "Hkv", "T", "d"))
        dt = _DTYPES[case["dtype"]]
        q, k, v = _randn(g, B, T, Hq, d), _keys(g, case, B, T, Hkv, d), _randn(g, B, T, Hkv, d)
        do = _randn(g, B, T, Hq, d)
        return {"q": q.to(dt), "k": k.to(dt), "v": v.to(dt), "do": do.to(dt)}
    if op == "decode":
        B, Hq, Hkv, d, n, L = (case[x] for x in ("B", "Hq", "Hkv", "d", "cache", "new"))
        bf = torch.bfloat16
        cap = -(-(n + L) // 256) * 256  # the cache grows in steps, as LucidCache's does
        dp = 64 if d <= 64 else 128
        kc, vc = (torch.zeros(B, Hkv, cap, dp, dtype=bf, device=DEV) for _ in range(2))
        for c in (kc, vc):
            c[:, :, :n, :d] = torch.randn(B, Hkv, n, d, generator=g, device=DEV, dtype=bf)
        q, k, v = (_randn(g, B, L, h, d).to(bf).transpose(1, 2) for h in (Hq, Hkv, Hkv))
        return {"q": q, "k": k, "v": v, "kc": kc, "vc": vc}
    if op == "path":
        B, HQ, H, T, K = (case[n] for n in ("B", "HQ", "H", "T", "K"))
        dt = _DTYPES[case["dtype"]]
        q, k, v, w = (_randn(g, B, T, h, K) for h in (HQ, H, H, H))
        w = w / w.norm(dim=-1, keepdim=True)
        beta = 2 * torch.sigmoid(_randn(g, B, T, H))
        do = _randn(g, B, T, HQ, K)
        return {n: x.to(dt) for n, x in (("q", q), ("k", k), ("v", v), ("w", w), ("beta", beta), ("do", do))}
    hid, inter, kv = case["hidden"], case["inter"], 64 * case["kv"]
    out = {"x": _randn(g, case["B"], case["T"], hid), "dy": _randn(g, case["B"], case["T"], hid)}
    for n, shape in (("self_attn.q_proj.weight", (hid, hid)), ("self_attn.k_proj.weight", (kv, hid)),
                     ("self_attn.v_proj.weight", (kv, hid)), ("self_attn.o_proj.weight", (hid, hid)),
                     ("mlp.gate_proj.weight", (inter, hid)), ("mlp.up_proj.weight", (inter, hid)),
                     ("mlp.down_proj.weight", (hid, inter))):
        out[n] = _randn(g, *shape) * hid ** -0.5
    for n in ("input_layernorm.weight", "post_attention_layernorm.weight"):
        out[n] = 1 + 0.1 * _randn(g, hid)
    return {n: x.to(torch.bfloat16) for n, x in out.items()}


def prepare(case, seed):
    x = _inputs(case, seed)
    op = case["op"]
    if op == "attention":  # the [B, H, T, d] views of the projections that the layer passes on
        leaves = [x[n].transpose(1, 2).requires_grad_(case["grad"]) for n in ("q", "k", "v")]
        return {"case": case, "leaves": leaves, "do": x["do"]}
    if op == "decode":
        return {"case": case, **x}
    if op == "path":
        leaves = [x[n].requires_grad_(case["grad"]) for n in ("q", "k", "v", "w", "beta")]
        return {"case": case, "leaves": leaves, "do": x["do"]}
    from lucid_amd.modeling_lucid import LlamaDecoderLayer, LlamaRotaryEmbedding, LucidConfig

    cfg = LucidConfig(hidden_size=case["hidden"], intermediate_size=case["inter"], num_attention_heads=case["heads"],
                      num_key_value_heads=case["kv"], use_rope=case["rope"])
    with torch.device(DEV):
        layer = LlamaDecoderLayer(cfg, 0).to(torch.bfloat16)
        rotary = LlamaRotaryEmbedding(cfg)
    inp = x.pop("x").requires_grad_()
    dy = x.pop("dy")
    layer.load_state_dict(x)
    pos = torch.arange(case["T"], device=DEV)[None].expand(case["B"], -1)
    return {"case": case, "layer": layer, "x": inp, "dy": dy, "pe": rotary(inp, pos),
            "leaves": [inp] + [dict(layer.named_parameters())[n] for n in _BLOCK_PARAMS]}


_BLOCK_PARAMS = ("self_attn.q_proj.weight", "self_attn.k_proj.weight", "self_attn.v_proj.weight",
                 "self_attn.o_proj.weight", "mlp.gate_proj.weight", "mlp.up_proj.weight", "mlp.down_proj.weight",
                 "input_layernorm.weight", "post_attention_layernorm.weight")


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "attention":
        from lucid_amd import lucid_attention

        q, k, v = state["leaves"]
        if not case["grad"]:
            with torch.no_grad():
                o, vp = lucid_attention(q, k, v, return_vprime=True)
            return {"o": o, "vprime": vp}
        o = lucid_attention(q, k, v)
        dq, dk, dv = torch.autograd.grad(o, (q, k, v), state["do"])
        return {"o": o.detach(), "dq": dq, "dk": dk, "dv": dv}
    if op == "decode":
        from lucid_amd.lucid import lucid_decode

        n, L, d = case["cache"], case["new"], case["d"]
        with torch.no_grad():
            o, vp = lucid_decode(state["q"], state["k"], state["v"], state["kc"], state["vc"], n)
        # with the rows that the call wrote into the caches (nothing else in them changes)
        return {"o": o, "vprime": vp, "k_rows": state["kc"][:, :, n:n + L, :d], "vprime_rows": state["vc"][:, :, n:n + L, :d]}
    if op == "path":
        from lucid_amd.lucid_path import (lucid_path_layer_attention, parallel_lucid_path_attention,
                                          parallel_path_attention)

        q, k, v, w, beta = state["leaves"]
        with torch.set_grad_enabled(case["grad"]):
            if case["kind"] == "layer":
                o = lucid_path_layer_attention(q, k, v, w, beta)
            elif case["kind"] == "solve":
                o, _ = parallel_lucid_path_attention(k, v, w, beta, q=q)
            else:
                o, _ = parallel_path_attention(q, k, v, w, beta)
        if not case["grad"]:
            return {"o": o}
        dq, dk, dv, dw, dbeta = torch.autograd.grad(o, (q, k, v, w, beta), state["do"])
        return {"o": o.detach(), "dq": dq, "dk": dk, "dv": dv, "dw": dw, "dbeta": dbeta}
    y = state["layer"](state["x"], state["pe"])
    grads = torch.autograd.grad(y, state["leaves"], state["dy"])
    return {"y": y.detach(), "dx": grads[0], **{"d " + n: g for n, g in zip(_BLOCK_PARAMS, grads[1:])}}


def work(case):
    op = case["op"]
    if op == "attention":
        # P (or the softmax) and its product with V', T^2 d each over the causal half; backward:
        # the scores once more and four products
        B, Hq, Hkv, T, d = (case[n] for n in ("B", "Hq", "Hkv", "T", "d"))
        size = 4 if case["dtype"] == "f32" else 2
        n = (7 if case["grad"] else 2) * T * T * d * B * (Hq + Hkv)
        moved = B * T * d * (Hq + Hkv) * size * (4 if case["grad"] else 2)  # q, k, v, o (do, dq, dk, dv)
        return {"bytes": moved + (0 if case["grad"] else B * T * d * Hkv * (4 - size)), "flops": n}
    if op == "decode":
        B, Hq, Hkv, d, n, L = (case[x] for x in ("B", "Hq", "Hkv", "d", "cache", "new"))
        return {"bytes": 2 * B * (2 * Hkv * n * d + 2 * Hq * L * d + 6 * Hkv * L * d),
                "flops": 4 * B * (Hq + Hkv) * L * n * d}
    if op == "path":
        B, HQ, H, T, K = (case[n] for n in ("B", "HQ", "H", "T", "K"))
        size = 4 if case["dtype"] == "f32" else 2
        per = (7 if case["grad"] else 2) * T * T * K * B
        n = per * ((H if case["kind"] == "layer" else 0) + HQ)
        return {"bytes": B * T * K * (2 * HQ + 3 * H) * size * (2 if case["grad"] else 1), "flops": n}
    B, T, hid, inter, kv = case["B"], case["T"], case["hidden"], case["inter"], 64 * case["kv"]
    weights = 2 * hid * hid + 2 * kv * hid + 3 * hid * inter
    return {"bytes": 2 * (2 * weights + 4 * B * T * hid),
            "flops": 6 * B * T * weights + 7 * T * T * 64 * B * (case["heads"] + case["kv"])}


def tolerance(case):
    """About four times what the worst output of a case is off ``exact`` by (2-norm; measured over
    the listed cases and 40 others of their ranges).  ``max`` is the largest difference over a
    result's root mean square: bf16 probabilities and their products leave a few rows (the first
    of a long sequence, with few keys) far above the rest."""
    f32 = case.get("dtype") == "f32"
    if case["op"] == "attention":
        if f32:  # 8e-6 (1.7e-5 along a common key direction), max 6.5e-4
            return {"rel": 7e-5 if case["shared"] else 4e-5, "max": 3e-3}
        return {"rel": 1.5e-2, "max": 0.6}  # 3e-3 to 5.4e-3, max 0.33
    if case["op"] == "path":
        return {"rel": 7e-5, "max": 3e-3} if f32 else {"rel": 1.5e-2, "max": 0.6}  # 1.7e-5, 2.7e-4; 3.9e-3, 0.25
    if case["op"] == "decode":
        return {"rel": 9e-3, "max": 4e-2}  # 2.3e-3, 8.4e-3
    return {"rel": 3e-2, "max": 0.2}  # 9.8e-3, 5.5e-2


# --------------------------------------------------------------------------------------------
# the definitions in float64
# --------------------------------------------------------------------------------------------

def _causal(T, strict=False):
    return torch.ones(T, T, dtype=torch.bool, device=DEV).tril_(-1 if strict else 0)


def _v_prime(k, v, scale):
    """V' = P^-1 V of one kv head, P_ij = exp(s K^_i K^_j - 1/s) for j <= i, K^ = RMSNorm(K)."""
    kh = k * torch.rsqrt(k.pow(2).mean(-1, keepdim=True) + EPS)
    p = torch.exp((scale * (kh @ kh.T) - 1.0 / scale).masked_fill(~_causal(k.shape[0]), float("-inf")))
    return torch.linalg.solve_triangular(p, v, upper=False)


def _softmax_on(q, k, vp, scale):
    s = (scale * (q @ k.T)).masked_fill(~_causal(q.shape[0]), float("-inf"))
    return torch.softmax(s, -1) @ vp


def _attention(q, k, v, do):
    """[B, T, H, d] float64: O, V' and (do given) dq, dk, dv, one kv head after the other."""
    B, T, Hq, d = q.shape
    Hkv = k.shape[2]
    G, scale = Hq // Hkv, d ** -0.5
    out = {"o": torch.empty_like(q), "vprime": torch.empty_like(v)}
    if do is not None:
        out.update(dq=torch.empty_like(q), dk=torch.empty_like(k), dv=torch.empty_like(v))
    for b in range(B):
        for h in range(Hkv):
            kb, vb = (x[b, :, h].detach().clone().requires_grad_(do is not None) for x in (k, v))
            vp = _v_prime(kb, vb, scale)
            vl = vp.detach().clone().requires_grad_(do is not None)
            out["vprime"][b, :, h] = vl.detach()
            for i in range(h * G, h * G + G):
                qb = q[b, :, i].detach().clone().requires_grad_(do is not None)
                o = _softmax_on(qb, kb, vl, scale)
                out["o"][b, :, i] = o.detach()
                if do is not None:
                    o.backward(do[b, :, i])
                    out["dq"][b, :, i] = qb.grad
                del o, qb
            if do is not None:
                vp.backward(vl.grad)
                out["dk"][b, :, h], out["dv"][b, :, h] = kb.grad, vb.grad
            del vp, vl, kb, vb
    return out


def _decode(x, n, L):
    q, k, v, kc, vc = (x[i].double() for i in ("q", "k", "v", "kc", "vc"))
    B, Hq, _, d = q.shape
    Hkv = k.shape[1]
    G, scale = Hq // Hkv, d ** -0.5
    keys = torch.cat([kc[:, :, :n, :d], k], 2)
    kh = keys * torch.rsqrt(keys.pow(2).mean(-1, keepdim=True) + EPS)
    vps = torch.cat([vc[:, :, :n, :d], torch.zeros_like(v)], 2)
    vp = torch.empty_like(v)
    o = torch.empty(B, L, Hq, d, dtype=torch.float64, device=DEV)
    for t in range(L):
        m = n + t
        p = torch.exp(scale * (kh[:, :, m:m + 1] @ kh[:, :, :m + 1].transpose(-1, -2)) - 1.0 / scale)
        vp[:, :, t] = (v[:, :, t] - (p[..., :m] @ vps[:, :, :m])[:, :, 0]) / p[:, :, 0, m:]
        vps[:, :, m] = vp[:, :, t]
        s = scale * (q[:, :, t].reshape(B, Hkv, G, d) @ keys[:, :, :m + 1].transpose(-1, -2).contiguous())
        o[:, t] = (torch.softmax(s, -1) @ vps[:, :, :m + 1]).reshape(B, Hq, d)
    return {"o": o, "vprime": vp, "k_rows": k, "vprime_rows": vp}


def _path_logits(q, k, w, beta):
    """A_ij = q_i H_i ... H_{j+1} k_j (j <= i), H = I - beta w w^T: the whole sequence as one
    block of the WY form."""
    T = k.shape[0]
    wb = beta[:, None] * w
    a = torch.eye(T, dtype=w.dtype, device=DEV) + (wb @ w.T).tril(-1)
    inner = torch.linalg.solve_triangular(a, (wb @ k.T).tril(-1), upper=False, unitriangular=True)
    return q @ k.T - (q @ w.T).tril() @ inner


def _path_head(kind, q, k, v, w, beta, scale):
    A = _path_logits(q, k, w, beta)
    if kind == "softmax":
        return torch.softmax((scale * A).masked_fill(~_causal(A.shape[0]), float("-inf")), -1) @ v
    L = torch.exp((scale * A - 1.0 / scale).masked_fill(~_causal(A.shape[0], True), float("-inf")))
    return torch.linalg.solve_triangular(L, v, upper=False, unitriangular=True)


def _path(case, x):
    names = ("q", "k", "v", "w", "beta")
    full = {n: x[n].double() for n in names}
    B, T, HQ, K = full["q"].shape
    H = full["k"].shape[2]
    G, scale, grad = HQ // H, K ** -0.5, case["grad"]
    out = {"o": torch.empty(B, T, HQ, K, dtype=torch.float64, device=DEV)}
    if grad:
        out.update({"d" + n: torch.zeros_like(full[n]) for n in names})
    for b in range(B):
        for h in range(H):
            k, v, w, beta = (full[n][b, :, h].detach().clone().requires_grad_(grad) for n in names[1:])
            vp = _path_head("solve", k, k, v, w, beta, scale) if case["kind"] == "layer" else v
            vl = vp.detach().clone().requires_grad_(grad)
            for i in range(h * G, h * G + G):
                q = full["q"][b, :, i].detach().clone().requires_grad_(grad)
                o = _path_head("solve" if case["kind"] == "solve" else "softmax", q, k, vl, w, beta, scale)
                out["o"][b, :, i] = o.detach()
                if grad:
                    o.backward(x["do"][b, :, i].double())
                    out["dq"][b, :, i] = q.grad
                del o, q
            if grad:
                vp.backward(vl.grad)
                for n, t in zip(names[1:], (k, v, w, beta)):
                    out["d" + n][b, :, h] = t.grad
            del vp, vl
    return out


def _block(case, x):
    p = {n: t.double().requires_grad_() for n, t in x.items() if n != "dy"}
    B, T, hid, heads, kv = case["B"], case["T"], case["hidden"], case["heads"], case["kv"]

    def norm(h, w):
        return w * (h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + EPS))

    def rotate(t):
        if not case["rope"]:
            return t
        freq = 10000.0 ** (-torch.arange(0, 64, 2, device=DEV).double() / 64)
        ang = torch.arange(T, device=DEV).double()[:, None] * torch.cat((freq, freq))
        half = torch.cat((-t[..., 32:], t[..., :32]), -1)
        return t * ang.cos()[:, None] + half * ang.sin()[:, None]

    h = norm(p["x"], p["input_layernorm.weight"])
    q = rotate((h @ p["self_attn.q_proj.weight"].T).view(B, T, heads, 64))
    k = rotate((h @ p["self_attn.k_proj.weight"].T).view(B, T, kv, 64))
    v = (h @ p["self_attn.v_proj.weight"].T).view(B, T, kv, 64)
    rows = []
    for b in range(B):
        vps = [_v_prime(k[b, :, j], v[b, :, j], 0.125) for j in range(kv)]
        rows.append(torch.stack([_softmax_on(q[b, :, i], k[b, :, i * kv // heads], vps[i * kv // heads], 0.125)
                                 for i in range(heads)], 1))
    h = p["x"] + torch.stack(rows).reshape(B, T, hid) @ p["self_attn.o_proj.weight"].T
    m = norm(h, p["post_attention_layernorm.weight"])
    gate = torch.nn.functional.silu(m @ p["mlp.gate_proj.weight"].T) * (m @ p["mlp.up_proj.weight"].T)
    y = h + gate @ p["mlp.down_proj.weight"].T
    grads = torch.autograd.grad(y, [p["x"]] + [p[n] for n in _BLOCK_PARAMS], x["dy"].double())
    return {"y": y.detach(), "dx": grads[0], **{"d " + n: g for n, g in zip(_BLOCK_PARAMS, grads[1:])}}


def exact(case, seed):
    x = _inputs(case, seed)
    if case["op"] == "attention":
        q, k, v = (x[n].double() for n in ("q", "k", "v"))
        out = _attention(q, k, v, x["do"].double() if case["grad"] else None)
        names = ("dq", "dk", "dv") if case["grad"] else ("vprime",)
        return {"o": out["o"], **{n: out[n].transpose(1, 2) for n in names}}
    if case["op"] == "decode":
        return _decode(x, case["cache"], case["new"])
    if case["op"] == "path":
        # the dense logits take a T x T x T product and solve per head
        if case["T"] ** 3 * case["B"] * (case["HQ"] + (case["H"] if case["kind"] == "layer" else 0)) > 2e13:
            return None
        return _path(case, x)
    return _block(case, x)
