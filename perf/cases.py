"""The work a decoder hands to this framework, as cases that can be timed.

A case is one call sequence through the public classes of tsugumi_amd, with the
buffers a decoder holds when it makes it. Six kinds:

  qmv       one int4 projection of 1..8 token rows (DequantInt4GEMV)
  dense     what a decoder layer has beside its experts, layer after layer: the
            Q, K, V and O projections and the dense int4 MLP of 1..8 token rows
            (DequantInt4GEMV, SharedExpertInt4)
  decode    the MoE layers of one decoded token (MoE.encode_decode_layer*)
  verify    the MoE layers of a speculative block of 2..8 tokens
  prefill   one MoE layer of a prompt chunk: router, grouping, grouped GEMMs,
            token-major sum
  qmm       one int4 projection of a prompt chunk (PrefillInt4QMM)

Weights are synthetic: nibbles uniform in 0..15, bf16 group scales
|N(0, 0.02)| / 7, under the affine scheme biases near -7.5 scales, router rows
N(0, 1 / sqrt(d)). Hidden states are N(0, 1) in fp16; `share` is the part of
their power that all rows of a call have in common, which gives the experts
loads as uneven as a real router's (0.5 of it comes near Zipf(1.1) over 128
experts) and lets the tokens of a speculative block agree on about half of
their experts (0.9).
"""
import math

import numpy as np
import torch

import tsugumi_amd as tsg

TOP_K = 8
GEMMA = {"d": 2816, "f": 704, "experts": 128, "act": "gelu"}
QWEN = {"d": 2048, "f": 512, "experts": 256, "act": "silu"}
SYM32 = {"group": 32, "scheme": "sym"}
AFFINE64 = {"group": 64, "scheme": "affine"}


def listed():
    return [
        # the smallest call: one gate-sized projection of one token
        {"name": "qmv_704", "kind": "qmv", "rows": 1, "m": 704, "n": 2816, **SYM32},
        # one token through the dense matrices of a 30-layer decoder
        {"name": "dense_token", "kind": "dense", "rows": 1, "d": 2816, "q": 4096, "kv": 2048,
         "f": 2112, "layers": 30, **SYM32},
        # the same for a speculative block of five, in the default format
        {"name": "dense_block5", "kind": "dense", "rows": 5, "d": 2816, "q": 4096, "kv": 2048,
         "f": 2112, "layers": 30, **AFFINE64},
        # the routed experts of one decoded token: the headline path
        {"name": "decode_token", "kind": "decode", "router": "bf16", "layers": 8, **GEMMA, **SYM32},
        # the default formats: INT8-affine router, affine group-64 experts
        {"name": "decode_int8_affine", "kind": "decode", "router": "int8", "layers": 8, **GEMMA,
         **AFFINE64},
        # a speculative block: four drafted tokens and the one before them
        {"name": "verify_block5", "kind": "verify", "rows": 5, "share": 0.9, "layers": 8, **GEMMA,
         **SYM32},
        # a short prompt of a chat turn: few rows for each expert
        {"name": "prefill_67", "kind": "prefill", "rows": 67, "share": 0.5, **GEMMA, **SYM32},
        # a medium prompt, in the default format
        {"name": "prefill_509_affine", "kind": "prefill", "rows": 509, "share": 0.5, **GEMMA,
         **AFFINE64},
        # a whole prompt chunk, and the longest with the many small experts
        {"name": "prefill_2048", "kind": "prefill", "rows": 2048, "share": 0.5, **GEMMA, **SYM32},
        {"name": "prefill_4096_silu", "kind": "prefill", "rows": 4096, "share": 0.5, **QWEN,
         **SYM32},
        # a dense projection of a short prompt, and of a whole prompt chunk
        {"name": "qmm_67", "kind": "qmm", "rows": 67, "m": 4096, "n": 2816, **SYM32},
        {"name": "qmm_2048_affine", "kind": "qmm", "rows": 2048, "m": 2816, "n": 4096, **AFFINE64},
    ]


def _log_int(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(v / step)) * step))


def draw(rng):
    fmt = dict(rng.choice([SYM32, AFFINE64, {"group": 32, "scheme": "affine"},
                           {"group": 64, "scheme": "sym"}]))
    kind = rng.choice(["qmv", "dense", "decode", "verify", "prefill", "prefill", "qmm", "qmm"])
    if kind == "qmv":
        return {"kind": kind, "rows": rng.randint(1, 8), "m": _log_int(rng, 256, 8192),
                "n": _log_int(rng, 512, 8192, 64), **fmt}
    if kind == "dense":
        return {"kind": kind, "rows": rng.randint(1, 8), "d": _log_int(rng, 1024, 4096, 64),
                "q": _log_int(rng, 1024, 8192, 64), "kv": _log_int(rng, 256, 2048, 64),
                "f": _log_int(rng, 512, 8192, 64), "layers": rng.randint(2, 12), **fmt}
    if kind == "qmm":
        return {"kind": kind, "rows": _log_int(rng, 9, 2048), "m": _log_int(rng, 704, 4096, 64),
                "n": _log_int(rng, 704, 4096, 64), **fmt}
    shape = dict(rng.choice([GEMMA, QWEN, None]) or
                 {"d": rng.randrange(768, 2817, 64), "f": rng.randrange(256, 705, 64),
                  "experts": rng.choice([32, 64, 96, 128]), "act": rng.choice(["gelu", "silu"])})
    if kind == "decode":
        return {"kind": kind, "router": rng.choice(["bf16", "int8"]), "layers": rng.randint(2, 8),
                **shape, **fmt}
    if kind == "verify":
        return {"kind": kind, "rows": rng.randint(2, 8), "share": rng.choice([0.8, 0.9, 0.95]),
                "layers": rng.randint(2, 8), **shape, **fmt}
    return {"kind": kind, "rows": _log_int(rng, 9, 2048), "share": rng.choice([0.3, 0.5, 0.7]),
            **shape, **fmt}


# ------------------------------------------------------------------- inputs

class _Random:
    """Draws on the GPU from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def bytes(self, *shape):
        n = math.prod(shape)
        words = torch.randint(-2**63, 2**63 - 1, ((n + 7) // 8,), generator=self.g,
                              dtype=torch.int64, device="cuda")
        return words.view(torch.uint8)[:n].view(*shape)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.g, device="cuda")

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.g, device="cuda")

    def scales(self, *shape):
        return (self.normal(*shape).abs() * 0.02 / 7.0).bfloat16()

    def biases(self, scales):
        return (-(6.5 + 2.0 * self.uniform(*scales.shape)) * scales.float()).bfloat16()

    def hidden(self, rows, d, share=0.0):
        common = self.normal(1, d) * math.sqrt(share)
        return (common + self.normal(rows, d) * math.sqrt(1.0 - share)).half()


def _projection(r, case, m, n):
    """(packed weights, scales, biases or None) of one [m, n] matrix."""
    s = r.scales(m, n // case["group"])
    return r.bytes(m, n // 2), s, None if case["scheme"] == "sym" else r.biases(s)


def _dense(case, w, s, b):
    """The matrix in float64."""
    q = torch.stack([w & 15, w >> 4], dim=-1).view(w.shape[0], -1).double()
    s = s.double().repeat_interleave(case["group"], dim=1)
    if b is None:
        return (q - 8.0) * s
    return q * s + b.double().repeat_interleave(case["group"], dim=1)


def _blob_layout(case):
    """Byte offsets of gate, up and down (weights, scales, biases) in an expert
    blob, and the stride of the experts."""
    d, f, g = case["d"], case["f"], case["group"]
    offs, at = [], 0
    for m, n in ((f, d), (f, d), (d, f)):
        w, s = m * n // 2, m * (n // g) * 2
        biased = case["scheme"] != "sym"
        offs += [at, at + w, at + w + s if biased else at + w]
        at += w + s * (2 if biased else 1)
    return offs, -(-at // 16384) * 16384, at


def _expert_layer(r, case):
    """One layer's experts [experts, stride] as they lie in HBM."""
    offs, stride, _ = _blob_layout(case)
    d, f, g, e = case["d"], case["f"], case["group"], case["experts"]
    image = r.bytes(e, stride)
    for j, (m, n) in enumerate(((f, d), (f, d), (d, f))):
        s = r.scales(e, m * (n // g))
        at = offs[3 * j + 1]
        image[:, at:at + 2 * s.shape[1]] = s.view(torch.uint8)
        if case["scheme"] != "sym":
            at = offs[3 * j + 2]
            image[:, at:at + 2 * s.shape[1]] = r.biases(s).view(torch.uint8)
    return image


def _expert(case, image, e):
    """Expert e's gate, up and down in float64."""
    offs, _, _ = _blob_layout(case)
    d, f, g = case["d"], case["f"], case["group"]
    out = []
    for j, (m, n) in enumerate(((f, d), (f, d), (d, f))):
        ow, os_, ob = offs[3 * j:3 * j + 3]
        w = image[e, ow:ow + m * n // 2].view(m, n // 2)
        ns = 2 * m * (n // g)
        s = image[e, os_:os_ + ns].view(torch.bfloat16).view(m, n // g)
        b = None
        if case["scheme"] != "sym":
            b = image[e, ob:ob + ns].view(torch.bfloat16).view(m, n // g)
        out.append(_dense(case, w, s, b))
    return out


def _moe_inputs(case, seed):
    """What the MoE kinds' layers are made of, by the seed alone."""
    r = _Random(seed)
    d, e, g = case["d"], case["experts"], case["group"]
    rows, layers = case.get("rows", 1), case.get("layers", 1)
    v = {"images": [_expert_layer(r, case) for _ in range(layers)]}
    if case.get("router") == "int8":
        v["router_q"] = r.bytes(layers, e, d)
        v["router_s"] = (r.uniform(layers, e, d // g) * 0.5 + 0.75).div(74.0 * math.sqrt(d)).bfloat16()
        v["router_b"] = (-127.5 * v["router_s"].float()).bfloat16()
    else:
        v["router_w"] = (r.normal(layers, e, d) / math.sqrt(d)).bfloat16()
    v["effective_scale"] = (1.0 + 0.1 * r.normal(layers, d)).bfloat16()
    v["expert_gain"] = (1.0 + 0.1 * r.normal(layers, e)).bfloat16()
    share = case.get("share", 0.0)
    v["x"] = torch.stack([r.hidden(rows, d, share) for _ in range(layers)])
    # as large as the experts' own output, as a shared expert's output is
    v["residual"] = torch.stack([r.hidden(rows, d) * 0.03 for _ in range(layers)])
    return v


def _context(case):
    return tsg.Context(0, group_size=case["group"], scheme=case["scheme"])


def _buffer(*shape, dtype=torch.float16):
    return torch.zeros(*shape, dtype=dtype, device="cuda")


# ------------------------------------------------------------------ prepare

def prepare(case, seed):
    st = {"kind": case["kind"], "case": case, "ctx": _context(case)}
    kind, rows = case["kind"], case.get("rows", 1)
    if kind in ("qmv", "qmm"):
        r = _Random(seed)
        st["w"], st["s"], st["b"] = _projection(r, case, case["m"], case["n"])
        st["x"] = r.hidden(rows, case["n"])
        st["y"] = _buffer(rows, case["m"])
        st["op"] = (tsg.DequantInt4GEMV if kind == "qmv" else tsg.PrefillInt4QMM)(st["ctx"])
        return st
    if kind == "dense":
        st.update(_dense_inputs(case, seed))
        st["op"], st["mlp"] = tsg.DequantInt4GEMV(st["ctx"]), tsg.SharedExpertInt4(st["ctx"])
        d, q, kv, f, L = case["d"], case["q"], case["kv"], case["f"], case["layers"]
        st["out"] = {"q": _buffer(L, rows, q), "k": _buffer(L, rows, kv), "v": _buffer(L, rows, kv),
                     "o": _buffer(L, rows, d), "mlp": _buffer(L, rows, d)}
        st["scratch"] = [_buffer(rows, f) for _ in range(3)]
        mat = st["mlp"].projection
        st["steps"] = [{"projections": [(m, st["a" if n == "o" else "x"][l], st["out"][n][l])
                                        for n, m in zip("qkvo", mats)],
                        "x": st["x"][l], "y": st["out"]["mlp"][l], "mats": mats[4:],
                        "mlp": (mat(*mats[4], f, d), mat(*mats[5], f, d), mat(*mats[6], d, f))}
                       for l, mats in enumerate(st["mats"])]
        return st
    st.update(_moe_inputs(case, seed))
    d, f, e = case["d"], case["f"], case["experts"]
    offs, stride, _ = _blob_layout(case)
    st["moe"] = tsg.MoE(st["ctx"], router_weight_bits=8 if case.get("router") == "int8" else 16,
                        gate_activation=case["act"])
    st["layers"] = [tsg.ResidentLayer(st["ctx"], e, stride, offs, device_tensor=im)
                    for im in st["images"]]
    L = len(st["layers"])
    st["y"] = _buffer(L, rows, d)
    st["idx"] = _buffer(L, rows, TOP_K, dtype=torch.int32)
    st["wts"] = _buffer(L, rows, TOP_K)
    keys = [k for k in ("router_w", "router_q", "router_s", "router_b", "effective_scale",
                        "expert_gain", "x", "residual", "y", "idx", "wts") if k in st]
    st["steps"] = [{"layer": st["layers"][l], **{k: st[k][l] for k in keys}} for l in range(L)]
    if kind == "decode":
        st["acts"] = _buffer(TOP_K, f)
    if kind == "prefill":
        st["router"] = tsg.PrefillRouter(st["moe"])
        st["group"] = tsg.PrefillGroupedRoutedMoE(st["moe"])
        st["reduce"] = tsg.PrefillMoE(st["ctx"])
        pairs = rows * TOP_K
        st["max_blocks"] = -(-pairs // 128) + e
        st["sorted"] = _buffer(pairs, 4, dtype=torch.int32)
        st["offsets"] = _buffer(e, dtype=torch.int32)
        st["counts"] = _buffer(e, dtype=torch.int32)
        st["blocks"] = _buffer(st["max_blocks"], 4, dtype=torch.int32)
        st["n_blocks"] = _buffer(1, dtype=torch.int32)
        st["scratch"] = _buffer(st["group"].scratch_bytes(rows, TOP_K, e) // 4 + 1,
                                dtype=torch.int32)
        st["act"] = _buffer(pairs, f)
        st["partials"] = _buffer(pairs, d)
    return st


def _dense_inputs(case, seed):
    r = _Random(seed)
    d, q, kv, f, L, rows = (case[k] for k in ("d", "q", "kv", "f", "layers", "rows"))
    shapes = ((q, d), (kv, d), (kv, d), (d, q), (f, d), (f, d), (d, f))
    return {"mats": [[_projection(r, case, m, n) for m, n in shapes] for _ in range(L)],
            "x": torch.stack([r.hidden(rows, d) for _ in range(L)]),
            "a": torch.stack([r.hidden(rows, q) for _ in range(L)])}


# ---------------------------------------------------------------------- run

def run(st):
    return _RUN[st["kind"]](st, st["case"])


def _run_qmv(st, c):
    if c["rows"] == 1:
        st["op"].encode(st["w"], st["s"], st["b"], st["x"], st["y"], c["m"], c["n"])
    else:
        st["op"].encode_rows(st["w"], st["s"], st["b"], st["x"], c["n"], st["y"], c["m"],
                             c["rows"], c["m"], c["n"])
    return st["y"]


def _run_dense(st, c):
    op, mlp, t, d, f = st["op"], st["mlp"], c["rows"], c["d"], c["f"]
    g, u, a = st["scratch"]
    for step in st["steps"]:
        for (w, s, b), x, y in step["projections"]:
            m, n = y.shape[1], x.shape[1]
            if t == 1:
                op.encode(w, s, b, x, y, m, n)
            else:
                op.encode_rows(w, s, b, x, n, y, m, t, m, n)
        if t == 1:
            mlp.encode(step["x"], *step["mlp"], step["y"], g, u, a)
        else:
            gate, up, down = step["mats"]
            op.encode_rows(*gate, step["x"], d, g, f, t, f, d)
            op.encode_rows(*up, step["x"], d, u, f, t, f, d)
            mlp.encode_gelu_mul(g, u, a, t * f)
            op.encode_rows(*down, a, f, step["y"], d, t, d, f)
    return st["out"]


def _run_decode(st, c):
    d, f, e, moe, acts = c["d"], c["f"], c["experts"], st["moe"], st["acts"]
    for s in st["steps"]:
        x = s["x"]
        tail = (x, s["effective_scale"], s["expert_gain"], x, s["residual"], s["y"], s["idx"],
                s["wts"], acts, e, d, f)
        if c["router"] == "int8":
            moe.encode_decode_layer_int8(s["layer"], s["router_q"], s["router_s"], s["router_b"],
                                         *tail)
        else:
            moe.encode_decode_layer(s["layer"], s["router_w"], *tail)
    return {"y": st["y"], "idx": st["idx"], "wts": st["wts"]}


def _run_verify(st, c):
    d, f, e, moe = c["d"], c["f"], c["experts"], st["moe"]
    for s in st["steps"]:
        moe.encode_verify_layer(s["layer"], s["router_w"], s["x"], s["effective_scale"],
                                s["expert_gain"], s["x"], d, s["y"], s["idx"], s["wts"], c["rows"],
                                e, d, f)
    return {"y": st["y"], "idx": st["idx"], "wts": st["wts"]}


def _run_prefill(st, c):
    d, f, e, t, g = c["d"], c["f"], c["experts"], c["rows"], st["group"]
    s = st["steps"][0]
    x, idx, wts = s["x"], s["idx"], s["wts"]
    st["router"].encode_gemma4_bf16(s["router_w"], x, d, s["effective_scale"], s["expert_gain"],
                                    idx, wts, t, e, d)
    g.group_pairs_device(idx, wts, t, TOP_K, e, st["sorted"], st["offsets"], st["counts"],
                         st["blocks"], st["max_blocks"], st["n_blocks"], st["scratch"],
                         tile_rows=128)
    g.encode_gate_up_down(st["layers"][0], x, d, st["sorted"], st["blocks"], st["max_blocks"],
                          st["act"], st["partials"], TOP_K, d, f, n_blocks_device=st["n_blocks"])
    st["reduce"].encode_reduce_token_major(st["partials"], wts, s["y"], t, TOP_K, d)
    return {"y": st["y"], "idx": st["idx"], "wts": st["wts"]}


def _run_qmm(st, c):
    st["op"].encode(st["w"], st["s"], st["b"], st["x"], st["y"], c["rows"], c["m"], c["n"])
    return st["y"]


_RUN = {"qmv": _run_qmv, "dense": _run_dense, "decode": _run_decode, "verify": _run_verify,
        "prefill": _run_prefill, "qmm": _run_qmm}


# --------------------------------------------------------------------- work

def _matrix_bytes(case, m, n):
    return m * n // 2 + 2 * m * (n // case["group"]) * (1 if case["scheme"] == "sym" else 2)


def _routed_experts(case):
    """Mean number of experts that a layer's rows reach, of logits with
    `share` of their variance in common."""
    rng = np.random.default_rng(7)
    rows, e, share = case.get("rows", 1), case["experts"], case.get("share", 0.0)
    reps = max(1, 256 // rows)
    logits = (rng.normal(size=(reps, 1, e)) * math.sqrt(share) +
              rng.normal(size=(reps, rows, e)) * math.sqrt(1.0 - share))
    top = np.argpartition(-logits, TOP_K - 1, axis=2)[:, :, :TOP_K].reshape(reps, -1)
    return float(np.mean([len(set(t.tolist())) for t in top]))


def work(case):
    kind, rows = case["kind"], case.get("rows", 1)
    if kind in ("qmv", "qmm"):
        m, n = case["m"], case["n"]
        return {"bytes": _matrix_bytes(case, m, n) + 2 * rows * (m + n), "flops": 2 * rows * m * n}
    d, L = case["d"], case.get("layers", 1)
    f = case["f"]
    expert = 2 * _matrix_bytes(case, f, d) + _matrix_bytes(case, d, f)
    if kind == "dense":
        q, kv = case["q"], case["kv"]
        size = expert + sum(_matrix_bytes(case, m, n) for m, n in ((q, d), (kv, d), (kv, d), (d, q)))
        return {"bytes": L * (size + 2 * rows * (2 * d + 2 * q + 2 * kv + d)),
                "flops": 2 * L * rows * (2 * q * d + 2 * kv * d + 3 * f * d)}
    e = case["experts"]
    router = e * d + 4 * e * (d // case["group"]) if case.get("router") == "int8" else 2 * e * d
    # the rows once (and a residual in decode), the outputs, ids and weights
    rows_bytes = rows * (4 * d + 6 * TOP_K) + (2 * d if kind == "decode" else 0)
    return {"bytes": L * (_routed_experts(case) * expert + router + 2 * (d + e) + rows_bytes),
            "flops": 2 * L * rows * (TOP_K * 3 * d * f + e * d)}


# ---------------------------------------------------------------- tolerance

def tolerance(case):
    """About four times the distance to float64 that the outputs show: 2.1e-4
    for one fp16 rounding of a 32-bit sum, 4.4e-4 with the fp16 activations
    between two matrices, 5.2e-4 with the fp16 weights and partial rows of the
    prompt's GEMMs."""
    kind = case["kind"]
    if kind in ("qmv", "qmm"):
        return {"rel": 8e-4}
    if kind == "prefill":
        # a tie in the router's 32-bit logits may fall the other way
        return {"rel": 2e-3, "differ": 1e-3}
    return {"rel": 1.8e-3}


# -------------------------------------------------------------------- exact

def _activation(case, g):
    if case.get("act", "gelu") == "silu":
        return g * torch.sigmoid(g)
    return 0.5 * g * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (g + 0.044715 * g ** 3)))


def _exact_routing(case, v, l):
    """Ids [rows, 8] and weights [rows, 8] of layer l in float64."""
    if case.get("router") == "int8":
        g = case["group"]
        w = (v["router_q"][l].double() * v["router_s"][l].double().repeat_interleave(g, dim=1) +
             v["router_b"][l].double().repeat_interleave(g, dim=1))
    else:
        w = v["router_w"][l].double()
    logits = (v["x"][l].double() * v["effective_scale"][l].double()) @ w.t()
    top, ids = torch.sort(logits, dim=1, descending=True, stable=True)
    top, ids = top[:, :TOP_K], ids[:, :TOP_K]
    return ids, torch.softmax(top, dim=1) * v["expert_gain"][l].double()[ids]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("qmv", "qmm"):
        r = _Random(seed)
        mat = _dense(case, *_projection(r, case, case["m"], case["n"]))
        return r.hidden(case["rows"], case["n"]).double() @ mat.t()
    if kind == "dense":
        v = _dense_inputs(case, seed)
        out = {name: [] for name in ("q", "k", "v", "o", "mlp")}
        for l, mats in enumerate(v["mats"]):
            x = v["x"][l].double()
            for name, mat in zip("qkvo", mats):
                row = v["a"][l].double() if name == "o" else x
                out[name].append(row @ _dense(case, *mat).t())
            gate, up, down = (_dense(case, *m) for m in mats[4:])
            out["mlp"].append((_activation(case, x @ gate.t()) * (x @ up.t())) @ down.t())
        return {name: torch.stack(rows) for name, rows in out.items()}
    v = _moe_inputs(case, seed)
    ys, ws = [], []
    for l, image in enumerate(v["images"]):
        ids, w = _exact_routing(case, v, l)
        x = v["x"][l].double()
        y = v["residual"][l].double().clone() if kind == "decode" else torch.zeros_like(x)
        for e in torch.unique(ids).tolist():
            tok, slot = torch.nonzero(ids == e, as_tuple=True)
            gate, up, down = _expert(case, image, e)
            h = _activation(case, x[tok] @ gate.t()) * (x[tok] @ up.t())
            y.index_add_(0, tok, (h @ down.t()) * w[tok, slot, None])
        ys.append(y)
        ws.append(w)
    return {"y": torch.stack(ys), "idx": None, "wts": torch.stack(ws)}
