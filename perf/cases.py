"""The work this framework is used for, as cases that can be prepared, run and checked.

A quantised decoder layer is four Marlin W4A16 projections: QKV, O, gate/up and
the SiLU-gated down projection.  Tensors kept in the rowwise layout (2 to 8
bits) are run one activation row at a time, or over a batch of rows.  A decode
step also looks up one embedding row and runs the narrow b/a projections, and
ends in the vocabulary projection.  The cases call the public entry points:
``neurova_amd.ops.cuda_ops()`` with buffers a program keeps, or the tensor
objects of ``neurova_amd.store``.

``listed()`` holds the sizes of the model this repository is built around;
``draw`` gives others of the same ranges: batches from 1 to 2048 rows, ragged
ones among them, hidden sizes from 1024 to 5120, both scale modes of the Marlin
layout, every bit width, and rows whose code stream ends inside a byte.
"""
from __future__ import annotations

import math

import torch

from neurova_amd.ops import cuda_ops
from neurova_amd.store import LowBitMarlinTensor, LowBitTensor

DEV = "cuda"


def listed():
    attn = dict(hidden=5120, qkv=14336, o_in=6144, inter=17408, group=128)
    gdn = dict(hidden=5120, qkv=16384, o_in=6144, inter=17408, group=128)
    plain = dict(hidden=5120, qkv=7168, o_in=5120, inter=17408, group=128)
    mlp = dict(hidden=5120, inter=17408)
    return [
        # the smallest calls of a decode step: one embedding row of a 4-bit
        # table and the 48-row b and a projections that share one input
        {"name": "embed_and_ba", "kind": "lookup", "vocab": 248320, "cols": 5120, "rows": 48, "bits": 4, "group": 128},
        # one token through an attention layer
        {"name": "decode_layer_m1", "kind": "layer", "m": 1, "api": "ops", **attn},
        # a verification step of three drafted tokens through a linear-attention layer
        {"name": "verify_layer_m3", "kind": "layer", "m": 3, "api": "ops", **gdn},
        # batched decoding: 16 sequences, then 32 with the one-call MLP
        {"name": "decode_layer_m16", "kind": "layer", "m": 16, "api": "ops", **attn},
        {"name": "decode_layer_m32_fused", "kind": "layer", "m": 32, "api": "fused", **plain},
        # a prompt chunk through the tensor objects (which run up to 256 rows as one product)
        {"name": "chunk_layer_m200", "kind": "layer", "m": 200, "api": "store", **attn},
        # a long prompt
        {"name": "prefill_layer_m2048", "kind": "layer", "m": 2048, "api": "ops", **plain},
        # the vocabulary projection of one token
        {"name": "lm_head_m1", "kind": "head", "m": 1, "hidden": 5120, "vocab": 248320},
        # an MLP in the rowwise layout: gate and up as a pair, then down, for one token ...
        {"name": "rowwise_mlp_b3_m1", "kind": "rowwise", "m": 1, "bits": 3, "group": 64, **mlp},
        {"name": "rowwise_mlp_b8_m1", "kind": "rowwise", "m": 1, "bits": 8, "group": 128, **mlp},
        # ... for a decode batch, and for a prompt chunk
        {"name": "rowwise_mlp_b4_m16", "kind": "rowwise", "m": 16, "bits": 4, "group": 128, **mlp},
        {"name": "rowwise_mlp_b2_m384", "kind": "rowwise", "m": 384, "bits": 2, "group": 64, **mlp},
    ]


def _log_int(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    u = rng.random()
    hidden = _log_int(rng, 1024, 5120, 256)
    inter = _log_int(rng, 2048, 17408, 128)
    if u < 0.55:
        m = _log_int(rng, 1, 32) if u < 0.3 else _log_int(rng, 33, 2048)
        api = rng.choice(["ops", "ops", "store" if m <= 256 else "ops", "fused"])
        return {"kind": "layer", "m": m, "api": api, "hidden": hidden, "qkv": _log_int(rng, 1024, 16384, 256),
                "o_in": _log_int(rng, 1024, 6144, 128), "inter": inter, "group": rng.choice([128, 128, 128, 128, -1])}
    if u < 0.92:
        m = 1 if u < 0.73 else _log_int(rng, 2, 384)
        if rng.random() < 0.25:  # rows that end inside a byte or a 32-code unit
            hidden, inter = hidden + rng.randrange(1, 32), inter + rng.randrange(1, 32)
        else:
            inter += 32 * rng.randrange(0, 4) if inter < 17000 else 0
        return {"kind": "rowwise", "m": m, "bits": rng.choice([2, 3, 4, 5, 6, 7, 8]), "group": rng.choice([32, 64, 128, 128]),
                "hidden": hidden, "inter": inter}
    if u < 0.96:
        return {"kind": "head", "m": _log_int(rng, 1, 8), "hidden": hidden, "vocab": _log_int(rng, 32000, 248320, 256) // 256 * 256}
    return {"kind": "lookup", "vocab": _log_int(rng, 32000, 248320), "cols": hidden, "rows": _log_int(rng, 16, 128),
            "bits": rng.choice([4, 8]), "group": rng.choice([64, 128])}


# ------------------------------------------------------------------ inputs ---

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _codes(g, shape, bits):
    """Codes of bell-shaped weights: three standard deviations fill the range."""
    top = 2 ** bits
    v = torch.randn(shape, device=DEV, generator=g, dtype=torch.float16 if bits < 8 else torch.float32)
    return v.mul_(top / 6).add_(top / 2).round_().clamp_(0, top - 1).to(torch.int32)


def _scales(g, shape, bits, k):
    """Group scales that give outputs of about unit size."""
    v = torch.rand(shape, device=DEV, generator=g).add_(0.5)
    return v.mul_(6 / 2 ** bits / math.sqrt(k)).half()


def _marlin(g, k, n, group):
    """qweight int32 [k/16, 2n] of eight codes a word, scales fp16 [groups, n]."""
    q = torch.zeros((k // 16, 2 * n), dtype=torch.int32, device=DEV)
    for i in range(8):
        q |= _codes(g, q.shape, 4) << (4 * i)
    return q, _scales(g, (k // 128 if group == 128 else 1, n), 4, k)


def _rowwise(g, rows, cols, bits, group):
    """qweight uint8 [rows, ceil(cols*bits/8)], scales fp16 [rows, groups]."""
    q = torch.empty((rows, (cols * bits + 7) // 8), dtype=torch.uint8, device=DEV)
    step = max(1, (1 << 25) // cols)
    for r in range(0, rows, step):
        part = q[r:r + step]
        c = _codes(g, (part.shape[0], (cols + 7) // 8, 8), bits).long()
        word = c[..., 0].clone()
        for i in range(1, 8):  # eight codes are `bits` bytes
            word |= c[..., i] << (bits * i)
        by = torch.stack([(word >> (8 * j)) & 255 for j in range(bits)], dim=-1).to(torch.uint8)
        part.copy_(by.reshape(part.shape[0], -1)[:, :part.shape[1]])
    return q, _scales(g, (rows, -(-cols // group)), bits, cols)


def _rows(g, m, k):
    return torch.randn((m, k), device=DEV, generator=g).half()


def _empty(m, n):
    return torch.empty((m, n), dtype=torch.float16, device=DEV)


def _workspace(n):
    return torch.zeros((n // 128 * 16,), dtype=torch.int32, device=DEV)


def prepare(case, seed):
    g = _gen(seed)
    s = {"case": case, "ops": cuda_ops()}
    kind = case["kind"]
    if kind == "layer":
        m, h, it, gr = case["m"], case["hidden"], case["inter"], case["group"]
        shapes = {"qkv": (h, case["qkv"]), "o": (case["o_in"], h), "gate_up": (h, 2 * it), "down": (it, h)}
        w = {name: _marlin(g, k, n, gr) for name, (k, n) in shapes.items()}
        s.update(w=w, x=_rows(g, m, h), attn=_rows(g, m, case["o_in"]), x2=_rows(g, m, h))
        if case["api"] == "store":
            s["t"] = {name: LowBitMarlinTensor(name, *w[name], cols=shapes[name][0], group_size=gr) for name in shapes}
        else:
            s["out"] = {name: _empty(m, n) for name, (_, n) in shapes.items()}
            s["ws"] = _workspace(max(n for _, n in shapes.values()))
            if case["api"] == "fused":
                s["mlp_ws"] = torch.zeros((s["ops"].lowbit_marlin_mlp_fused_workspace_len(m, h, it),), dtype=torch.int32,
                                          device=DEV)
    elif kind == "head":
        s.update(w=_marlin(g, case["hidden"], case["vocab"], 128), x=_rows(g, case["m"], case["hidden"]),
                 out=_empty(case["m"], case["vocab"]), ws=_workspace(case["vocab"]))
    elif kind == "rowwise":
        h, it, b, gr = case["hidden"], case["inter"], case["bits"], case["group"]
        s["t"] = {name: LowBitTensor(name, *_rowwise(g, n, k, b, gr), cols=k, group_size=gr, bits=b)
                  for name, n, k in (("gate", it, h), ("up", it, h), ("down", h, it))}
        s.update(x=_rows(g, case["m"], h), act=_rows(g, case["m"], it))
        if case["m"] == 1:
            s.update(x=s["x"][0].contiguous(), act=s["act"][0].contiguous())
    else:
        cols, b, gr = case["cols"], case["bits"], case["group"]
        s["table"] = LowBitTensor("embed", *_rowwise(g, case["vocab"], cols, b, gr), cols=cols, group_size=gr, bits=b)
        s["b"] = _rowwise(g, case["rows"], cols, b, gr)
        s["a"] = _rowwise(g, case["rows"], cols, b, gr)
        s["x"] = _rows(g, 1, cols)[0].contiguous()
        s["token"] = torch.randint(0, case["vocab"], (1,), device=DEV, generator=g)
    return s


# --------------------------------------------------------------------- run ---

def run(s):
    case, ops = s["case"], s["ops"]
    kind = case["kind"]
    if kind == "layer":
        h, it, gr = case["hidden"], case["inter"], case["group"]
        if case["api"] == "store":
            t = s["t"]
            qkv, o, mixed = t["qkv"].gemm(s["x"]), t["o"].gemm(s["attn"]), t["gate_up"].gemm(s["x2"])
            return {"qkv": qkv, "o": o, "gate_up": mixed, "down": t["down"].gemm_silu_packed(mixed, it)}
        w, out, ws = s["w"], s["out"], s["ws"]
        ops.lowbit_marlin_gemm_out(*w["qkv"], s["x"], out["qkv"], ws, h, gr)
        ops.lowbit_marlin_gemm_out(*w["o"], s["attn"], out["o"], ws, case["o_in"], gr)
        if case["api"] == "fused":
            ops.lowbit_marlin_mlp_fused_out(*w["gate_up"], *w["down"], s["x2"], out["down"], s["mlp_ws"], h, it, gr, gr)
            return {"qkv": out["qkv"], "o": out["o"], "down": out["down"]}
        ops.lowbit_marlin_gemm_out(*w["gate_up"], s["x2"], out["gate_up"], ws, h, gr)
        ops.lowbit_marlin_gemm_silu_packed_out(*w["down"], out["gate_up"], out["down"], ws, it, gr)
        return dict(out)
    if kind == "head":
        ops.lowbit_marlin_gemm_out(*s["w"], s["x"], s["out"], s["ws"], case["hidden"], 128)
        return s["out"]
    if kind == "rowwise":
        t = s["t"]
        if case["m"] == 1:
            gate, up = ops.lowbit_gemv_pair(t["gate"].qweight, t["gate"].scales, t["up"].qweight, t["up"].scales, s["x"],
                                            case["hidden"], case["group"], case["bits"])
            return {"gate": gate, "up": up, "down": t["down"].gemv(s["act"])}
        return {"gate": t["gate"].gemm(s["x"]), "up": t["up"].gemm(s["x"]), "down": t["down"].gemm(s["act"])}
    b, a = ops.lowbit_gemv_pair(*s["b"], *s["a"], s["x"], case["cols"], case["group"], case["bits"])
    return {"row": s["table"].row_dequant(s["token"]), "b": b, "a": a}


# ---------------------------------------------------------- what it has to do ---

def _marlin_work(m, k, n, group):
    return k * n / 2 + (k // 128 if group == 128 else 1) * n * 2 + m * k * 2 + m * n * 2, 2.0 * m * k * n


def _rowwise_work(m, k, n, bits, group):
    return n * math.ceil(k * bits / 8) + n * math.ceil(k / group) * 2 + m * k * 2 + m * n * 2, 2.0 * m * k * n


def work(case):
    kind = case["kind"]
    if kind == "layer":
        m, h, it, gr = case["m"], case["hidden"], case["inter"], case["group"]
        parts = [_marlin_work(m, h, case["qkv"], gr), _marlin_work(m, case["o_in"], h, gr), _marlin_work(m, h, 2 * it, gr),
                 _marlin_work(m, it, h, gr)]
        more = 0 if case["api"] == "fused" else m * it * 2  # the gated product reads [gate | up]
        less = m * 3 * it * 2 if case["api"] == "fused" else 0  # ... which the one-call MLP need not write or read
        return {"bytes": sum(p[0] for p in parts) + more - less, "flops": sum(p[1] for p in parts)}
    if kind == "head":
        b, f = _marlin_work(case["m"], case["hidden"], case["vocab"], 128)
        return {"bytes": b, "flops": f}
    if kind == "rowwise":
        m, h, it, b, gr = (case[k] for k in ("m", "hidden", "inter", "bits", "group"))
        parts = [_rowwise_work(m, h, it, b, gr), _rowwise_work(m, h, it, b, gr), _rowwise_work(m, it, h, b, gr)]
        return {"bytes": sum(p[0] for p in parts) - m * h * 2, "flops": sum(p[1] for p in parts)}  # gate and up share x
    cols, b, gr = case["cols"], case["bits"], case["group"]
    row = _rowwise_work(0, cols, 1, b, gr)[0] + cols * 2
    ba = _rowwise_work(1, cols, case["rows"], b, gr)
    return {"bytes": row + 2 * ba[0] - cols * 2, "flops": 2 * ba[1] + cols}


def tolerance(case):
    # fp16 outputs of fp32 sums: against exact() the 2-norm error measures
    # 2.1e-4 (the rounding of the outputs) and 4.4e-4 for the down projection
    # (the fp16 gate/up outputs and gated activations before it); the largest
    # error is about one fp16 step, 2^-10.
    return {"rel": 1e-3, "max": 4e-3}


# ------------------------------------------------------------------- exact ---

def _marlin_weight(q, s, group):
    """W[k, n] in 64 bits: the format's fp16 weight fp16(q - 8) * s, or with one scale a column its codes q - 8."""
    kb, n2 = q.shape
    n = n2 // 2
    nib = (q.reshape(kb, n // 64, 8, 4, 4, 1) >> torch.arange(0, 32, 4, device=q.device, dtype=torch.int32)) & 15
    # [k/16, chunk, c, pair, j, k odd, half, k high] -> k = 8 high + 2 pair + odd, column = 16 j + 8 half + c
    nib = nib.reshape(kb, n // 64, 8, 4, 4, 2, 2, 2).permute(0, 7, 3, 5, 1, 4, 6, 2).reshape(kb * 16, n)
    w = (nib - 8).half()
    if group == 128:
        sc = s.reshape(-1, n // 64, 8, 8).transpose(2, 3).reshape(-1, n)  # column 8 j + i is stored at 8 i + j
        w = (w.reshape(-1, 128, n) * sc[:, None]).reshape(kb * 16, n)
    return w.double()


def _marlin_exact(x, q, s, group):
    n = q.shape[1] // 2
    out = torch.empty((x.shape[0], n), dtype=torch.float64, device=DEV)
    for c in range(0, n, 8192):
        e = min(n, c + 8192)
        out[:, c:e] = x.double() @ _marlin_weight(q[:, 2 * c:2 * e].contiguous(), s[:, c:e].contiguous(), group)
    if group != 128:
        r = torch.arange(n, device=DEV)
        r32 = r & 31
        out *= s[0][(r - r32) + 8 * ((r32 >> 1) & 3) + ((r32 >> 3) << 1) + (r32 & 1)].double()
    return out


def _rowwise_weight(q, s, cols, bits, group):
    bit = torch.arange(cols, device=DEV) * bits
    at = bit >> 3
    word = q[:, at].int() | (q[:, (at + 1).clamp(max=q.shape[1] - 1)].int() << 8)
    code = ((word >> (bit & 7).int()) & (2 ** bits - 1)) - 2 ** (bits - 1)
    return code.double() * s.double().repeat_interleave(group, dim=1)[:, :cols]


def _rowwise_exact(x, t):
    step = max(1, (1 << 26) // t.cols)
    parts = [_rowwise_weight(t.qweight[r:r + step], t.scales[r:r + step], t.cols, t.bits, t.group_size) @ x.double().reshape(-1, t.cols).T
             for r in range(0, t.rows, step)]
    return torch.cat(parts).T.reshape(x.shape[:-1] + (t.rows,))


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "layer":
        w, gr = s["w"], case["group"]
        mixed = _marlin_exact(s["x2"], *w["gate_up"], gr)
        gate, up = mixed[:, :case["inter"]], mixed[:, case["inter"]:]
        got = {"qkv": _marlin_exact(s["x"], *w["qkv"], gr), "o": _marlin_exact(s["attn"], *w["o"], gr), "gate_up": mixed,
               "down": _marlin_exact(gate * torch.sigmoid(gate) * up, *w["down"], gr)}
        if case["api"] == "fused":
            del got["gate_up"]
        return got
    if kind == "head":
        return _marlin_exact(s["x"], *s["w"], 128)
    if kind == "rowwise":
        return {"gate": _rowwise_exact(s["x"], s["t"]["gate"]), "up": _rowwise_exact(s["x"], s["t"]["up"]),
                "down": _rowwise_exact(s["act"], s["t"]["down"])}
    t = s["table"]
    ba = {name: LowBitTensor(name, *s[name], cols=t.cols, group_size=t.group_size, bits=t.bits) for name in ("b", "a")}
    row = int(s["token"])
    return {"row": _rowwise_weight(t.qweight[row:row + 1], t.scales[row:row + 1], t.cols, t.bits, t.group_size)[0],
            "b": _rowwise_exact(s["x"], ba["b"]), "a": _rowwise_exact(s["x"], ba["a"])}
