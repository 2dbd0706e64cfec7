"""The work whose speed counts, as a program that serves the decoder with this library issues it.

Shapes are the ones of the library's layer classes, tests and benchmark: d_model 2048, GDN layers of 16 key and
32 value heads of 128 (8192 convolution channels), attention layers of 16 query and 2 KV heads of 256, MoE layers of
256 experts (8 picked, 512 wide) with a shared expert, a vocabulary of 248320, Q4_K and Q6_K weights. What varies is
what varies in use: the number of tokens of a prompt (from a handful to thousands, rarely a round number), the
position in the context, the weight type and the width of the shared expert.

Kinds of a case:
  gdn_decode, attn_decode, moe_decode   one token through `layers` layers of one kind (norm, layer, residual), captured
                                        once in a HIP graph as a serving loop does, and replayed for each token
  token                                 one token from its id to its logits: embedding row, three GDN layers and one
                                        attention layer, each followed by a MoE layer, final norm, LM head
  gdn_prompt                            `rows` prompt tokens through a GDN layer in one pass
  attn_prompt                           the attention layer's input side for `rows` prompt tokens: the three
                                        projections in one call, query / gate split, Q/K norm and rotation
  rows_f32                              the elementwise and reduction kernels over `rows` tokens, fp32
  rows_bf16                             the residual norm and the expert activations over `rows` tokens, bf16
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path.cwd() / "qwen-3.5-cuda_amd"))

from qwen35_hip import ops  # noqa: E402
from qwen35_hip.decode_layers import AttnLayerDecode, GdnLayerDecode, MoeLayerDecode  # noqa: E402

DM, VOCAB, EPS, THETA, ROPE = 2048, 248320, 1e-6, 1e7, 64
HK, HV, DK, DV = 16, 32, 128, 128
KD, VD = HK * DK, HV * DV
CD = 2 * KD + VD
QH, KVH, HD = 16, 2, 256
E, TOPK, INTER = 256, 8, 512
DEV = "cuda"
F32, F64, BF16 = torch.float32, torch.float64, torch.bfloat16
BLOCK = {"Q4_K": 144, "Q6_K": 210}


# ---------------------------------------------------------------- which cases
def listed():
    return [
        # a chat turn's decode: every generated token crosses each kind of layer
        {"name": "gdn_decode", "kind": "gdn_decode", "layers": 4, "wtype": "Q4_K"},
        {"name": "attn_decode", "kind": "attn_decode", "layers": 4, "pos": 2047, "wtype": "Q4_K"},
        {"name": "moe_decode", "kind": "moe_decode", "layers": 4, "shared": 2048, "wtype": "Q4_K"},
        # late in a long context, where the KV cache is the traffic
        {"name": "attn_decode_long", "kind": "attn_decode", "layers": 1, "pos": 30010, "wtype": "Q4_K"},
        # a whole token with its logits, small shared expert
        {"name": "token", "kind": "token", "pos": 700, "shared": 512, "wtype": "Q4_K"},
        # prompts: a few words added to a cached conversation, a question, a page with Q6_K weights, a document
        {"name": "gdn_prompt_9", "kind": "gdn_prompt", "rows": 9, "wtype": "Q4_K"},
        {"name": "gdn_prompt_77", "kind": "gdn_prompt", "rows": 77, "wtype": "Q4_K"},
        {"name": "gdn_prompt_777_q6", "kind": "gdn_prompt", "rows": 777, "wtype": "Q6_K"},
        {"name": "gdn_prompt_4096", "kind": "gdn_prompt", "rows": 4096, "wtype": "Q4_K"},
        # the attention layer's projections of a short prompt
        {"name": "attn_prompt_300", "kind": "attn_prompt", "rows": 300, "wtype": "Q4_K"},
        # the fused per-token kernels over a document (fp32) and over a page (bf16)
        {"name": "rows_f32_4096", "kind": "rows_f32", "rows": 4096},
        {"name": "rows_bf16_1500", "kind": "rows_bf16", "rows": 1500},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gdn_decode", "attn_decode", "moe_decode", "token"] + 2 * ["gdn_prompt", "attn_prompt"] +
                      ["gdn_prompt", "rows_f32", "rows_bf16"])
    wtype = rng.choice(["Q4_K", "Q4_K", "Q6_K"])
    if kind == "gdn_decode":
        return {"kind": kind, "layers": rng.choice([1, 2, 3, 5, 6, 7, 8]), "wtype": wtype}
    if kind == "attn_decode":
        pos = _log_int(rng, 8, 32000)
        return {"kind": kind, "layers": 1 if pos > 8000 else rng.randint(1, 4), "pos": pos, "wtype": wtype}
    if kind == "moe_decode":
        return {"kind": kind, "layers": rng.randint(1, 3), "shared": rng.choice([512, 2048]), "wtype": wtype}
    if kind == "token":
        return {"kind": kind, "pos": _log_int(rng, 8, 4000), "shared": rng.choice([512, 2048]), "wtype": "Q4_K"}
    if kind == "gdn_prompt":
        return {"kind": kind, "rows": _log_int(rng, 2, 4096 if wtype == "Q4_K" else 3000), "wtype": wtype}
    if kind == "attn_prompt":
        return {"kind": kind, "rows": _log_int(rng, 2, 4096 if wtype == "Q4_K" else 3000), "wtype": wtype}
    return {"kind": kind, "rows": _log_int(rng, 1, 4096)}


# ---------------------------------------------------------------- inputs
class _Rng:
    """Tensors on the GPU from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed) * 1000003 + 12345)

    def normal(self, *shape, mu=0.0, sigma=1.0, dtype=F32):
        return (mu + sigma * torch.randn(shape, generator=self.g, device=DEV)).to(dtype)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return lo + (hi - lo) * torch.rand(shape, generator=self.g, device=DEV)

    def ints(self, lo, hi, *shape, dtype=torch.int32):
        return torch.randint(lo, hi, shape, generator=self.g, device=DEV, dtype=dtype)

    def weight(self, wtype, rows, cols):
        """A quantized [rows x cols] matrix as a file holds it: GGML blocks whose values are spread around zero with
        standard deviation 1 / sqrt(cols)."""
        nb = rows * cols // 256
        std = 1.0 / math.sqrt(cols)
        b = self.ints(0, 256, nb, BLOCK[wtype], dtype=torch.uint8)
        spread = self.uniform(nb, lo=0.7, hi=1.3)
        if wtype == "Q6_K":   # (d sc) (q - 32), scales of either sign
            sc = self.ints(32, 128, nb, 16, dtype=torch.int16) * (1 - 2 * self.ints(0, 2, nb, 16, dtype=torch.int16))
            b[:, 192:208] = sc.to(torch.int8).view(torch.uint8)
            b[:, 208:210] = (spread * (std / 1530.0)).to(torch.float16).view(torch.uint8).view(nb, 2)
            return b.view(-1)
        # (d sc) q - dmin m with m near sc and dmin = 7.5 d, so that the middle of 0..15 is near zero
        sc = self.ints(24, 64, nb, 8, dtype=torch.uint8)
        mn = (sc.to(torch.int16) + self.ints(-4, 5, nb, 8, dtype=torch.int16)).clamp_(0, 63).to(torch.uint8)
        b[:, 4:8] = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
        b[:, 8:12] = mn[:, :4] | ((mn[:, 4:] >> 4) << 6)
        b[:, 12:16] = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
        d = spread * (std / 209.0)
        b[:, 0:2] = d.to(torch.float16).view(torch.uint8).view(nb, 2)
        b[:, 2:4] = (7.5 * d).to(torch.float16).view(torch.uint8).view(nb, 2)
        return b.view(-1)


def _norm_w(r, n):
    return r.normal(n, mu=1.0, sigma=0.1)


def _gdn_tensors(r, wtype):
    return {"qkv": r.weight(wtype, CD, DM), "z": r.weight(wtype, VD, DM), "beta": r.weight(wtype, HV, DM),
            "alpha": r.weight(wtype, HV, DM), "out": r.weight(wtype, DM, VD), "conv": r.normal(CD, 4, sigma=0.5),
            "a": -torch.exp(r.normal(HV)), "dt": r.uniform(HV, lo=-1.0, hi=1.0), "norm": _norm_w(r, DV),
            "history": r.normal(CD, 3), "state": r.normal(HV, DK, DV, sigma=0.1)}


def _attn_tensors(r, wtype, pos):
    return {"qg": r.weight(wtype, 2 * QH * HD, DM), "k": r.weight(wtype, KVH * HD, DM),
            "v": r.weight(wtype, KVH * HD, DM), "out": r.weight(wtype, DM, QH * HD), "qn": _norm_w(r, HD),
            "kn": _norm_w(r, HD), "keys": r.normal(pos, KVH * HD), "values": r.normal(pos, KVH * HD)}


def _moe_tensors(r, wtype, shared):
    return {"router": r.weight(wtype, E, DM), "gate": r.weight(wtype, E * INTER, DM),
            "up": r.weight(wtype, E * INTER, DM), "down": r.weight(wtype, E * DM, INTER),
            "sgate": r.weight(wtype, 1, DM), "sg": r.weight(wtype, shared, DM), "su": r.weight(wtype, shared, DM),
            "sd": r.weight(wtype, DM, shared)}


def _layer_kinds(case):
    if case["kind"] == "token":
        return ["gdn", "moe"] * 3 + ["attn", "moe"]
    return [case["kind"].split("_")[0]] * case["layers"]


def _decode_inputs(case, seed):
    r = _Rng(seed)
    make = {"gdn": lambda: _gdn_tensors(r, case["wtype"]), "attn": lambda: _attn_tensors(r, case["wtype"], case["pos"]),
            "moe": lambda: _moe_tensors(r, case["wtype"], case["shared"])}
    t = {"layers": [(k, make[k](), _norm_w(r, DM)) for k in _layer_kinds(case)]}
    if case["kind"] == "token":
        t["embed"] = r.weight("Q4_K", VOCAB, DM)
        t["head"] = r.weight("Q6_K", VOCAB, DM)
        t["norm"] = _norm_w(r, DM)
        t["id"] = r.ints(0, VOCAB, 1)
    else:
        t["x"] = r.normal(1, DM)
    return t


def _prompt_inputs(case, seed):
    r = _Rng(seed)
    xs = r.normal(case["rows"], DM)   # the layer's normed input
    if case["kind"] == "gdn_prompt":
        return {"xs": xs, **_gdn_tensors(r, case["wtype"])}
    return {"xs": xs, **_attn_tensors(r, case["wtype"], 0)}


def _rows_inputs(case, seed):
    r, n = _Rng(seed), case["rows"]
    if case["kind"] == "rows_bf16":
        return {"x": r.normal(n, DM, dtype=BF16), "branch": r.normal(n, DM, dtype=BF16), "w": _norm_w(r, DM),
                "g": r.normal(n, TOPK, INTER, sigma=2.0, dtype=BF16),
                "u": r.normal(n, TOPK, INTER, sigma=2.0, dtype=BF16),
                "sg": r.normal(n, INTER, sigma=2.0, dtype=BF16), "su": r.normal(n, INTER, sigma=2.0, dtype=BF16),
                "logits": r.normal(n)}
    return {"q4": r.weight("Q4_K", 65536, DM), "q6": r.weight("Q6_K", 65536, DM), "ids": r.ints(0, 65536, n),
            "x": r.normal(n, DM), "w": _norm_w(r, DM), "q": r.normal(n, QH, HD), "k": r.normal(n, KVH, HD),
            "qn": _norm_w(r, HD), "kn": _norm_w(r, HD), "pos": torch.arange(n, dtype=torch.int32, device=DEV) + 17,
            "qkv": r.normal(n, CD), "conv": r.normal(CD, 4, sigma=0.5), "history": r.normal(CD, 3),
            "core": r.normal(n, HV, DV), "z": r.normal(n, HV, DV), "norm": _norm_w(r, DV), "router": r.normal(n, E),
            "experts": r.normal(n, TOPK, DM), "acc": r.normal(n, DM)}


# ---------------------------------------------------------------- the calls
def _gdn_layer(t, wtype):
    layer = GdnLayerDecode(t["qkv"], t["z"], t["beta"], t["alpha"], t["out"], t["conv"], t["a"], t["dt"], t["norm"],
                           wtype=wtype)
    layer.history.copy_(t["history"])
    layer.state.copy_(t["state"])
    return layer


def _attn_layer(t, wtype, pos):
    layer = AttnLayerDecode(t["qg"], t["k"], t["v"], t["out"], t["qn"], t["kn"], wtype=wtype,
                            max_seq_len=max(64, pos + 1))
    layer.k_cache[:pos].copy_(t["keys"])
    layer.v_cache[:pos].copy_(t["values"])
    return layer


def _moe_layer(t, wtype, shared):
    return MoeLayerDecode(t["router"], t["gate"], t["up"], t["down"], t["sgate"], t["sg"], t["su"], t["sd"],
                          wtype=wtype, shared=shared)


def _decode_token(s):
    """One token through the layers: rows of [1 x d_model], every buffer kept between tokens."""
    x, pos = s["token"], s["pos"]
    if s["embed"] is not None:
        ops.dequant_gather_rows(s["embed"], "Q4_K", VOCAB * DM, s["id"], DM, out=x)
    for i, (kind, layer, norm_w) in enumerate(s["layers"]):
        if i == 0:
            ops.rmsnorm_rows(x, norm_w, out=s["normed"], eps=EPS)
        else:
            x, _ = ops.residual_rmsnorm_rows(x, s["branch"], norm_w, resid=s["x"][i & 1], normed=s["normed"], eps=EPS)
        if kind == "attn":
            layer.forward(s["normed"].view(-1), pos, s["branch"].view(-1))
        else:
            layer.forward(s["normed"].view(-1), s["branch"].view(-1))
    if s["head"] is None:
        ops.residual_add(x, s["branch"], out=s["out"])
        return
    ops.residual_rmsnorm_rows(x, s["branch"], s["norm"], resid=s["out"], normed=s["normed"], eps=EPS)
    ops.matmul_dispatch(s["head"], "Q6_K", VOCAB * DM, s["normed"].view(-1), VOCAB, DM, out=s["logits"])


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("rows_f32", "rows_bf16"):
        return {"kind": kind, **_rows_inputs(case, seed)}
    if kind == "gdn_prompt":
        t = _prompt_inputs(case, seed)
        return {"kind": kind, "xs": t["xs"], "layer": _gdn_layer(t, case["wtype"])}
    if kind == "attn_prompt":
        t = _prompt_inputs(case, seed)
        return {"kind": kind, "wtype": case["wtype"], **t}

    t = _decode_inputs(case, seed)
    wtype, pos = case["wtype"], case.get("pos", 0)
    build = {"gdn": lambda w: _gdn_layer(w, wtype), "attn": lambda w: _attn_layer(w, wtype, pos),
             "moe": lambda w: _moe_layer(w, wtype, case["shared"])}
    layers = [(k, build[k](w), n) for k, w, n in t["layers"]]
    token = torch.zeros(1, DM, device=DEV) if kind == "token" else t["x"]
    s = {"kind": kind, "layers": layers, "pos": pos, "embed": t.get("embed"), "head": t.get("head"), "id": t.get("id"),
         "norm": t.get("norm"), "token": token, "x": torch.empty(2, 1, DM, device=DEV),
         "normed": torch.empty(1, DM, device=DEV), "branch": torch.empty(1, DM, device=DEV),
         "out": torch.empty(1, DM, device=DEV),
         "logits": torch.empty(VOCAB, device=DEV) if kind == "token" else None, "parity": 0}
    # A GDN layer's history alternates between two buffers, so a serving loop holds one graph per parity. The first two,
    # uncaptured tokens load the kernels; the layers' state is set back after them.
    _decode_token(s)
    _decode_token(s)
    s["graphs"] = []
    torch.cuda.synchronize()
    for _ in range(2):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            _decode_token(s)
        s["graphs"].append(g)
    for (k, layer, _), (_, w, _) in zip(layers, t["layers"]):
        if k == "gdn":
            layer.history.copy_(w["history"])
            layer.state.copy_(w["state"])
            w["history"] = w["state"] = None
        elif k == "attn":
            w["keys"] = w["values"] = None
    return s


def run(s):
    kind = s["kind"]
    if kind == "rows_bf16":
        resid, normed = ops.residual_rmsnorm_rows(s["x"], s["branch"], s["w"], eps=EPS)
        act, shared = ops.swiglu_routed_shared_bf16(s["g"], s["u"], s["sg"], s["su"], s["logits"])
        return {"resid": resid, "normed": normed, "act": act, "shared": shared}
    if kind == "rows_f32":
        e4 = ops.dequant_gather_rows(s["q4"], "Q4_K", 65536 * DM, s["ids"], DM)
        e6 = ops.dequant_gather_rows(s["q6"], "Q6_K", 65536 * DM, s["ids"], DM)
        normed = ops.rmsnorm_rows(s["x"], s["w"], eps=EPS)
        q, k = s["q"].clone(), s["k"].clone()   # normed and rotated in place
        ops.attn_qk_norm_rope_rows(q, k, s["qn"], s["kn"], pos=s["pos"], rope_dim=ROPE, theta=THETA, eps=EPS)
        conv, history = ops.gdn_frontend_rows(s["qkv"], s["conv"], s["history"], k_heads=HK, key_dim=DK, eps=EPS)
        gated = ops.gdn_norm_gate_rows(s["core"], s["z"], s["norm"], eps=EPS)
        idx, w = ops.moe_topk_rows(s["router"], TOPK)
        acc = ops.moe_weighted_sum_rows(s["acc"].clone(), s["experts"], w)
        return {"e4": e4, "e6": e6, "normed": normed, "q": q, "k": k, "conv": conv, "history": history, "gated": gated,
                "idx": idx, "w": w, "acc": acc}
    if kind == "gdn_prompt":
        out = s["layer"].prefill(s["xs"])
        return {"out": out, "state": s["layer"].state, "history": s["layer"].history}
    if kind == "attn_prompt":
        rows, t = s["xs"].shape[0], s["wtype"]
        qg, k, v = ops.matmul_rows_multi([(s["qg"], t, 2 * QH * HD * DM, 2 * QH * HD, 0, None),
                                          (s["k"], t, KVH * HD * DM, KVH * HD, 0, None),
                                          (s["v"], t, KVH * HD * DM, KVH * HD, 0, None)], s["xs"], DM)
        q, g = ops.attn_split_qg(qg, rows * QH, HD)
        q, k = ops.attn_qk_norm_rope_rows(q.view(rows, QH, HD), k.view(rows, KVH, HD), s["qn"], s["kn"],
                                          rope_dim=ROPE, theta=THETA, eps=EPS)
        return {"q": q, "gate": g, "k": k, "v": v}
    s["graphs"][s["parity"]].replay()
    s["parity"] ^= 1
    states = {}
    for i, (k, layer, _) in enumerate(s["layers"]):
        if k == "gdn":
            history = layer._history_next if s["parity"] else layer.history
            states[f"state{i}"], states[f"history{i}"] = layer.state, history
        elif k == "attn":
            states[f"key{i}"], states[f"value{i}"] = layer.k_cache[s["pos"]], layer.v_cache[s["pos"]]
    if kind == "token":
        states["logits"] = s["logits"]
    return {"out": s["out"], **states}


# ---------------------------------------------------------------- what a pass cannot do without
def _wbytes(wtype, rows, cols):
    return rows * cols // 256 * BLOCK[wtype]


def _gdn_work(wtype, rows):
    m = CD + VD + 2 * HV
    b = _wbytes(wtype, m, DM) + _wbytes(wtype, DM, VD) + 4 * (CD * 4 + 2 * CD * 3 + 2 * HV * DK * DV + 2 * rows * DM)
    return b, rows * (2 * m * DM + 2 * DM * VD + 6 * HV * DK * DV + 8 * CD)


def _attn_work(wtype, pos):
    m = 2 * QH * HD + 2 * KVH * HD
    b = _wbytes(wtype, m, DM) + _wbytes(wtype, DM, QH * HD) + 2 * (pos + 1) * KVH * HD * 4
    return b, 2 * m * DM + 2 * DM * QH * HD + 4 * QH * HD * (pos + 1)


def _moe_work(wtype, shared):
    m = E + 1 + TOPK * 2 * INTER + 2 * shared
    b = _wbytes(wtype, m, DM) + TOPK * _wbytes(wtype, DM, INTER) + _wbytes(wtype, DM, shared)
    return b, 2 * m * DM + 2 * DM * (TOPK * INTER + shared)


def work(case):
    kind, n = case["kind"], case.get("rows", 1)
    if kind == "gdn_prompt":
        b, f = _gdn_work(case["wtype"], n)
        return {"bytes": b, "flops": f}
    if kind == "attn_prompt":
        m = 2 * QH * HD + 2 * KVH * HD
        return {"bytes": _wbytes(case["wtype"], m, DM) + 4 * n * (DM + m), "flops": 2 * n * m * DM}
    if kind == "rows_bf16":
        return {"bytes": n * (4 * DM * 2 + 3 * (TOPK + 1) * INTER * 2 + 4), "flops": n * (5 * DM + 6 * TOPK * INTER)}
    if kind == "rows_f32":
        b = (_wbytes("Q4_K", n, DM) + _wbytes("Q6_K", n, DM) + 8 * n * DM + 8 * n * DM + 8 * n * (QH + KVH) * HD +
             8 * n * CD + 4 * CD * (4 + 6) + 12 * n * VD + 4 * n * (E + 2 * TOPK) + 4 * n * (TOPK + 2) * DM)
        return {"bytes": b, "flops": n * (4 * DM + 10 * (QH + KVH) * HD + 15 * CD + 10 * VD + 2 * TOPK * DM)}
    b = f = 0
    for k in _layer_kinds(case):
        lb, lf = (_gdn_work(case["wtype"], 1) if k == "gdn" else _attn_work(case["wtype"], case["pos"]) if k == "attn"
                  else _moe_work(case["wtype"], case["shared"]))
        b, f = b + lb, f + lf
    if kind == "token":
        b, f = b + _wbytes("Q6_K", VOCAB, DM) + 4 * VOCAB, f + 2 * VOCAB * DM
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times the error against exact(): 1.7e-3 for bf16 results, 7e-8 for the fp32 row kernels, up to 9e-7
    for fp32 sums through a layer's projections, recurrence or attention."""
    kind = case["kind"]
    if kind == "rows_bf16":
        return {"rel": 7e-3, "max": 2e-2}
    if kind == "rows_f32":
        return {"rel": 5e-7, "max": 5e-5}
    return {"rel": 4e-6, "max": 2e-4}


# ---------------------------------------------------------------- the same in 64 bits, from torch alone
def _half(b):
    return b.contiguous().view(torch.float16).to(F64)


def _dequant(w, wtype, rows, cols):
    """[rows x cols] float64 of GGML blocks (rows x cols / 256 of them)."""
    b = w.view(-1, BLOCK[wtype])
    nb = b.shape[0]
    if wtype == "Q4_K":
        d, dmin = _half(b[:, 0:2]), _half(b[:, 2:4])
        s = b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).to(F64)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).to(F64)
        q = b[:, 16:].view(nb, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).view(nb, 8, 32).to(F64)
        return ((d * sc).unsqueeze(2) * q - (dmin * mn).unsqueeze(2)).view(rows, cols)
    ql, qh = b[:, :128].view(nb, 2, 64), b[:, 128:192].view(nb, 2, 32)
    lo = torch.stack([ql[:, :, :32] & 15, ql[:, :, 32:] & 15, ql[:, :, :32] >> 4, ql[:, :, 32:] >> 4], 2)
    hi = torch.stack([(qh >> (2 * k)) & 3 for k in range(4)], 2)
    q = (lo | (hi << 4)).to(F64) - 32.0
    sc = b[:, 192:208].contiguous().view(torch.int8).to(F64) * _half(b[:, 208:210])
    return (q.view(nb, 16, 16) * sc.unsqueeze(2)).view(rows, cols)


def _mm(x, w, wtype, rows, cols, step=16384):
    """x [n x cols] times the transpose of the quantized [rows x cols] matrix, float64."""
    size = cols // 256 * BLOCK[wtype]
    return torch.cat([x @ _dequant(w[r * size:min(r + step, rows) * size], wtype, min(step, rows - r), cols).t()
                      for r in range(0, rows, step)], 1)


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.to(F64)


def _silu(x):
    return x * torch.sigmoid(x)


def _rope(x, pos):
    """x [n, heads, dim] rotated at pos [n] (split halves of the first ROPE dims). The angle is defined in 32 bits:
    pos over the rounded power of theta, rounded."""
    den = torch.tensor([THETA ** (2.0 * i / ROPE) for i in range(ROPE // 2)], dtype=F64).to(F32).to(x.device)
    a = (pos.to(F32)[:, None] / den).to(F64)[:, None, :]
    c, s = a.cos(), a.sin()
    u, v = x[..., :ROPE // 2], x[..., ROPE // 2:ROPE]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., ROPE:]], -1)


def _front(qkv, conv_w, history):
    """Depthwise convolution with the carried history, SiLU, L2 norms of the q and k heads."""
    n = qkv.shape[0]
    ext = torch.cat([history.to(F64).t(), qkv], 0)
    y = _silu(sum(ext[j:j + n] * conv_w[:, j].to(F64) for j in range(4)))
    q, k = y[:, :KD].view(n, HK, DK), y[:, KD:2 * KD].view(n, HK, DK)
    q = q * torch.rsqrt((q * q).sum(-1, keepdim=True) + EPS) / math.sqrt(DK)
    k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + EPS)
    return torch.cat([q.reshape(n, KD), k.reshape(n, KD), y[:, 2 * KD:]], 1), ext[n:].t().contiguous()


def _gdn_exact(xs, t, wtype):
    n = xs.shape[0]
    qkv, z = _mm(xs, t["qkv"], wtype, CD, DM), _mm(xs, t["z"], wtype, VD, DM)
    beta = torch.sigmoid(_mm(xs, t["beta"], wtype, HV, DM))
    sp = torch.nn.functional.softplus(_mm(xs, t["alpha"], wtype, HV, DM) + t["dt"].to(F64), threshold=60.0)
    decay = torch.exp(t["a"].to(F64) * sp)
    y, history = _front(qkv, t["conv"], t["history"])
    q = y[:, :KD].view(n, 1, HK, DK).expand(n, HV // HK, HK, DK).reshape(n, HV, 1, DK)
    k = y[:, KD:2 * KD].view(n, 1, HK, DK).expand(n, HV // HK, HK, DK).reshape(n, HV, 1, DK)
    v = y[:, 2 * KD:].view(n, HV, 1, DV)
    S, core = t["state"].to(F64), torch.empty(n, HV, 1, DV, dtype=F64, device=xs.device)
    for i in range(n):
        S = S * decay[i][:, None, None]
        S = torch.baddbmm(S, k[i].transpose(1, 2).contiguous(), (v[i] - torch.bmm(k[i], S)) * beta[i][:, None, None])
        core[i] = torch.bmm(q[i], S)
    normed = _rms(core.view(n, HV, DV), t["norm"]) * _silu(z.view(n, HV, DV))
    return _mm(normed.reshape(n, VD), t["out"], wtype, DM, VD), S, history


def _attn_exact(x, t, wtype, pos):
    at = torch.tensor([pos], device=x.device)
    qg = _mm(x, t["qg"], wtype, 2 * QH * HD, DM).view(QH, 2, HD)
    k = _rope(_rms(_mm(x, t["k"], wtype, KVH * HD, DM).view(1, KVH, HD), t["kn"]), at)
    v = _mm(x, t["v"], wtype, KVH * HD, DM)
    q = _rope(_rms(qg[:, 0].view(1, QH, HD), t["qn"]), at).view(KVH, QH // KVH, HD)
    keys = torch.cat([t["keys"].to(F64), k.view(1, -1)], 0).view(-1, KVH, HD)
    vals = torch.cat([t["values"].to(F64), v], 0).view(-1, KVH, HD)
    p = torch.softmax(torch.bmm(q, keys.permute(1, 2, 0).contiguous()) / math.sqrt(HD), -1)
    o = torch.bmm(p, vals.transpose(0, 1).contiguous()).view(QH, HD) * torch.sigmoid(qg[:, 1])
    return _mm(o.view(1, -1), t["out"], wtype, DM, QH * HD), k.view(-1), v.view(-1)


def _moe_exact(x, t, wtype, shared):
    top = torch.topk(_mm(x, t["router"], wtype, E, DM).view(-1), TOPK)
    w, ids = torch.softmax(top.values, 0), top.indices.tolist()
    out = torch.zeros(1, DM, dtype=F64, device=x.device)
    size = INTER * DM // 256 * BLOCK[wtype]
    for j, e in enumerate(ids):
        gate, up, down = (t[n][e * size:(e + 1) * size] for n in ("gate", "up", "down"))
        h = _silu(_mm(x, gate, wtype, INTER, DM)) * _mm(x, up, wtype, INTER, DM)
        out = out + w[j] * _mm(h, down, wtype, DM, INTER)
    h = _silu(_mm(x, t["sg"], wtype, shared, DM)) * _mm(x, t["su"], wtype, shared, DM)
    return out + torch.sigmoid(_mm(x, t["sgate"], wtype, 1, DM)) * _mm(h, t["sd"], wtype, DM, shared)


def exact(case, seed):
    kind = case["kind"]
    if kind == "rows_bf16":
        t = _rows_inputs(case, seed)
        resid = (t["x"].to(F64) + t["branch"].to(F64)).to(BF16).to(F64)   # the stored sum is what is normed
        act = _silu(t["g"].to(F64)) * t["u"].to(F64)
        sh = _silu(t["sg"].to(F64)) * t["su"].to(F64) * torch.sigmoid(t["logits"].to(F64))[:, None]
        return {"resid": resid, "normed": _rms(resid, t["w"]), "act": act, "shared": sh}
    if kind == "rows_f32":
        t = _rows_inputs(case, seed)
        n, ids = case["rows"], t["ids"].long()
        row = {w: DM // 256 * BLOCK[w] for w in BLOCK}
        top = torch.topk(t["router"].to(F64), TOPK, -1)
        w = torch.softmax(top.values, -1)
        y, history = _front(t["qkv"].to(F64), t["conv"], t["history"])
        return {"e4": _dequant(t["q4"].view(-1, row["Q4_K"])[ids].contiguous(), "Q4_K", n, DM),
                "e6": _dequant(t["q6"].view(-1, row["Q6_K"])[ids].contiguous(), "Q6_K", n, DM),
                "normed": _rms(t["x"].to(F64), t["w"]), "q": _rope(_rms(t["q"].to(F64), t["qn"]), t["pos"]),
                "k": _rope(_rms(t["k"].to(F64), t["kn"]), t["pos"]), "conv": y, "history": history,
                "gated": _rms(t["core"].to(F64), t["norm"]) * _silu(t["z"].to(F64)), "idx": None, "w": w,
                "acc": t["acc"].to(F64) + (w[:, :, None] * t["experts"].to(F64)).sum(1)}
    if kind == "gdn_prompt":
        t = _prompt_inputs(case, seed)
        out, state, history = _gdn_exact(t["xs"].to(F64), t, case["wtype"])
        return {"out": out, "state": state, "history": history}
    if kind == "attn_prompt":
        t, n, wt = _prompt_inputs(case, seed), case["rows"], case["wtype"]
        xs, at = t["xs"].to(F64), torch.arange(case["rows"], device=DEV)
        qg = _mm(xs, t["qg"], wt, 2 * QH * HD, DM).view(n, QH, 2, HD)
        return {"q": _rope(_rms(qg[:, :, 0], t["qn"]), at), "gate": qg[:, :, 1].reshape(-1),
                "k": _rope(_rms(_mm(xs, t["k"], wt, KVH * HD, DM).view(n, KVH, HD), t["kn"]), at),
                "v": _mm(xs, t["v"], wt, KVH * HD, DM)}

    t, wt = _decode_inputs(case, seed), case["wtype"]
    states = {}
    if kind == "token":
        size, i = DM // 256 * BLOCK["Q4_K"], int(t["id"])
        x = _dequant(t["embed"][i * size:(i + 1) * size], "Q4_K", 1, DM)
    else:
        x = t["x"].to(F64)
    for i, (k, w, norm_w) in enumerate(t["layers"]):
        h = _rms(x, norm_w)
        if k == "gdn":
            h, states[f"state{i}"], states[f"history{i}"] = _gdn_exact(h, w, wt)
        elif k == "attn":
            h, states[f"key{i}"], states[f"value{i}"] = _attn_exact(h, w, wt, case["pos"])
        else:
            h = _moe_exact(h, w, wt, case["shared"])
        x = x + h
    if kind == "token":
        states["logits"] = _mm(_rms(x, t["norm"]), t["head"], "Q6_K", VOCAB, DM).view(-1)
    return {"out": x, **states}
