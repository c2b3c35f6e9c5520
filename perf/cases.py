"""Performance cases of libkai_gdn_hip.so: the work a program gives the
library, through its C entry points.

Kinds (the shapes are the Qwen3.5-4B layer's unless a case says otherwise:
hidden 2560, 16 key and 32 value heads of 128, conv over 8192 channels, 16
query and 4 KV heads of 256, MLP 9216):

  layer_step  one token per sequence through the recurrence half of a GDN
              layer: conv cache update, gating prologue, delta-rule step,
              gated RMSNorm (four calls, as a decode loop makes them)
  chunk       the chunked delta rule over a prompt (prefill of one layer)
  conv        the causal conv with SiLU over a prompt
  scan        the diagonal gated scan (the reference's own recurrence)
  glue        the gating prologue and the gated RMSNorm around a prefill
  matmul      one int8-weight projection, decode rows to prompt rows
  attention   decode attention of one full-attention layer over a KV cache
  model       the whole hybrid model: a prompt, then tokens fed one at a
              time (scoring a given continuation); returns every logit row
"""
from __future__ import annotations

import math

import numpy as np
import torch

import orionsbelt_amd as ob
from orionsbelt_amd import hybrid

D = 128            # GDN head dim
DEV = "cuda"
# (N, K) of the 4B model's projections: GDN in, attention in, out / o, gate|up, down
MATRICES = [(12352, 2560), (10240, 2560), (2560, 4096), (18432, 2560), (2560, 9216)]


def listed():
    return [
        # one user's decode loop, a layer's recurrence at batch 1: latency and launches
        {"name": "layer_step_b1", "kind": "layer_step", "batch": 1, "hk": 16, "hv": 32, "f16": False},
        # a full server batch, fp32 state: the library's headline decode workload
        {"name": "layer_step_b64", "kind": "layer_step", "batch": 64, "hk": 16, "hv": 32, "f16": False},
        # a long prompt through one layer, the gates of the library's benchmark
        {"name": "chunk_16k", "kind": "chunk", "batch": 1, "seq": 16384, "hk": 16, "hv": 32, "gates": "short",
         "f16": False},
        # two documents of ragged length whose heads forget at very different rates
        {"name": "chunk_2x5001_mixed", "kind": "chunk", "batch": 2, "seq": 5001, "hk": 16, "hv": 32,
         "gates": "mixed", "f16": False},
        # a chat turn's prompts, batched, the state kept in fp16
        {"name": "chunk_3x700_f16", "kind": "chunk", "batch": 3, "seq": 700, "hk": 16, "hv": 32, "gates": "short",
         "f16": True},
        # the layer's conv over a 4K prompt: a pure streaming kernel
        {"name": "conv_4096", "kind": "conv", "seq": 4096, "channels": 8192},
        # the reference's scan at an odd length, bf16 state carried
        {"name": "scan_1111_bf16", "kind": "scan", "seq": 1111, "channels": 4096, "state": "bf16"},
        # glue of a 3K-token prompt
        {"name": "glue_3001", "kind": "glue", "rows": 3001, "hk": 16, "hv": 32},
        # the MLP's down projection for a prompt of a few hundred tokens
        {"name": "matmul_down_333", "kind": "matmul", "m": 333, "n": 2560, "k": 9216},
        # a batch of chats deep in their contexts, one attention layer
        {"name": "attention_8x12289", "kind": "attention", "batch": 8, "length": 12289},
        # four chat prompts and eight tokens of each answer
        {"name": "model_chat", "kind": "model", "batch": 4, "prompt": 200, "steps": 8},
        # one long document to its next-token logits
        {"name": "model_document", "kind": "model", "batch": 1, "prompt": 20000, "steps": 0},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer_step", "chunk", "conv", "scan", "glue", "matmul", "attention", "model"])
    heads = rng.choice([(16, 32), (16, 32), (16, 16), (8, 16)])
    if kind == "layer_step":
        return {"kind": kind, "batch": _logint(rng, 1, 96), "hk": heads[0], "hv": heads[1],
                "f16": rng.random() < 0.4}
    if kind == "chunk":
        total = _logint(rng, 60, 16384)
        batch = min(rng.choice([1, 1, 2, 3, 5]), max(1, total // 20))
        return {"kind": kind, "batch": batch, "seq": max(1, total // batch), "hk": heads[0], "hv": heads[1],
                "gates": rng.choice(["short", "mixed", "long"]), "f16": rng.random() < 0.3}
    if kind == "conv":
        return {"kind": kind, "seq": _logint(rng, 16, 4096), "channels": 4 * rng.randint(512, 2048)}
    if kind == "scan":
        return {"kind": kind, "seq": _logint(rng, 64, 4096), "channels": 4 * rng.randint(512, 2048),
                "state": rng.choice(["f32", "f16", "bf16"])}
    if kind == "glue":
        return {"kind": kind, "rows": _logint(rng, 64, 16384), "hk": heads[0], "hv": heads[1]}
    if kind == "matmul":
        n, k = rng.choice(MATRICES)
        return {"kind": kind, "m": _logint(rng, 1, 8192), "n": n, "k": k}
    if kind == "attention":
        return {"kind": kind, "batch": rng.randint(1, 16), "length": _logint(rng, 32, 32768)}
    batch = rng.choice([1, 1, 2, 4, 8, 16])
    return {"kind": kind, "batch": batch, "prompt": _logint(rng, 8, 8192 // batch), "steps": rng.randint(0, 12)}


# ---- inputs -------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV)


def _unit(x):
    return x / x.norm(dim=-1, keepdim=True)


def _gates(g, shape, kind):
    """log gates [.., heads] <= 0: "short" memory is the benchmark's
    distribution, "long" gates hardly forget, "mixed" heads span both."""
    base = -torch.nn.functional.softplus(_randn(g, *shape))
    if kind == "short":
        return base * torch.exp(-2.0 * _rand(g, *shape))
    lo, hi = (math.log(1e-3), 0.0) if kind == "mixed" else (math.log(5e-4), math.log(5e-3))
    return base * torch.exp(lo + (hi - lo) * _rand(g, shape[-1]))


def _layer_step_inputs(c, g):
    b, hk, hv = c["batch"], c["hk"], c["hv"]
    ch = (2 * hk + hv) * D
    t = {
        "x": _randn(g, b, 1, ch), "conv_state": _randn(g, b, ch, 4), "w": 0.25 * _randn(g, ch, 4),
        "a": _randn(g, b, hv), "b": _randn(g, b, hv),
        "A_log": math.log(16.0) * _rand(g, hv), "dt_bias": 1.0 + 0.5 * _randn(g, hv),
        "S": 0.02 * _randn(g, b, hv, D, D), "z": _randn(g, b, hv, D), "norm_w": 1.0 + 0.1 * _randn(g, D),
    }
    if c["f16"]:
        t["S"] = t["S"].half()
    return t


def _chunk_inputs(c, g):
    b, s, hk, hv = c["batch"], c["seq"], c["hk"], c["hv"]
    t = {
        "q": _unit(_randn(g, b, s, hk, D)).bfloat16(), "k": _unit(_randn(g, b, s, hk, D)).bfloat16(),
        "v": _randn(g, b, s, hv, D).bfloat16(), "g": _gates(g, (b, s, hv), c["gates"]).contiguous(),
        "beta": torch.sigmoid(_randn(g, b, s, hv)), "S": 0.02 * _randn(g, b, hv, D, D),
    }
    if c["f16"]:
        t["S"] = t["S"].half()
    return t


def _conv_inputs(c, g):
    s, ch = c["seq"], c["channels"]
    return {"x": _randn(g, s, ch), "w": 0.25 * _randn(g, 4, ch), "hist": _randn(g, 3, ch)}


_STATE = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def _scan_inputs(c, g):
    s, ch = c["seq"], c["channels"]
    return {"g": torch.sigmoid(2.0 + _randn(g, s, ch)), "x": _randn(g, s, ch),
            "state": _randn(g, ch).to(_STATE[c["state"]])}


def _glue_inputs(c, g):
    r, hk, hv = c["rows"], c["hk"], c["hv"]
    return {"x": _randn(g, r, (2 * hk + hv) * D), "a": _randn(g, r, hv), "b": _randn(g, r, hv),
            "A_log": math.log(16.0) * _rand(g, hv), "dt_bias": 1.0 + 0.5 * _randn(g, hv),
            "o": (0.1 * _randn(g, r, hv, D)).bfloat16(), "z": _randn(g, r, hv, D).bfloat16(),
            "norm_w": (1.0 + 0.1 * _randn(g, D)).bfloat16()}


def _matmul_inputs(c, g):
    m, n, k = c["m"], c["n"], c["k"]
    w = torch.randint(-127, 128, (n, k), generator=g, device=DEV, dtype=torch.int8)
    return {"x": _randn(g, m, k).half(), "w": w, "scale": (0.5 + _rand(g, n)) * (0.06 / 127)}


def _attention_inputs(c, g):
    b, n = c["batch"], c["length"]
    cap = (n + 256) // 256 * 256      # the cache's capacity in positions
    return {"q": _randn(g, b, 16, 256).half(), "K": _randn(g, b, 4, cap, 256).half(),
            "V": _randn(g, b, 4, cap, 256).half()}


def _model_tokens(c, seed):
    rs = np.random.RandomState(seed % (2 ** 32))
    return rs.randint(0, 151936, (c["batch"], c["prompt"] + c["steps"])).astype(np.int32)


# ---- prepare and run ------------------------------------------------------------

def prepare(case, seed):
    c, L = case, ob.lib()
    st = torch.cuda.current_stream().cuda_stream
    if c["kind"] == "model":
        # the model is the program's own, kept for its lifetime; its weights come from the seed
        cap = max(4096, c["prompt"] + c["steps"] + 1)
        m = hybrid.HybridModel(hybrid.qwen35_4b(c["batch"], cap), seed % (2 ** 31))
        tok = torch.from_numpy(_model_tokens(c, seed)).to(DEV)
        p = c["prompt"]
        return {"model": m, "prompt": tok[:, :p].contiguous(),
                "steps": [tok[:, p + i].contiguous() for i in range(c["steps"])],
                "next": torch.empty(c["batch"], dtype=torch.int32, device=DEV),
                "logits": torch.empty(c["steps"] + 1, c["batch"], m.cfg.vocab, device=DEV)}
    t = globals()[f"_{c['kind']}_inputs"](c, _gen(seed))
    s = {"keep": t}
    new = lambda *shape, dtype=torch.float32: torch.empty(*shape, dtype=dtype, device=DEV)
    P = lambda x: x.data_ptr()
    if c["kind"] == "layer_step":
        b, hk, hv = c["batch"], c["hk"], c["hv"]
        o = {"conv": new(b, 1, (2 * hk + hv) * D), "q": new(b, hk, D), "k": new(b, hk, D), "v": new(b, hv, D),
             "g": new(b, hv), "beta": new(b, hv), "o": new(b, hv, D), "y": new(b, hv, D)}
        step = L.kai_run_gdn_delta_rule_decode_f16state_hip if c["f16"] else L.kai_run_gdn_delta_rule_decode_f32_hip
        s["calls"] = [
            (L.kai_run_gdn_causal_conv1d_update_f32_hip,
             (P(t["x"]), P(t["conv_state"]), P(t["w"]), P(o["conv"]), b, 1, (2 * hk + hv) * D, 1, st)),
            (L.kai_run_gdn_gating_prologue_f32_hip,
             (P(o["conv"]), P(t["a"]), P(t["b"]), P(t["A_log"]), P(t["dt_bias"]), P(o["q"]), P(o["k"]), P(o["v"]),
              P(o["g"]), P(o["beta"]), b, hk, hv, st)),
            (step, (P(t["S"]), P(o["q"]), P(o["k"]), P(o["v"]), P(o["g"]), P(o["beta"]), P(o["o"]), b, hv, hk, D, D,
                    D ** -0.5, st)),
            (L.kai_run_gdn_gated_rmsnorm_f32_hip, (P(o["o"]), P(t["z"]), P(t["norm_w"]), P(o["y"]), b * hv, 1e-6, st)),
        ]
        s["keep2"] = o
        s["out"] = {"y": o["y"], "S": t["S"], "conv_state": t["conv_state"]}
    elif c["kind"] == "chunk":
        o = new(c["batch"], c["seq"], c["hv"], D, dtype=torch.bfloat16)
        f = (L.kai_run_gdn_chunk_delta_rule_bf16_f16state_hip if c["f16"]
             else L.kai_run_gdn_chunk_delta_rule_bf16_f32_hip)
        s["calls"] = [(f, (P(t["q"]), P(t["k"]), P(t["v"]), P(t["g"]), P(t["beta"]), P(o), P(t["S"]), c["batch"],
                           c["seq"], c["hv"], c["hk"], D ** -0.5, st))]
        s["out"] = {"o": o, "S": t["S"]}
    elif c["kind"] == "conv":
        o = new(c["seq"], c["channels"])
        s["calls"] = [(L.kai_run_gdn_causal_dwconv1d_silu_f32_k4_hip,
                       (P(t["x"]), P(t["w"]), P(o), P(t["hist"]), c["seq"], c["channels"], st))]
        s["out"] = {"out": o, "hist": t["hist"]}
    elif c["kind"] == "scan":
        o = new(c["seq"], c["channels"])
        f = getattr(L, f"kai_run_gdn_gated_scan_{c['state']}_hip")
        s["calls"] = [(f, (P(t["g"]), P(t["x"]), P(o), P(t["state"]), c["seq"], c["channels"], st))]
        s["out"] = {"s": o, "state": t["state"]}
    elif c["kind"] == "glue":
        r, hk, hv, bf = c["rows"], c["hk"], c["hv"], torch.bfloat16
        o = {"q": new(r, hk, D, dtype=bf), "k": new(r, hk, D, dtype=bf), "v": new(r, hv, D, dtype=bf),
             "g": new(r, hv), "beta": new(r, hv), "y": new(r, hv, D, dtype=bf)}
        s["calls"] = [
            (L.kai_run_gdn_gating_prologue_bf16_hip,
             (P(t["x"]), P(t["a"]), P(t["b"]), P(t["A_log"]), P(t["dt_bias"]), P(o["q"]), P(o["k"]), P(o["v"]),
              P(o["g"]), P(o["beta"]), r, hk, hv, st)),
            (L.kai_run_gdn_gated_rmsnorm_bf16_hip, (P(t["o"]), P(t["z"]), P(t["norm_w"]), P(o["y"]), r * hv, 1e-6,
                                                   st)),
        ]
        s["out"] = o
    elif c["kind"] == "matmul":
        m, n, k = c["m"], c["n"], c["k"]
        wt = torch.empty_like(t["w"])
        ob.check(L.kai_run_gdn_w8_tile_hip(P(t["w"]), P(wt), n, k, st), "tile")  # laid out once, with the weights
        wb = L.kai_gdn_w8a16_gemm_tiled_workspace_bytes(m, n, k)
        ws = torch.zeros(max(wb, 16), dtype=torch.uint8, device=DEV)
        y = new(m, n)
        s["calls"] = [(L.kai_run_gdn_w8a16_gemm_tiled_hip,
                       (P(t["x"]), P(wt), P(t["scale"]), P(y), m, n, k, P(ws), wb, st))]
        s["keep2"] = (wt, ws)
        s["out"] = y
    else:
        b, n = c["batch"], c["length"]
        wb = L.kai_gdn_attn_decode_workspace_bytes(b, 16, n)
        ws = torch.empty(max(wb, 16), dtype=torch.uint8, device=DEV)
        o = new(b, 16, 256)
        s["calls"] = [(L.kai_run_gdn_attn_decode_f16kv_hip,
                       (P(t["q"]), P(t["K"]), P(t["V"]), P(o), b, 16, 4, t["K"].shape[2], n, 1.0 / 16.0, P(ws), wb,
                        st))]
        s["keep2"] = ws
        s["out"] = o
    return s


def run(state):
    if "model" in state:
        m, lg = state["model"], state["logits"]
        m.prefill(state["prompt"], state["next"], lg[0])
        for i, tok in enumerate(state["steps"]):
            m.step(tok, state["next"], lg[i + 1])
        return lg
    for f, args in state["calls"]:
        rc = f(*args)
        if rc:
            ob.check(rc, f.__name__)
    return state["out"]


# ---- work and tolerance -----------------------------------------------------------

def work(case):
    c, k = case, case["kind"]
    if k == "layer_step":
        b, ch = c["batch"], (2 * c["hk"] + c["hv"]) * D
        st = b * c["hv"] * D * D
        small = b * ch * 4 + 2 * b * ch * 16 + 2 * b * c["hv"] * D * 4 + 2 * b * c["hv"] * 4 + ch * 16
        return {"bytes": 2 * st * (2 if c["f16"] else 4) + small, "flops": 8 * st}
    if k == "chunk":
        tok = c["batch"] * c["seq"]
        st = c["batch"] * c["hv"] * D * D * (2 if c["f16"] else 4)
        # the chunk products of the WY form at chunk 64, per 64 tokens and head
        flops = tok * c["hv"] * (5 * 2 * 64 * D + 3 * 2 * D * D)
        return {"bytes": tok * (2 * c["hk"] * D * 2 + 2 * c["hv"] * D * 2 + c["hv"] * 8) + 2 * st, "flops": flops}
    if k == "conv":
        return {"bytes": (2 * c["seq"] + 4 + 6) * c["channels"] * 4, "flops": 12 * c["seq"] * c["channels"]}
    if k == "scan":
        return {"bytes": 3 * c["seq"] * c["channels"] * 4 + 2 * c["channels"] * (4 if c["state"] == "f32" else 2),
                "flops": 2 * c["seq"] * c["channels"]}
    if k == "glue":
        n, ch = c["rows"], (2 * c["hk"] + c["hv"]) * D
        return {"bytes": n * (ch * 6 + c["hv"] * 16 + c["hv"] * D * 6), "flops": n * (ch * 4 + c["hv"] * D * 10)}
    if k == "matmul":
        m, n, kk = c["m"], c["n"], c["k"]
        return {"bytes": n * kk + n * 4 + m * kk * 2 + m * n * 4, "flops": 2 * m * n * kk}
    if k == "attention":
        kv = c["batch"] * 4 * c["length"] * 256
        return {"bytes": 2 * kv * 2 + c["batch"] * 16 * 256 * 6, "flops": 4 * 4 * kv}
    # model: int8 matrices once per pass over them, the KV cache and states
    # the steps read, the matrix products and the causal attention
    b, p, n = c["batch"], c["prompt"], c["steps"]
    per_layer = 24 * (12352 * 2560 + 2560 * 4096) + 8 * (10240 * 2560 + 2560 * 4096) + 32 * 3 * 9216 * 2560
    head = 151936 * 2560
    state = 24 * b * 32 * D * D * 4
    kv_token = 8 * 2 * 4 * 256 * 2
    step_bytes = per_layer + head + 2 * state + b * (p + n / 2) * kv_token + b * 151936 * 4
    pre_bytes = per_layer + head + state + b * p * kv_token + b * 151936 * 4
    gdn = 24 * 32 * (5 * 2 * 64 * D + 3 * 2 * D * D)
    flops = b * p * (2 * per_layer + gdn) + b * 8 * 16 * 2 * 256 * p * p + 2 * b * head
    flops += n * b * (2 * per_layer + 2 * head + 24 * 32 * 8 * D * D + 8 * 16 * 4 * 256 * p)
    return {"bytes": int(pre_bytes + n * step_bytes), "flops": int(flops)}


def tolerance(case):
    """Largest relative differences between correct implementations: about
    four times the distance measured between the path and its 64-bit result."""
    c = case
    if c["kind"] == "chunk":
        return {"rel": 1.2e-2}      # bf16 operands and output; measured 3e-3
    if c["kind"] == "model":
        return {"rel": 6e-2}        # fp16 activations through 32 layers; measured 1.5e-2 to 2.4e-2
    if c["kind"] == "glue":
        return {"rel": 1e-2}        # bf16 outputs; measured 2.8e-3
    if c["kind"] == "matmul":
        return {"rel": 2.5e-6}      # exact products, fp32 sums; measured 6e-7
    if c["kind"] == "attention":
        return {"rel": 1.2e-6}      # fp32 softmax and sums; measured 3e-7
    if c["kind"] == "scan":         # the carried state is rounded to its own type
        return {"rel": {"f32": 3e-7, "f16": 1e-3, "bf16": 6e-3}[c["state"]]}
    if c["kind"] == "layer_step":
        return {"rel": 1e-3 if c["f16"] else 1e-6}
    return {"rel": 3e-7}            # conv: four fp32 products and a SiLU; measured 7e-8


# ---- 64-bit results ------------------------------------------------------------------

def exact(case, seed):
    c = case
    if c["kind"] == "model":
        if c["batch"] * (c["prompt"] + c["steps"]) > 2000:
            return None             # a sequential recurrence and 4B weights in 64 bits: minutes
        return _exact_model(c, seed)
    t = globals()[f"_{c['kind']}_inputs"](c, _gen(seed))
    return globals()[f"_exact_{c['kind']}"](c, {k: (v if k == "w" else v.double()) for k, v in t.items()})


def _silu(x):
    return x * torch.sigmoid(x)


def _recurrence(q, k, v, g, beta, S, out):
    """S [B, Hv, D, D] through every token; q, k [B, T, Hv, D]."""
    a = torch.exp(g)
    for i in range(q.shape[1]):
        S = S * a[:, i, :, None, None]
        ki = k[:, i, :, :, None]
        d = (v[:, i] - (S * ki).sum(-2)) * beta[:, i, :, None]
        S = S + ki * d[:, :, None, :]
        out[:, i] = (S * q[:, i, :, :, None]).sum(-2) * D ** -0.5
    return S


def _prologue(x, a, b, A_log, dt_bias, hk, hv):
    rows = x.shape[0]
    q, k, v = x[:, :hk * D], x[:, hk * D:2 * hk * D], x[:, 2 * hk * D:]
    q, k, v = (z.reshape(rows, -1, D) for z in (q, k, v))
    n = lambda z: z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6)
    return n(q), n(k), v, -torch.exp(A_log) * torch.nn.functional.softplus(a + dt_bias), torch.sigmoid(b)


def _rms(x, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _exact_layer_step(c, t):
    b, hk, hv = c["batch"], c["hk"], c["hv"]
    state = torch.cat([t["conv_state"][:, :, 1:], t["x"].reshape(b, -1, 1)], dim=2)
    cv = _silu((state * t["w"].double()).sum(-1))
    q, k, v, g, beta = _prologue(cv, t["a"], t["b"], t["A_log"], t["dt_bias"], hk, hv)
    q, k = (z.repeat_interleave(hv // hk, dim=1) for z in (q, k))
    o = torch.empty(b, 1, hv, D, dtype=torch.float64, device=DEV)
    S = _recurrence(q[:, None], k[:, None], v[:, None], g[:, None], beta[:, None], t["S"], o)
    return {"y": t["norm_w"] * _rms(o[:, 0]) * _silu(t["z"]), "S": S, "conv_state": state}


def _exact_chunk(c, t):
    r = c["hv"] // c["hk"]
    q, k = (t[n].repeat_interleave(r, dim=2) for n in ("q", "k"))
    o = torch.empty_like(t["v"])
    return {"o": o, "S": _recurrence(q, k, t["v"], t["g"], t["beta"], t["S"], o)}


def _exact_conv(c, t):
    x = torch.cat([t["hist"], t["x"]])
    s, w = c["seq"], t["w"].double()
    return {"out": _silu(sum(x[i:i + s] * w[i] for i in range(4))), "hist": x[-3:]}


def _exact_scan(c, t):
    s, o = t["state"], torch.empty_like(t["x"])
    for i in range(c["seq"]):
        s = t["g"][i] * s + t["x"][i]
        o[i] = s
    return {"s": o, "state": s}


def _exact_glue(c, t):
    q, k, v, g, beta = _prologue(t["x"], t["a"], t["b"], t["A_log"], t["dt_bias"], c["hk"], c["hv"])
    return {"q": q, "k": k, "v": v, "g": g, "beta": beta, "y": t["norm_w"] * _rms(t["o"]) * _silu(t["z"])}


def _exact_matmul(c, t):
    return t["x"] @ t["w"].double().t() * t["scale"]


def _exact_attention(c, t):
    n = c["length"]
    q = t["q"].reshape(c["batch"], 4, 4, 256)
    K, V = t["K"][:, :, :n], t["V"][:, :, :n]
    p = torch.softmax(q @ K.transpose(2, 3).contiguous() / 16.0, dim=-1)
    return (p @ V).reshape(c["batch"], 16, 256)


# The hybrid model in 64 bits from its definition: values drawn by a
# counter-based hash of (seed, tensor, index), matrices quantised per output
# channel, one causal forward over prompt and continuation.

_M1, _M2, _GOLD = (x - (1 << 64) for x in (0xBF58476D1CE4E5B9, 0x94D049BB133111EB, 0x9E3779B97F4A7C15))


def _shr(z, n):
    return (z >> n) & ((1 << (64 - n)) - 1)


def _mix(z):
    z = z + _GOLD
    z = (z ^ _shr(z, 30)) * _M1
    z = (z ^ _shr(z, 27)) * _M2
    return z ^ _shr(z, 31)


def _drawn(seed, stream, shape, amp, center, dtype=torch.float32):
    n = math.prod(shape)
    key = (seed ^ (stream * 0x100000001B3)) & (2 ** 64 - 1)
    key = _mix(torch.tensor([key - 2 ** 64 if key >= 2 ** 63 else key], device=DEV))
    out = torch.empty(n, dtype=dtype, device=DEV)
    for lo in range(0, n, 1 << 26):
        i = torch.arange(lo, min(n, lo + (1 << 26)), device=DEV)
        u = _shr(_mix(key + i), 40).float() * 2.0 ** -24
        out[lo:lo + i.numel()] = ((u * 2.0 - 1.0) * amp + center).to(dtype)
    return out.reshape(shape)


def _weight(seed, stream, n, k):
    """The quantised matrix [n, k] with its scales applied, in 64 bits."""
    w = _drawn(seed, stream, (n, k), 0.034641016, 0.0)
    s = w.abs().amax(1, keepdim=True) / 127.0
    v = w * (1.0 / s)
    q = torch.trunc(v)
    q = q + torch.sign(v) * ((v - q).abs() >= 0.5)
    return q.double() * s.double()


def _rotate(x, theta):
    """Rotary embedding of dims 0..63 of x [B, T, heads, 256]."""
    i = torch.arange(32, device=DEV, dtype=torch.float64)
    f = torch.arange(x.shape[1], device=DEV, dtype=torch.float64)[:, None] / theta ** (i / 32.0)
    cs, sn = torch.cos(f)[:, None, :], torch.sin(f)[:, None, :]
    lo, hi = x[..., :32], x[..., 32:64]
    return torch.cat([lo * cs - hi * sn, hi * cs + lo * sn, x[..., 64:]], dim=-1)


def _exact_model(c, case_seed):
    seed, B, T, H, hk, hv = case_seed % (2 ** 31), c["batch"], c["prompt"] + c["steps"], 2560, 16, 32
    tok = torch.from_numpy(_model_tokens(c, case_seed)).long().to(DEV)
    h = _drawn(seed, 1, (151936, H), 1.0, 0.0, torch.float16)[tok].double()
    ch = (2 * hk + hv) * D
    vec = lambda stream, n, amp, center: _drawn(seed, stream, (n,), amp, center).double()
    mul = lambda x, stream, n: x @ _weight(seed, stream, n, x.shape[-1]).t()
    for layer in range(32):
        s = 64 * (layer + 1)
        x = _rms(h) * (1.0 + vec(s + 0, H, 0.1, 0.0))
        if (layer + 1) % 4:
            qkv = torch.nn.functional.pad(mul(x, s + 2, ch), (0, 0, 3, 0))
            w = _drawn(seed, s + 7, (ch, 4), 0.5, 0.0).double()
            cv = _silu(sum(qkv[:, j:j + T] * w[:, j] for j in range(4)))
            q, k, v, g, beta = _prologue(cv.reshape(B * T, ch), mul(x, s + 5, hv).reshape(B * T, hv),
                                         mul(x, s + 4, hv).reshape(B * T, hv),
                                         vec(s + 9, hv, 1.3862944, 1.3862944), vec(s + 8, hv, 0.5, 1.0), hk, hv)
            q, k = (z.reshape(B, T, hk, D).repeat_interleave(hv // hk, dim=2) for z in (q, k))
            o = torch.empty(B, T, hv, D, dtype=torch.float64, device=DEV)
            S = torch.zeros(B, hv, D, D, dtype=torch.float64, device=DEV)
            _recurrence(q, k, v.reshape(B, T, hv, D), g.reshape(B, T, hv), beta.reshape(B, T, hv), S, o)
            y = vec(s + 10, D, 0.1, 1.0) * _rms(o) * _silu(mul(x, s + 3, hv * D).reshape(B, T, hv, D))
            h = h + mul(y.reshape(B, T, hv * D), s + 6, H)
        else:
            qg = mul(x, s + 11, 16 * 512).reshape(B, T, 16, 512)
            q = _rotate(_rms(qg[..., :256]) * (1.0 + vec(s + 15, 256, 0.1, 0.0)), 1e7)
            k = _rotate(_rms(mul(x, s + 12, 1024).reshape(B, T, 4, 256)) * (1.0 + vec(s + 16, 256, 0.1, 0.0)), 1e7)
            v = mul(x, s + 13, 1024).reshape(B, T, 4, 256)
            k, v = (z.repeat_interleave(4, dim=2).transpose(1, 2).contiguous() for z in (k, v))
            a = q.transpose(1, 2).contiguous() @ k.transpose(2, 3).contiguous() / 16.0
            a = torch.softmax(a.masked_fill(torch.ones(T, T, device=DEV, dtype=torch.bool).triu(1), -math.inf), -1)
            o = (a @ v).transpose(1, 2) * torch.sigmoid(qg[..., 256:])
            h = h + mul(o.reshape(B, T, 4096), s + 14, H)
        x = _rms(h) * (1.0 + vec(s + 1, H, 0.1, 0.0))
        h = h + mul(_silu(mul(x, s + 17, 9216)) * mul(x, s + 18, 9216), s + 19, H)
    x = _rms(h[:, c["prompt"] - 1:]) * (1.0 + vec(2, H, 0.1, 0.0))
    return mul(x, 3, 151936).transpose(0, 1)
