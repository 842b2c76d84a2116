"""Performance cases of the decode and prefill attention paths.

Each case is one call (or one captured decode step) as a generation program issues it, on
inputs that are already on the GPU, with the workspace, rotary table and output buffers that
such a program keeps.  Shapes are Gemma-4's: local layers with head_dim 256 and a 1024-token
window, global layers with head_dim 512 and GQA 8; contexts from a few hundred tokens to
131,072.

Kinds
  step         the attention of 12 layers (every 6th global) of one decode step, replayed from
               a HIP graph: what a decode loop does for every generated token
  local        one decode call of a sliding layer (ring cache, separate K and V)
  global       one decode call of a global layer over one K = V buffer (attention_k_eq_v)
  raw, q8      one decode call of a global layer over a raw-K / quantized raw-K stream, with
               the per-model rotary table or (table = False) without it
  prefill      attention of a chunk of new tokens over the cached keys
  prefill_raw  a chunk over a raw-K / q8 stream: K and V rebuilt, then attended
"""
from __future__ import annotations

import math

import torch

from apertura_amd.decode import (DecodeCall, DecodeStep, RawCall, RawQ8Call, RawStep, new_raw_workspace, new_workspace,
                                 q8_step_for, rope_table)
from apertura_amd.prefill import PrefillStep, prefill, prefill_workspace_bytes, raw_prefill_kv, raw_q8_prefill_kv

DEV = "cuda"
BF = torch.bfloat16
WINDOW = 1024
EPS = 1e-6


def listed() -> list[dict]:
    return [
        # one sliding layer for one user: 1024 rows, the smallest call, latency only
        {"name": "local_b1", "kind": "local", "batch": 1, "hq": 16, "hkv": 8, "length": 1024},
        # a decode loop's token for one user at an ordinary depth, from a graph
        {"name": "step_b1_4k", "kind": "step", "batch": 1, "length": 4321},
        # one sliding layer of a serving batch
        {"name": "local_b32", "kind": "local", "batch": 32, "hq": 32, "hkv": 16, "length": 32768},
        # one global layer for one user: an ordinary and a full context
        {"name": "global_b1_8k", "kind": "global", "batch": 1, "hq": 32, "hkv": 4, "length": 8193},
        {"name": "global_b1_128k", "kind": "global", "batch": 1, "hq": 32, "hkv": 4, "length": 131072},
        # one global layer of a serving batch, lengths drawn from 1024 .. 32768
        {"name": "global_b16", "kind": "global", "batch": 16, "hq": 32, "hkv": 4, "length": 32768},
        # raw-K and q8 raw-K caches: a long document, and the longest context
        {"name": "raw_b1_61k", "kind": "raw", "batch": 1, "hq": 32, "hkv": 4, "length": 61440, "table": True},
        {"name": "q8_b1_128k", "kind": "q8", "batch": 1, "hq": 32, "hkv": 4, "length": 131072, "table": True},
        # a chunk of a long prompt on a global layer, and a chat turn on the same layer
        {"name": "prefill_global_chunk", "kind": "prefill", "hq": 32, "hkv": 4, "dim": 512, "queries": 512,
         "past": 15872, "window": 0, "shared": True},
        {"name": "prefill_global_turn", "kind": "prefill", "hq": 32, "hkv": 4, "dim": 512, "queries": 333,
         "past": 5600, "window": 0, "shared": True},
        # a fresh prompt on a sliding layer
        {"name": "prefill_local_4k", "kind": "prefill", "hq": 32, "hkv": 16, "dim": 256, "queries": 4096,
         "past": 0, "window": WINDOW, "shared": False},
        # a chat turn on a global layer with a raw-K cache
        {"name": "prefill_raw_turn", "kind": "prefill_raw", "hq": 32, "hkv": 4, "queries": 200, "past": 8056,
         "q8": False},
    ]


def _log_uniform(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng) -> dict:
    kind = rng.choice(["step", "local", "global", "global", "raw", "q8", "prefill", "prefill", "prefill",
                       "prefill_raw", "prefill_raw"])
    if kind == "step":
        return {"kind": kind, "batch": 1, "length": _log_uniform(rng, 512, 16384)}
    if kind == "local":
        hq, hkv = rng.choice([(16, 8), (32, 16)])
        return {"kind": kind, "batch": _log_uniform(rng, 1, 32), "hq": hq, "hkv": hkv,
                "length": _log_uniform(rng, 512, 32768)}
    hq, hkv = rng.choice([(32, 4), (32, 4), (16, 2)])
    if kind in ("global", "raw", "q8"):
        batch = rng.choice([1, _log_uniform(rng, 1, 16)])
        case = {"kind": kind, "batch": batch, "hq": hq, "hkv": hkv,
                "length": _log_uniform(rng, 512, 131072 if batch == 1 else 32768)}
        if kind != "global":
            case["table"] = rng.random() < 0.7
        return case
    queries = _log_uniform(rng, 16, 4096)
    if kind == "prefill_raw":
        queries = min(queries, 1024)
        past = rng.choice([0, _log_uniform(rng, 64, 12000), _log_uniform(rng, 64, 12000)])
        return {"kind": kind, "hq": hq, "hkv": hkv, "queries": min(queries, 512 if past > 6000 else 1024),
                "past": past, "q8": rng.random() < 0.5}
    if rng.random() < 0.5:
        hq, hkv = rng.choice([(16, 8), (32, 16)])
        return {"kind": kind, "hq": hq, "hkv": hkv, "dim": 256, "queries": queries,
                "past": rng.choice([0, _log_uniform(rng, 64, 30000)]), "window": WINDOW, "shared": False}
    past = rng.choice([0, _log_uniform(rng, 64, 15000), _log_uniform(rng, 64, 15000)])
    queries = min(queries, 512 if past else 4000)
    return {"kind": kind, "hq": hq, "hkv": hkv, "dim": 512, "queries": queries, "past": past, "window": 0,
            "shared": rng.random() < 0.7}


# ------------------------------------------------------------------------------ inputs

def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _rms_rows(shape, g) -> torch.Tensor:
    """bf16 rows of unit root mean square: what a q, k or v norm leaves."""
    x = torch.randn(shape, device=DEV, dtype=torch.float32, generator=g)
    x *= torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    return x.to(BF)


def _point_at(k: torch.Tensor, q: torch.Tensor, g) -> None:
    """Turns about one cached key in 100 towards its kv head's first query head, a logit of
    +4 at scale 1 / sqrt(D): attention that dwells on some rows.  k [.., rows, D], q [.., D]."""
    if k.shape[-2] == 0:
        return
    hit = torch.rand(k.shape[:-1], device=DEV, generator=g) < 0.01
    qh = q.float()
    add = (4.0 * qh / qh.norm(dim=-1, keepdim=True)).unsqueeze(-2)
    idx = hit.nonzero(as_tuple=True)
    lead = idx[:-1] + (torch.zeros_like(idx[-1]),)
    k[idx] = (k[idx].float() + add[lead]).to(BF)


def _lengths(case: dict, g) -> list[int]:
    """Rows of each sequence after this step: the length itself for one user, else drawn up
    to it (the longest first)."""
    B, n = case["batch"], case["length"]
    if B == 1:
        return [n]
    u = torch.rand(B, device=DEV, generator=g)
    lo = min(1024, n)
    return [n] + [lo + int(x * (n - lo)) for x in u.tolist()[1:]]


def _pos(lengths: list[int]) -> torch.Tensor:
    return torch.tensor([n - 1 for n in lengths], dtype=torch.int32, device=DEV)


def _local_inputs(case: dict, g) -> dict:
    B, Hq, Hkv, D = case["batch"], case["hq"], case["hkv"], 256
    s = {"lengths": _lengths(case, g), "q": _rms_rows((B, Hq, D), g), "k": _rms_rows((B, Hkv, WINDOW, D), g),
         "v": _rms_rows((B, Hkv, WINDOW, D), g), "k_new": _rms_rows((B, Hkv, D), g), "v_new": _rms_rows((B, Hkv, D), g)}
    _point_at(s["k"], s["q"][:, :: Hq // Hkv], g)
    return s


def _global_inputs(case: dict, g) -> dict:
    B, Hq, Hkv, D = case["batch"], case["hq"], case["hkv"], 512
    s = {"lengths": _lengths(case, g), "q": _rms_rows((B, Hq, D), g)}
    s["k"] = torch.empty((B, Hkv, case["length"], D), dtype=BF, device=DEV)
    for b in range(B):
        s["k"][b] = _rms_rows((Hkv, case["length"], D), g)
        _point_at(s["k"][b], s["q"][b, :: Hq // Hkv], g)
    s["k_new"] = _rms_rows((B, Hkv, D), g)
    return s


def _raw_weights(g) -> dict:
    """A k-norm weight that carries the softmax scale (the model's own is 1), and Gemma-4's
    global rotary frequencies: 64 of 256 pairs rotate."""
    kw = (0.06 * (1.0 + 0.25 * torch.randn(512, device=DEV, generator=g))).to(BF)
    inv = torch.zeros(256, dtype=torch.float32, device=DEV)
    inv[:64] = (1.0 / (1.0e6 ** (torch.arange(64, dtype=torch.float64, device=DEV) * 2 / 512))).float()
    return {"kw": kw, "inv_freq": inv}


def _raw_rows(shape, g) -> torch.Tensor:
    """k_proj rows before the norm: a magnitude that differs from row to row."""
    x = torch.randn(shape, device=DEV, dtype=torch.float32, generator=g)
    x *= 2.0 * torch.exp(0.3 * torch.randn(shape[:-1], device=DEV, generator=g)).unsqueeze(-1)
    return x.to(BF)


def _quantized(x: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Per-row affine u8 of bf16 rows: q, scale, bias with x ~ q * scale + bias."""
    x = x.float()
    lo, hi = x.amin(-1, keepdim=True), x.amax(-1, keepdim=True)
    sc = torch.clamp((hi - lo) / 255.0, min=1e-8)
    q = torch.clamp(torch.floor((x - lo) / sc + 0.5), max=255.0).to(torch.uint8)
    return q, sc.squeeze(-1), lo.squeeze(-1)


def _raw_inputs(case: dict, g) -> dict:
    B, Hq, Hkv, n = case["batch"], case["hq"], case["hkv"], case["length"]
    s = {"lengths": _lengths(case, g), "q": _rms_rows((B, Hq, 512), g), "k_new": _raw_rows((B, Hkv, 512), g),
         **_raw_weights(g)}
    q8 = case["kind"] == "q8"
    s["k"] = torch.empty((B, Hkv, n, 512), dtype=torch.uint8 if q8 else BF, device=DEV)
    if q8:
        s["sc"] = torch.empty((B, Hkv, n), dtype=torch.float32, device=DEV)
        s["bs"] = torch.empty((B, Hkv, n), dtype=torch.float32, device=DEV)
    for b in range(B):
        rows = _raw_rows((Hkv, n, 512), g)
        if q8:
            s["k"][b], s["sc"][b], s["bs"][b] = _quantized(rows)
        else:
            s["k"][b] = rows
    return s


def _prefill_inputs(case: dict, g) -> dict:
    """Keys of the past (a sliding layer keeps its last window + chunk) and of the chunk."""
    Hq, Hkv, D, Sq = case["hq"], case["hkv"], case["dim"], case["queries"]
    total = case["past"] + Sq
    Sk = min(total, case["window"] + Sq) if case["window"] else total
    s = {"q": _rms_rows((Hq, Sq, D), g), "k": _rms_rows((Hkv, Sk, D), g), "k_pos0": total - Sk}
    _point_at(s["k"], s["q"][:: Hq // Hkv, 0], g)
    s["v"] = s["k"] if case["shared"] else _rms_rows((Hkv, Sk, D), g)
    return s


def _prefill_raw_inputs(case: dict, g) -> dict:
    Hq, Hkv, Sq = case["hq"], case["hkv"], case["queries"]
    s = {"q": _rms_rows((Hq, Sq, 512), g), "raw": _raw_rows((Hkv, case["past"] + Sq, 512), g), **_raw_weights(g)}
    if case["q8"]:
        s["raw"], s["sc"], s["bs"] = _quantized(s["raw"])
    return s


STEP_LAYERS = 12


def _step_layers(case: dict, g) -> list[dict]:
    layers = []
    for i in range(STEP_LAYERS):
        if i % 6 == 5:
            c = {"kind": "global", "batch": case["batch"], "hq": 32, "hkv": 4, "length": case["length"]}
            layers.append({**_global_inputs(c, g), "case": c})
        else:
            c = {"kind": "local", "batch": case["batch"], "hq": 32, "hkv": 16, "length": case["length"]}
            layers.append({**_local_inputs(c, g), "case": c})
    return layers


# ------------------------------------------------------------------------------ the calls

def _decode_call(s: dict, kind: str, workspace=None) -> DecodeCall:
    if kind == "local":
        step = DecodeStep.for_cache(s["k"], s["q"].shape[1], window=WINDOW, ring=True, scale=1 / 16)
    else:
        step = DecodeStep.for_cache(s["k"], s["q"].shape[1], kv_shared=True, scale=512 ** -0.5)
    ws = workspace if workspace is not None else new_workspace(step, DEV)
    return DecodeCall(step, s["q"], s["k_new"], s.get("v_new"), s["k"], s.get("v"), _pos(s["lengths"]), workspace=ws)


def prepare(case: dict, seed: int) -> dict:
    g, kind = _gen(seed), case["kind"]
    if kind in ("local", "global"):
        s = (_local_inputs if kind == "local" else _global_inputs)(case, g)
        return {"kind": kind, "call": _decode_call(s, kind), **s}
    if kind == "step":
        layers = _step_layers(case, g)
        calls = [_decode_call(s, s["case"]["kind"]) for s in layers]
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            for c in calls:
                c(stream)
        torch.cuda.current_stream().wait_stream(stream)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for c in calls:
                c()
        return {"kind": kind, "graph": graph, "calls": calls, "layers": layers}
    if kind in ("raw", "q8"):
        s = _raw_inputs(case, g)
        tab = rope_table(s["inv_freq"], case["length"]) if case["table"] else None
        pos = _pos(s["lengths"])
        if kind == "raw":
            step = RawStep.for_cache(s["k"], case["hq"], eps=EPS)
            call = RawCall(step, s["q"], s["k_new"], s["k"], pos, s["kw"], s["inv_freq"],
                           workspace=new_raw_workspace(step, DEV), rope_table=tab)
        else:
            step = q8_step_for(s["k"], case["hq"], eps=EPS)
            call = RawQ8Call(step, s["q"], s["k_new"], s["k"], s["sc"], s["bs"], pos, s["kw"], s["inv_freq"],
                             workspace=new_raw_workspace(step, DEV), rope_table=tab)
        return {"kind": kind, "call": call, **s}
    if kind == "prefill":
        s = _prefill_inputs(case, g)
        out = torch.empty((case["queries"], case["hq"], case["dim"]), dtype=BF, device=DEV)
        step = PrefillStep.for_tensors(s["q"], s["k"], out, q_pos0=case["past"], k_pos0=s["k_pos0"],
                                       window=case["window"], scale=case["dim"] ** -0.5)
    else:
        s = _prefill_raw_inputs(case, g)
        out = torch.empty((case["queries"], case["hq"], 512), dtype=BF, device=DEV)
        shape = tuple(s["raw"].shape)
        s["k"], s["v"] = (torch.empty(shape, dtype=BF, device=DEV) for _ in range(2))
        step = PrefillStep.for_tensors(s["q"], s["k"], out, q_pos0=case["past"], scale=1.0)
    n = prefill_workspace_bytes(step)
    ws = torch.empty(n, dtype=torch.uint8, device=DEV) if n else None
    return {"kind": kind, "step": step, "out": out, "workspace": ws, **s}


def run(state: dict):
    kind = state["kind"]
    if kind == "step":
        state["graph"].replay()
        return [[c.out, s["k"]] + ([s["v"]] if "v" in s else []) for c, s in zip(state["calls"], state["layers"])]
    if kind in ("local", "global", "raw", "q8"):
        out = state["call"]()
        return [out] + [state[n] for n in ("k", "v", "sc", "bs") if n in state]
    if kind == "prefill_raw":
        if "sc" in state:
            k, v = raw_q8_prefill_kv(state["raw"], state["sc"], state["bs"], state["kw"], EPS, state["inv_freq"],
                                     k_out=state["k"], v_out=state["v"])
        else:
            k, v = raw_prefill_kv(state["raw"], state["kw"], EPS, state["inv_freq"], k_out=state["k"],
                                  v_out=state["v"])
        return [prefill(state["step"], state["q"], k, v, out=state["out"], workspace=state["workspace"]), k, v]
    return prefill(state["step"], state["q"], state["k"], state["v"], out=state["out"], workspace=state["workspace"])


# ------------------------------------------------------------------------------ work

def _visible(case: dict) -> float:
    """Rows attended over the batch (the expectation where lengths are drawn)."""
    B, n = case["batch"], case["length"]
    lo = min(1024, n)
    mean = (lo + n) / 2
    if case["kind"] == "local":
        return min(n, WINDOW) + (B - 1) * min(mean, WINDOW)
    return n + (B - 1) * mean


def _pairs(queries: int, past: int, window: int) -> int:
    """Visible (query, key) pairs of a chunk after `past` tokens."""
    total = 0
    if not window:
        return queries * past + queries * (queries + 1) // 2
    for i in range(queries):
        total += min(past + i + 1, window)
    return total


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "step":
        parts = [work({"kind": k, "batch": case["batch"], "hq": 32, "hkv": h, "length": case["length"]})
                 for k, h in (("local", 16), ("global", 4))]
        n = STEP_LAYERS // 6
        return {m: (STEP_LAYERS - n) * parts[0][m] + n * parts[1][m] for m in ("bytes", "flops")}
    hq, hkv = case["hq"], case["hkv"]
    if kind in ("local", "global", "raw", "q8"):
        dim = 256 if kind == "local" else 512
        row = {"local": 4 * dim, "global": 2 * dim, "raw": 2 * dim, "q8": dim + 8}[kind]
        rows = _visible(case)
        append = 2 * dim * (2 if kind == "local" else 1) + row  # the new row read and written
        return {"bytes": rows * hkv * row + case["batch"] * (4 * hq * dim + hkv * append),
                "flops": 4.0 * dim * rows * hq}
    Sq, past, dim = case["queries"], case["past"], case.get("dim", 512)
    window = case.get("window", 0)
    Sk = min(past + Sq, window + Sq) if window else past + Sq
    nbytes = 4 * Sq * hq * dim
    if kind == "prefill":
        nbytes += 2 * hkv * Sk * dim * (1 if case["shared"] else 2)
    else:  # the raw rows in, K and V out
        nbytes += hkv * Sk * ((520 if case["q8"] else 1024) + 2048)
    return {"bytes": float(nbytes), "flops": 4.0 * dim * hq * _pairs(Sq, past, window)}


def tolerance(case: dict) -> dict:
    """bf16 outputs of sums weighted by bf16 probabilities; measured against exact()."""
    return {"rel": 1e-2}


# ------------------------------------------------------------------------------ 64 bits

def _attend64(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, scale: float) -> torch.Tensor:
    """q [Hq, D], k / v [Hkv, n, D] -> [Hq, D], all float64."""
    Hkv, D = k.shape[0], k.shape[2]
    out = []
    for h, qh in enumerate(q.view(Hkv, -1, D)):
        out.append(torch.softmax(scale * (qh @ k[h].T), dim=-1) @ v[h])
    return torch.cat(out)


def _exact_decode(s: dict, case: dict) -> torch.Tensor:
    local = case["kind"] == "local"
    outs = []
    for b, n in enumerate(s["lengths"]):
        k = s["k"][b].double()
        v = s["v"][b].double() if local else k
        row = (n - 1) % WINDOW if local else n - 1
        k[:, row] = s["k_new"][b].double()
        if local:
            v[:, row] = s["v_new"][b].double()
        m = min(n, WINDOW) if local else n
        outs.append(_attend64(s["q"][b].double(), k[:, :m], v[:, :m], 1 / 16 if local else 512 ** -0.5))
    return torch.stack(outs)


def _cos_sin(rows: int, inv_freq: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """bf16 cos and sin of the fp32 angles row * inv_freq, as float64."""
    a = (torch.arange(rows, device=DEV, dtype=torch.float32).unsqueeze(1) * inv_freq).double()
    return a.cos().to(BF).double(), a.sin().to(BF).double()


def _raw_kv64(x: torch.Tensor, s: dict, cs, decode: bool) -> tuple[torch.Tensor, torch.Tensor]:
    """K and V of raw rows x [rows, 512] (float64): K rounded to bf16 once (decode), or at
    each op with V rounded too (prefill), as the entry points state."""
    rinv = torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    v = x * rinv
    k = v * s["kw"].double()
    c, sn = (torch.cat([t[: x.shape[0]], t[: x.shape[0]]], dim=1) for t in cs)
    if not decode:
        k = k.to(BF).double()
    turned = torch.cat([-k[:, 256:], k[:, :256]], dim=1)
    if decode:
        return (k * c + turned * sn).to(BF).double(), v
    k = ((k * c).to(BF).double() + (turned * sn).to(BF).double()).to(BF).double()
    return k, v.to(BF).double()


def _exact_raw(s: dict, case: dict) -> torch.Tensor:
    cs = _cos_sin(case["length"], s["inv_freq"])
    G = case["hq"] // case["hkv"]
    outs = []
    for b, n in enumerate(s["lengths"]):
        for h in range(case["hkv"]):
            new = s["k_new"][b, h]
            if case["kind"] == "q8":
                q, sc, bs = _quantized(new)
                x = s["k"][b, h, :n].double()
                scale, bias = s["sc"][b, h, :n].double(), s["bs"][b, h, :n].double()
                x[n - 1], scale[n - 1], bias[n - 1] = q.double(), sc.double(), bs.double()
                x = x * scale.unsqueeze(1) + bias.unsqueeze(1)
            else:
                x = s["k"][b, h, :n].double()
                x[n - 1] = new.double()
            k, v = _raw_kv64(x, s, cs, decode=True)
            outs.append(_attend64(s["q"][b, h * G:(h + 1) * G].double(), k.unsqueeze(0), v.unsqueeze(0), 1.0))
    return torch.cat(outs).view(case["batch"], case["hq"], 512)


def _exact_prefill(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, past: int, k_pos0: int, window: int,
                   scale: float) -> torch.Tensor:
    """q [Hq, Sq, D] bf16, k / v [Hkv, Sk, D] float64 -> [Sq, Hq, D] float64."""
    Hq, Sq, D = q.shape
    qa = past + torch.arange(Sq, device=DEV).unsqueeze(1)
    ka = k_pos0 + torch.arange(k.shape[1], device=DEV).unsqueeze(0)
    hidden = (ka > qa) | ((ka <= qa - window) if window else (ka < 0))
    out = torch.empty((Sq, Hq, D), dtype=torch.float64, device=DEV)
    for h in range(Hq):
        kvh = h // (Hq // k.shape[0])
        sc = scale * (q[h].double() @ k[kvh].T)
        out[:, h] = torch.softmax(sc.masked_fill(hidden, -math.inf), dim=-1) @ v[kvh]
    return out


def exact(case: dict, seed: int):
    g, kind = _gen(seed), case["kind"]
    if kind == "step":
        return [[_exact_decode(s, s["case"]), None] + ([None] if "v" in s else []) for s in _step_layers(case, g)]
    if kind in ("local", "global"):
        s = (_local_inputs if kind == "local" else _global_inputs)(case, g)
        return [_exact_decode(s, case), None] + ([None] if kind == "local" else [])
    if kind in ("raw", "q8"):
        return [_exact_raw(_raw_inputs(case, g), case), None] + ([None, None] if kind == "q8" else [])
    if kind == "prefill":
        s = _prefill_inputs(case, g)
        return _exact_prefill(s["q"], s["k"].double(), s["v"].double(), case["past"], s["k_pos0"], case["window"],
                              case["dim"] ** -0.5)
    s = _prefill_raw_inputs(case, g)
    cs = _cos_sin(case["past"] + case["queries"], s["inv_freq"])
    ks, vs = [], []
    for h in range(case["hkv"]):
        x = s["raw"][h].double()
        if case["q8"]:
            x = (x * s["sc"][h].double().unsqueeze(1) + s["bs"][h].double().unsqueeze(1)).to(BF).double()
        k, v = _raw_kv64(x, s, cs, decode=False)
        ks.append(k)
        vs.append(v)
    k, v = torch.stack(ks), torch.stack(vs)
    return [_exact_prefill(s["q"], k, v, case["past"], 0, 0, 1.0), k, v]
