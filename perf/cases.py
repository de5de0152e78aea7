"""The work this package is timed on: MoE FFN layers, dense FFNs, quantized linears and norms.

Every case is one call (or one captured decode loop) of a public entry point on weights in
GGUF block form.  Weights are normal matrices quantised here with the block formats'
published definitions, so scales, minima and codes have the distributions of a real file;
tokens are normal rows, as a norm leaves them.  `listed()` holds fixed cases, `draw(rng)`
more of the same ranges, `exact` the float64 result without the package's kernels.

Batches span one token (decode), the 9..64 rows of batched serving, a few hundred (a
chunk of a prompt beside running decodes) and whole prompts.
"""

from __future__ import annotations

import math
import os
import sys
from typing import Any, Callable, Dict, List, Optional, Tuple

import numpy as np
import torch
import torch.nn.functional as F

_PKG = os.path.join(os.getcwd(), "pytorch-engine_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

import pgmoe  # noqa: E402

F16, Q8_0, Q4_K, Q5_K, Q6_K = 1, 8, 12, 13, 14
_TYPES = {"f16": F16, "q8_0": Q8_0, "q4_k": Q4_K, "q5_k": Q5_K, "q6_k": Q6_K}
_BITS = {"f16": 16.0, "q8_0": 8.5, "q4_k": 4.5, "q5_k": 5.5, "q6_k": 6.5625}  # a weight, scales included

# Layer shapes of this repository's configurations (pgmoe.synth): hidden, experts, experts a
# token, intermediate size, formats of gate / up and of down, shared expert.
_MOE = {
    "qwen3_30b_a3b": dict(arch="qwen3moe", hidden=2048, experts=128, top_k=8, inter=768, gate_up="q4_k", down="q6_k",
                          norm_topk=True, shared=0),
    "mixtral_8x7b": dict(arch="mixtral", hidden=4096, experts=8, top_k=2, inter=14336, gate_up="q4_k", down="q4_k",
                         norm_topk=True, shared=0),
    "qwen2_57b_a14b": dict(arch="qwen2moe", hidden=3584, experts=64, top_k=8, inter=2560, gate_up="q8_0", down="q8_0",
                           norm_topk=False, shared=20480),
}


def _moe(shape: str, tokens: int, steps: int = 1, graph: bool = False, skew: bool = False) -> Dict[str, Any]:
    return dict(kind="moe", shape=shape, tokens=tokens, steps=steps, graph=graph, skew=skew)


def _dense(tokens: int, hidden: int = 4096, inter: int = 12288, gate_up: str = "q4_k", down: str = "q6_k"):
    return dict(kind="dense", tokens=tokens, hidden=hidden, inter=inter, gate_up=gate_up, down=down)


def _linear(tokens: int, cols: int, rows: int, qtype: str, parts: int = 1, bias: bool = False):
    return dict(kind="linear", tokens=tokens, cols=cols, rows=rows, qtype=qtype, parts=parts, bias=bias)


def listed() -> List[Dict[str, Any]]:
    return [
        # A single user's decode: one token a step, the layer captured in a HIP graph as a
        # serving loop does; eight steps on eight tokens, so each reads its own experts.
        dict(_moe("qwen3_30b_a3b", 1, steps=8, graph=True), name="moe_decode_1"),
        # A speculative verify step, or eight users: called eagerly.
        dict(_moe("qwen3_30b_a3b", 8), name="moe_decode_8"),
        # Batched serving: 32 users' decode step.
        dict(_moe("qwen3_30b_a3b", 32), name="moe_batch_32"),
        # A chunk of a prompt beside running decodes, of no round size; some experts are
        # asked for far more than others.
        dict(_moe("qwen3_30b_a3b", 301, skew=True), name="moe_chunk_301"),
        # A whole prompt.
        dict(_moe("qwen3_30b_a3b", 4096, skew=True), name="moe_prompt_4096"),
        # Few, wide experts: 24 users.
        dict(_moe("mixtral_8x7b", 24), name="moe_wide_batch_24"),
        # 8-bit experts with a gated shared expert: a small chunk.
        dict(_moe("qwen2_57b_a14b", 100), name="moe_shared_100"),
        # The dense FFN of an 8B-class model: a batch of decodes and a prompt.
        dict(_dense(20), name="ffn_batch_20"),
        dict(_dense(1500), name="ffn_prompt_1500"),
        # Its attention input projections, q | k | v packed, for a batch of decodes.
        dict(_linear(33, 4096, 6144, "q4_k", parts=3), name="qkv_batch_33"),
        # The output head of a decode step: the largest single matrix.
        dict(_linear(1, 2048, 151936, "q6_k"), name="head_1"),
        # The residual add and norm in front of a block, for a batch of decodes.
        dict(kind="norm", tokens=16, hidden=2048, name="norm_16"),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> Dict[str, Any]:
    kind = rng.choice(["moe", "moe", "moe", "dense", "linear", "linear", "norm"])
    if kind == "moe":
        shape = rng.choice(["qwen3_30b_a3b", "qwen3_30b_a3b", "mixtral_8x7b", "qwen2_57b_a14b"])
        tokens = _log_int(rng, 1, {"qwen3_30b_a3b": 4096, "mixtral_8x7b": 400, "qwen2_57b_a14b": 250}[shape])
        graph = tokens <= 8 and rng.random() < 0.5
        return _moe(shape, tokens, steps=rng.choice([2, 4]) if graph else 1, graph=graph,
                    skew=tokens > 64 and rng.random() < 0.5)
    if kind == "dense":
        hidden, inter = rng.choice([(4096, 12288), (2048, 5632), (1024, 2816)])
        gate_up, down = rng.choice([("q4_k", "q6_k"), ("q8_0", "q8_0"), ("q5_k", "q6_k"), ("q4_k", "q4_k")])
        return _dense(_log_int(rng, 1, 1500), hidden, inter, gate_up, down)
    if kind == "linear":
        cols, rows, parts = rng.choice([(4096, 6144, 3), (2048, 5120, 3), (4096, 4096, 1), (2048, 1024, 1),
                                        (2048, 151936, 1), (3584, 3584, 1)])
        tokens = _log_int(rng, 1, 64 if rows > 100000 else 2048)
        return _linear(tokens, cols, rows, rng.choice(["q4_k", "q6_k", "q8_0", "q5_k"]), parts, rng.random() < 0.3)
    return dict(kind="norm", tokens=_log_int(rng, 1, 4096), hidden=rng.choice([1024, 2048, 3584, 4096]))


# ------------------------------------------------------------------ block formats
# Quantisers and decoders of the GGUF block formats as ggml defines them, on flat tensors
# whose length is a whole number of blocks.
def _half_bytes(v: torch.Tensor) -> torch.Tensor:
    """fp16 values [n] as bytes [n, 2]."""
    return v.to(torch.float16).reshape(-1, 1).view(torch.uint8)


def _bytes_half(b: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    return b.contiguous().view(torch.float16).to(dtype)


def _div(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    return torch.where(b > 0, a / b.clamp_min(1e-30), torch.zeros_like(a))


def _quant_k45(w: torch.Tensor, levels: int) -> torch.Tensor:
    """Q4_K (levels 15) and Q5_K (31): 8 sub-blocks of 32, 6-bit scales and minima."""
    v = w.reshape(-1, 8, 32)
    lo = v.amin(2).clamp_max(0.0)
    step = (v.amax(2).clamp_min(0.0) - lo) / levels
    d = (step.amax(1) / 63).to(torch.float16).float()
    dmin = ((-lo).amax(1) / 63).to(torch.float16).float()
    sc = _div(step, d[:, None].expand_as(step)).round_().clamp_(0, 63)
    mn = _div(-lo, dmin[:, None].expand_as(lo)).round_().clamp_(0, 63)
    a, z = (d[:, None] * sc)[..., None], (dmin[:, None] * mn)[..., None]
    q = _div(v + z, a.expand_as(v)).round_().clamp_(0, levels).to(torch.uint8)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    packed = torch.cat([sc[:, :4] | ((sc[:, 4:] >> 4) << 6), mn[:, :4] | ((mn[:, 4:] >> 4) << 6),
                        (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)
    low = q & 15
    qs = (low[:, 0::2] | (low[:, 1::2] << 4)).reshape(-1, 128)
    out = [_half_bytes(d), _half_bytes(dmin), packed]
    if levels == 31:
        qh = torch.zeros(q.shape[0], 32, dtype=torch.uint8, device=w.device)
        for s in range(8):
            qh |= (q[:, s] >> 4) << s
        out.append(qh)
    return torch.cat(out + [qs], 1).reshape(-1)


def _dequant_k45(raw: torch.Tensor, levels: int, dtype: torch.dtype) -> torch.Tensor:
    b = raw.reshape(-1, 144 if levels == 15 else 176)
    d, dmin = _bytes_half(b[:, 0:2], dtype), _bytes_half(b[:, 2:4], dtype)
    s = b[:, 4:16]
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).to(dtype)
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).to(dtype)
    qs = b[:, -128:].reshape(-1, 4, 32)
    q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
    if levels == 31:
        q = q | torch.stack([((b[:, 16:48] >> i) & 1) << 4 for i in range(8)], 1)
    return ((d * sc)[..., None] * q.to(dtype) - (dmin * mn)[..., None]).reshape(-1)


def _quant_q6(w: torch.Tensor) -> torch.Tensor:
    v = w.reshape(-1, 16, 16)
    step = v.abs().amax(2) / 31
    d = (step.amax(1) / 127).to(torch.float16).float()
    sc = _div(step, d[:, None].expand_as(step)).round_().clamp_(0, 127)
    q = _div(v, (d[:, None] * sc)[..., None].expand_as(v)).round_().clamp_(-32, 31).add_(32).to(torch.uint8)
    q = q.reshape(-1, 2, 4, 32)  # 128-weight half, quarter of it, weight
    ql = torch.cat([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
    h = q >> 4
    qh = h[:, :, 0] | (h[:, :, 1] << 2) | (h[:, :, 2] << 4) | (h[:, :, 3] << 6)
    return torch.cat([ql.reshape(-1, 128), qh.reshape(-1, 64), sc.to(torch.uint8), _half_bytes(d)], 1).reshape(-1)


def _dequant_q6(raw: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    b = raw.reshape(-1, 210)
    ql, qh = b[:, :128].reshape(-1, 2, 64), b[:, 128:192].reshape(-1, 2, 32)
    sc = b[:, 192:208].contiguous().view(torch.int8).to(dtype)
    q = torch.stack([(ql[:, :, :32] & 15) | ((qh & 3) << 4), (ql[:, :, 32:] & 15) | (((qh >> 2) & 3) << 4),
                     (ql[:, :, :32] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 32:] >> 4) | ((qh >> 6) << 4)], 2)
    d = _bytes_half(b[:, 208:210], dtype)
    return ((d * sc)[..., None] * (q.to(dtype) - 32).reshape(-1, 16, 16)).reshape(-1)


def _quant(qtype: str, w: torch.Tensor) -> torch.Tensor:
    """float32 weights on the device -> their GGUF bytes (uint8, flat)."""
    w = w.reshape(-1)
    if qtype == "f16":
        return w.to(torch.float16).view(torch.uint8)
    if qtype == "q8_0":
        v = w.reshape(-1, 32)
        d = (v.abs().amax(1) / 127).to(torch.float16)
        q = _div(v, d.float()[:, None].expand_as(v)).round_().clamp_(-127, 127).to(torch.int8)
        return torch.cat([_half_bytes(d), q.view(torch.uint8)], 1).reshape(-1)
    return _quant_q6(w) if qtype == "q6_k" else _quant_k45(w, 15 if qtype == "q4_k" else 31)


def _dequant(qtype: str, raw: torch.Tensor, rows: int, cols: int, dtype: torch.dtype = torch.float64) -> torch.Tensor:
    if qtype == "f16":
        v = raw.view(torch.float16).to(dtype)
    elif qtype == "q8_0":
        b = raw.reshape(-1, 34)
        v = (_bytes_half(b[:, :2], dtype) * b[:, 2:].contiguous().view(torch.int8).to(dtype)).reshape(-1)
    elif qtype == "q6_k":
        v = _dequant_q6(raw, dtype)
    else:
        v = _dequant_k45(raw, 15 if qtype == "q4_k" else 31, dtype)
    return v.reshape(rows, cols)


# ------------------------------------------------------------------ inputs
class _Draw:
    """Seeded device tensors in a fixed order."""

    def __init__(self, seed: int) -> None:
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.gen = torch.Generator(device=self.dev).manual_seed(seed)

    def normal(self, *shape: int) -> torch.Tensor:
        return torch.randn(*shape, generator=self.gen, device=self.dev)

    def matrices(self, qtype: str, n: int, rows: int, cols: int) -> torch.Tensor:
        """GGUF bytes of n normal [rows, cols] matrices (std 0.02), [n, bytes a matrix]."""
        per = int(rows * cols * _BITS[qtype] / 8)
        out = torch.empty(n, per, dtype=torch.uint8, device=self.dev)
        step = max(1, (1 << 28) // (rows * cols))
        for i in range(0, n, step):
            m = min(step, n - i)
            out[i:i + m] = _quant(qtype, self.normal(m, rows, cols).mul_(0.02)).reshape(m, per)
        return out


def _moe_inputs(case: Dict[str, Any], seed: int) -> Tuple[Dict[str, Any], Dict[str, torch.Tensor]]:
    sp, d = _MOE[case["shape"]], _Draw(seed)
    H, E, I, S = sp["hidden"], sp["experts"], sp["inter"], sp["shared"]
    t = {"router": d.normal(E, H).mul_(0.02)}
    x = d.normal(case["steps"] * case["tokens"], H)
    if case["skew"]:
        # all tokens share a direction that the router's rows read with Zipf-like strengths,
        # so the experts' loads fall off as those of a trained router do
        u = F.normalize(d.normal(H), dim=0)
        rank = torch.argsort(d.normal(E)).float() + 1
        x += 4.0 * u
        t["router"] += (-1.1 * torch.log(rank) / 4.0)[:, None] * u
    t["x"] = x.to(torch.float16)
    t["gate"] = d.matrices(sp["gate_up"], E, I, H)
    t["up"] = d.matrices(sp["gate_up"], E, I, H)
    t["down"] = d.matrices(sp["down"], E, H, I)
    if S:
        t["sh_gate"] = d.matrices(sp["gate_up"], 1, S, H)
        t["sh_up"] = d.matrices(sp["gate_up"], 1, S, H)
        t["sh_down"] = d.matrices(sp["down"], 1, H, S)
        t["sh_inp"] = d.normal(H).mul_(0.02)
    return sp, t


def _dense_inputs(case: Dict[str, Any], seed: int) -> Dict[str, torch.Tensor]:
    d, H, I = _Draw(seed), case["hidden"], case["inter"]
    return {"x": d.normal(case["tokens"], H).to(torch.float16), "gate": d.matrices(case["gate_up"], 1, I, H),
            "up": d.matrices(case["gate_up"], 1, I, H), "down": d.matrices(case["down"], 1, H, I)}


def _linear_rows(case: Dict[str, Any]) -> List[int]:
    """Output rows of each packed projection: one, or q | k | v with few key / value heads."""
    n = case["rows"]
    return [n] if case["parts"] == 1 else [n - 2 * (n // 6 // 64 * 64)] + [n // 6 // 64 * 64] * 2


def _linear_inputs(case: Dict[str, Any], seed: int) -> Dict[str, Any]:
    d = _Draw(seed)
    out: Dict[str, Any] = {"x": d.normal(case["tokens"], case["cols"]).to(torch.float16)}
    out["w"] = [d.matrices(case["qtype"], 1, n, case["cols"])[0] for n in _linear_rows(case)]
    out["bias"] = [d.normal(n).to(torch.float16).float() if case["bias"] else None for n in _linear_rows(case)]
    return out


def _norm_inputs(case: Dict[str, Any], seed: int) -> Dict[str, torch.Tensor]:
    d, R, D = _Draw(seed), case["tokens"], case["hidden"]
    return {"x": d.normal(R, D) * 3.0, "delta": d.normal(R, D), "w": d.normal(D).mul_(0.1).add_(1.0)}


def _host(t: torch.Tensor) -> np.ndarray:
    """Bytes as a loader hands them over: host memory (page-locked, for the upload)."""
    h = torch.empty(t.shape, dtype=t.dtype, pin_memory=True)
    h.copy_(t)
    return h.numpy()


# ------------------------------------------------------------------ prepare and run
def _prepare_moe(case: Dict[str, Any], seed: int) -> Callable[[], Any]:
    sp, t = _moe_inputs(case, seed)
    H, E, I, S, arch = sp["hidden"], sp["experts"], sp["inter"], sp["shared"], sp["arch"]
    g = pgmoe.InMemoryGGUF({
        "general.architecture": arch, f"{arch}.embedding_length": H, f"{arch}.expert_count": E,
        f"{arch}.expert_used_count": sp["top_k"], f"{arch}.expert_feed_forward_length": I,
        f"{arch}.expert_weights_norm": sp["norm_topk"], f"{arch}.expert_shared_feed_forward_length": S})
    gu, dn = _TYPES[sp["gate_up"]], _TYPES[sp["down"]]
    g.add_tensor("blk.0.ffn_gate_inp.weight", (E, H), 0, _host(t["router"]))
    g.add_tensor("blk.0.ffn_gate_exps.weight", (E, I, H), gu, _host(t["gate"]))
    g.add_tensor("blk.0.ffn_up_exps.weight", (E, I, H), gu, _host(t["up"]))
    g.add_tensor("blk.0.ffn_down_exps.weight", (E, H, I), dn, _host(t["down"]))
    if S:
        g.add_tensor("blk.0.ffn_gate_shexp.weight", (S, H), gu, _host(t["sh_gate"]))
        g.add_tensor("blk.0.ffn_up_shexp.weight", (S, H), gu, _host(t["sh_up"]))
        g.add_tensor("blk.0.ffn_down_shexp.weight", (H, S), dn, _host(t["sh_down"]))
        g.add_tensor("blk.0.ffn_gate_inp_shexp.weight", (H,), 0, _host(t["sh_inp"]))
    dev = t["x"].device
    layer = pgmoe.HipSparseMoEMLP(g, g.build_model_config(), 0, dev)
    xs = list(t["x"].split(case["tokens"]))
    del t, g
    if not case["graph"]:
        return lambda: [layer(x) for x in xs]
    side = torch.cuda.Stream(dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        layer(xs[0])  # the stream's workspace, outside the capture
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        outs = [layer(x) for x in xs]

    def replay(layer=layer, xs=xs) -> Any:  # the graph reads the layer's and the tokens' memory
        graph.replay()
        return outs

    return replay


def _prepare_dense(case: Dict[str, Any], seed: int) -> Callable[[], Any]:
    t, H, I = _dense_inputs(case, seed), case["hidden"], case["inter"]
    g = pgmoe.InMemoryGGUF({"general.architecture": "qwen3", "qwen3.embedding_length": H,
                            "qwen3.feed_forward_length": I})
    gu, dn = _TYPES[case["gate_up"]], _TYPES[case["down"]]
    g.add_tensor("blk.0.ffn_gate.weight", (I, H), gu, _host(t["gate"]))
    g.add_tensor("blk.0.ffn_up.weight", (I, H), gu, _host(t["up"]))
    g.add_tensor("blk.0.ffn_down.weight", (H, I), dn, _host(t["down"]))
    x = t["x"]
    ffn = pgmoe.HipDenseMLP.from_gguf(g, g.build_model_config(), 0, x.device)
    return lambda: ffn(x)


def _prepare_linear(case: Dict[str, Any], seed: int) -> Callable[[], Any]:
    t, qt = _linear_inputs(case, seed), case["qtype"]
    x = t["x"]
    mode = "w4" if qt == "q4_k" else "w8"
    lins = [pgmoe.GGUFQuantLinear(mode, case["cols"], n, _TYPES[qt], raw=_host(w), bias=b, device=x.device)
            for n, w, b in zip(_linear_rows(case), t["w"], t["bias"])]
    if case["parts"] == 1:
        return lambda: lins[0](x)
    pack = pgmoe.FusedLinearPack(lins)
    return lambda: pack(x)


def _prepare_norm(case: Dict[str, Any], seed: int) -> Callable[[], Any]:
    t = _norm_inputs(case, seed)
    norm = pgmoe.GGUFRMSNorm(t["w"], 1e-6)
    return lambda: norm.forward_with_residual(t["x"], t["delta"])


def prepare(case: Dict[str, Any], seed: int) -> Callable[[], Any]:
    make = {"moe": _prepare_moe, "dense": _prepare_dense, "linear": _prepare_linear, "norm": _prepare_norm}
    return make[case["kind"]](case, seed)


def run(state: Callable[[], Any]) -> Any:
    return state()


# ------------------------------------------------------------------ work, tolerance, exact
def work(case: Dict[str, Any]) -> Dict[str, float]:
    M = case["tokens"]
    if case["kind"] == "moe":
        sp = _MOE[case["shape"]]
        H, E, K, I, S = sp["hidden"], sp["experts"], sp["top_k"], sp["inter"], sp["shared"]
        active = E * (1.0 - (1.0 - K / E) ** M)  # experts that M tokens of an even routing reach
        per = H * (2 * _BITS[sp["gate_up"]] + _BITS[sp["down"]]) / 8
        nbytes = active * I * per + S * per + 4 * E * H + (4 * H if S else 0) + M * H * 6
        flops = 2.0 * M * H * (3 * K * I + 3 * S + E)
        return {"bytes": case["steps"] * nbytes, "flops": case["steps"] * flops}
    if case["kind"] == "dense":
        H, I = case["hidden"], case["inter"]
        return {"bytes": H * I * (2 * _BITS[case["gate_up"]] + _BITS[case["down"]]) / 8 + M * H * 6,
                "flops": 6.0 * M * H * I}
    if case["kind"] == "linear":
        N, K = case["rows"], case["cols"]
        return {"bytes": N * K * _BITS[case["qtype"]] / 8 + 2 * M * (N + K), "flops": 2.0 * M * N * K}
    D = case["hidden"]
    return {"bytes": M * D * (4 + 4 + 4 + 2) + 4 * D, "flops": 6.0 * M * D}


def tolerance(case: Dict[str, Any]) -> Dict[str, float]:
    """About four times the error measured against `exact`: 4.2e-4 for batches (fp16 weights
    and rows in the matrix products), 3.5e-5 for decode FFNs (32-bit sums and rows), 2.9e-4
    and 2.1e-4 for fp16 outputs of linears and norms.  Each error is near normal, so the
    largest of some million values lies near 6 of its deviations."""
    if case["kind"] in ("moe", "dense"):
        return {"rel": 1.5e-4, "max": 1e-3} if case["tokens"] <= 8 else {"rel": 1.7e-3, "max": 1e-2}
    return {"rel": 1.2e-3, "max": 8e-3} if case["kind"] == "linear" else {"rel": 8.5e-4, "max": 4e-3}


def _ffn64(x: torch.Tensor, gate: torch.Tensor, up: torch.Tensor, down: torch.Tensor) -> torch.Tensor:
    return (F.silu(x @ gate.T) * (x @ up.T)) @ down.T


def _exact_moe(case: Dict[str, Any], seed: int) -> List[torch.Tensor]:
    sp, t = _moe_inputs(case, seed)
    H, E, K, I, S = sp["hidden"], sp["experts"], sp["top_k"], sp["inter"], sp["shared"]
    gu, dn = sp["gate_up"], sp["down"]
    x = t["x"].double()
    p = torch.softmax(x @ t["router"].double().T, dim=-1)
    w, idx = torch.topk(p, K, dim=-1)
    if sp["norm_topk"]:
        w = w / w.sum(-1, keepdim=True)
    out = torch.zeros_like(x)
    for e in range(E):
        tok, slot = torch.where(idx == e)
        if tok.numel():
            y = _ffn64(x[tok], _dequant(gu, t["gate"][e], I, H), _dequant(gu, t["up"][e], I, H),
                       _dequant(dn, t["down"][e], H, I))
            out.index_add_(0, tok, y * w[tok, slot, None])
    if S:
        y = _ffn64(x, _dequant(gu, t["sh_gate"][0], S, H), _dequant(gu, t["sh_up"][0], S, H),
                   _dequant(dn, t["sh_down"][0], H, S))
        out += torch.sigmoid(x @ t["sh_inp"].double())[:, None] * y
    return list(out.split(case["tokens"]))


def exact(case: Dict[str, Any], seed: int) -> Optional[Any]:
    if case["kind"] == "moe":
        return _exact_moe(case, seed)
    if case["kind"] == "dense":
        t, H, I = _dense_inputs(case, seed), case["hidden"], case["inter"]
        return _ffn64(t["x"].double(), _dequant(case["gate_up"], t["gate"][0], I, H),
                      _dequant(case["gate_up"], t["up"][0], I, H), _dequant(case["down"], t["down"][0], H, I))
    if case["kind"] == "linear":
        t, outs = _linear_inputs(case, seed), []
        for n, w, b in zip(_linear_rows(case), t["w"], t["bias"]):
            y = t["x"].double() @ _dequant(case["qtype"], w, n, case["cols"]).T
            outs.append(y if b is None else y + b.double())
        return outs[0] if case["parts"] == 1 else outs
    t = _norm_inputs(case, seed)
    h = t["x"].double() + t["delta"].double()
    return h, h * torch.rsqrt(h.square().mean(-1, keepdim=True) + 1e-6) * t["w"].double()
