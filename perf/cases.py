"""The work whose speed this framework is judged by: layers and blocks of LLM inference through its
public entry points (hipinfer_amd.hipinfer), over the shapes its tests, benchmark and README name.

A case is a dict of plain values; `kind` selects one of the builders below:

  gemv           one eager decode projection (no graph): the smallest call there is
  decode_mlp     the MLP half of `layers` decode layers (embed, fused-norm gate/up + SwiGLU, down +
                 residual), 1-8 rows, captured once in a graph and replayed, as a decode loop does
  decode_attn    the attention half of `layers` decode layers (embed, fused-norm QKV + RoPE + cache
                 write, decode attention, o + residual), 1-8 sequences, as a graph
  batched        one whole decode layer for 9-64 sequences of mixed lengths on the GEMM path, as a graph
  prefill_attn   the attention block of one prefill layer (QKV GEMM, RoPE + cache, flash attention,
                 o GEMM + residual + the next norm), eager
  prefill_mlp    the MLP block of one prefill layer (gate/up GEMM + SwiGLU, down GEMM + residual +
                 the next norm), eager
  flash          causal attention of one prompt chunk over a cache slot, with its log-sum-exp
  moe            one mixture-of-experts layer for M tokens: router, experts, combine
  engine         a whole model from a weight file: a prompt's logits, then one decode step

Residual blocks start from an embedding gather, as a model does, so a repeated pass starts from the
same rows. Weights are N(0, 0.02) (int8: rounded normals with one fp16 scale per row), activations
and cached keys and values N(0, 1), norm weights near 1.
"""
import math
import os
import tempfile

import numpy as np
import torch

from hipinfer_amd import hipinfer as hi
from hipinfer_amd import weights as wfile

EPS = 1e-5
EMBED_ROWS = 512  # rows of the embedding table a block gathers its residual stream from

# hidden, q heads, kv heads, head dim, MLP width, QKV bias
MODELS = {
    "tinyllama": (2048, 32, 4, 64, 5632, False),
    "qwen25_1p5b": (1536, 12, 2, 128, 8960, True),
    "llama32_3b": (3072, 24, 8, 128, 8192, False),
    "llama31_8b": (4096, 32, 8, 128, 14336, False),
}


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one output projection of a 1B model, called eagerly: launch and latency are all there is
        {"name": "gemv_o_int8", "kind": "gemv", "rows": 1, "n": 2048, "k": 2048, "int8": True, "epi": 0, "norm": False},
        # batch-1 decode, the bulk of a token's weight traffic, fp16 weights
        {"name": "decode_mlp_8b", "kind": "decode_mlp", "model": "llama31_8b", "rows": 1, "layers": 4, "int8": False},
        # batch-1 decode of a quantised model deep into a long conversation
        {"name": "decode_attn_8b_int8_4k", "kind": "decode_attn", "model": "llama31_8b", "rows": 1, "layers": 4,
         "int8": True, "ctx_lo": 4001, "ctx_hi": 4001},
        # five rows: the width of a 4-token speculative verification, ragged K, int8
        {"name": "verify_mlp_qwen_int8_r5", "kind": "decode_mlp", "model": "qwen25_1p5b", "rows": 5, "layers": 8,
         "int8": True},
        # continuous batching: one layer of a step over 48 sequences of 100 to 2000 tokens
        {"name": "batched_8b_b48", "kind": "batched", "model": "llama31_8b", "rows": 48, "int8": False, "ctx_lo": 100,
         "ctx_hi": 2000},
        # an ordinary prompt, not a multiple of any tile
        {"name": "prefill_attn_3b_t1000", "kind": "prefill_attn", "model": "llama32_3b", "rows": 1000, "p0": 0,
         "int8": False},
        # a short prompt of a quantised model, odd length
        {"name": "prefill_mlp_qwen_int8_t333", "kind": "prefill_mlp", "model": "qwen25_1p5b", "rows": 333, "int8": True},
        # a long prompt's chunk: the largest matrix products
        {"name": "prefill_mlp_8b_t2048", "kind": "prefill_mlp", "model": "llama31_8b", "rows": 2048, "int8": False},
        # a chunk far into a long prompt
        {"name": "flash_8b_t2048_p4096", "kind": "flash", "model": "llama31_8b", "rows": 2048, "p0": 4096},
        # one token through a fine-grained mixture of experts (32 experts, 8 chosen)
        {"name": "moe_b1", "kind": "moe", "rows": 1, "experts": 32, "top_k": 8, "hidden": 1024, "inter": 512},
        # a prompt through the same layer
        {"name": "moe_t700", "kind": "moe", "rows": 700, "experts": 32, "top_k": 8, "hidden": 1024, "inter": 512},
        # the whole path a server calls: prompt logits in two chunks, then a 4-sequence decode step
        {"name": "engine_tinyllama_t777", "kind": "engine", "model": "tinyllama", "layers": 4, "vocab": 32000,
         "rows": 777, "chunk": 512, "batch": 4, "int8": False},
    ]


def _log(rng, lo, hi, multiple=1):
    """A whole number spread over the logarithm of [lo, hi]."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))
    return max(lo, min(hi, int(v) // multiple * multiple))


def draw(rng):
    kind = rng.choice(["gemv", "decode_mlp", "decode_attn", "batched", "prefill_attn", "prefill_mlp", "flash", "moe",
                       "engine"])
    model = rng.choice(sorted(MODELS))
    int8 = rng.random() < 0.5
    if kind == "gemv":
        k = _log(rng, 1024, 8192, 32)
        return {"kind": kind, "rows": rng.randint(1, 8), "n": _log(rng, 1024, 32768, 32), "k": k, "int8": int8,
                "epi": rng.choice([0, 2]), "norm": rng.random() < 0.5}
    if kind == "decode_mlp":
        return {"kind": kind, "model": model, "rows": rng.choice([1, 1, rng.randint(2, 8)]), "layers": rng.randint(2, 4),
                "int8": int8}
    if kind == "decode_attn":
        hi_ = _log(rng, 64, 6000)
        return {"kind": kind, "model": model, "rows": rng.choice([1, 1, rng.randint(2, 8)]), "layers": rng.randint(2, 4),
                "int8": int8, "ctx_lo": max(1, hi_ - rng.randint(0, hi_ // 2)), "ctx_hi": hi_}
    if kind == "batched":
        hi_ = _log(rng, 100, 2000)
        return {"kind": kind, "model": model, "rows": rng.randint(9, 64), "int8": int8, "ctx_lo": max(1, hi_ // 8),
                "ctx_hi": hi_}
    if kind == "prefill_attn":
        return {"kind": kind, "model": model, "rows": _log(rng, 32, 2048), "p0": rng.choice([0, 0, rng.randint(1, 2048)]),
                "int8": int8}
    if kind == "prefill_mlp":
        return {"kind": kind, "model": model, "rows": _log(rng, 32, 2048), "int8": int8}
    if kind == "flash":
        return {"kind": kind, "model": model, "rows": _log(rng, 32, 2048), "p0": rng.choice([0, rng.randint(1, 4096)])}
    if kind == "moe":
        E, k, H, I = rng.choice([(32, 8, 1024, 512), (8, 2, 1024, 2048), (64, 6, 2048, 768)])
        return {"kind": kind, "rows": rng.choice([1, rng.randint(2, 8), _log(rng, 9, 2048)]), "experts": E, "top_k": k,
                "hidden": H, "inter": I}
    return {"kind": "engine", "model": "tinyllama", "layers": rng.randint(1, 4), "vocab": _log(rng, 2048, 32000, 32),
            "rows": _log(rng, 20, 900), "chunk": rng.choice([256, 512, 1024]), "batch": rng.randint(1, 6), "int8": int8}


# ------------------------------------------------------------------ inputs
class _Gen:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)
        self.cpu = torch.Generator()
        self.cpu.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return (torch.randn(*shape, device="cuda", generator=self.g) * std).half()

    def norm_weight(self, n):
        return (1.0 + 0.1 * torch.randn(n, device="cuda", generator=self.g)).half()

    def weight(self, n, k, int8, std=0.02):
        """A projection [n, k]: (fp16, None), or (int8, fp16 row scales)."""
        w = torch.randn(n, k, device="cuda", generator=self.g)
        if not int8:
            return (w * std).half(), None
        q = (w * 32.0).round().clamp(-127, 127).to(torch.int8)
        s = ((0.9 + 0.2 * torch.rand(n, device="cuda", generator=self.g)) * (std / 32.0)).half()
        return q, s

    def ints(self, lo, hi_, n):
        """n whole numbers of [lo, hi_] as a host list."""
        return torch.randint(lo, hi_ + 1, (n,), generator=self.cpu).tolist()


def _rope_table(max_seq, D, theta=500000.0):
    inv = 1.0 / theta ** (torch.arange(0, D, 2, device="cuda", dtype=torch.float64) / D)
    a = torch.arange(max_seq, device="cuda", dtype=torch.float64)[:, None] * inv[None, :]
    return torch.stack([a.cos(), a.sin()], -1).half().contiguous()


def _round_up(n, m):
    return (n + m - 1) // m * m


def _inputs(c, seed):
    """Everything of the case that both prepare() and exact() need, from the seed alone."""
    g, k = _Gen(seed), c["kind"]
    s = {"c": c}
    if k == "gemv":
        s["x"] = g.normal(c["rows"], c["k"])
        s["nw"] = g.norm_weight(c["k"]) if c["norm"] else None
        s["w"] = g.weight(c["n"], c["k"], c["int8"])
        return s
    if k == "moe":
        M, E, H, I = c["rows"], c["experts"], c["hidden"], c["inter"]
        s["xn"], s["x0"] = g.normal(M, H), g.normal(EMBED_ROWS, H)
        s["wr"] = g.normal(E, H, std=0.05)
        s["wgu"] = g.normal(E, 2 * I, H, std=0.03)
        s["wdown"] = g.normal(E, H, I, std=0.03)
        s["tok"] = torch.tensor(g.ints(0, EMBED_ROWS - 1, M), dtype=torch.int32, device="cuda")
        return s
    H, Hq, Hkv, D, I, bias = MODELS[c["model"]]
    if k == "flash":
        T, S = c["rows"], _round_up(c["p0"] + c["rows"], 256)
        s["q"], s["kc"], s["vc"] = g.normal(T, Hq * D), g.normal(Hkv, S, D), g.normal(Hkv, S, D)
        return s
    if k == "engine":
        V = c["vocab"]
        s["embed"], s["nf"], s["lm"] = g.normal(V, H), g.norm_weight(H), g.weight(V, H, c["int8"])
        s["inv_freq"] = (1.0 / 10000.0 ** (np.arange(0, D, 2) / D)).astype(np.float32)
        s["layers"] = [{"n1": g.norm_weight(H), "qkv": g.weight((Hq + 2 * Hkv) * D, H, c["int8"]),
                        "o": g.weight(H, Hq * D, c["int8"]), "n2": g.norm_weight(H),
                        "gu": g.weight(2 * I, H, c["int8"]), "down": g.weight(H, I, c["int8"])}
                       for _ in range(c["layers"])]
        # slot 0 holds the measured prompt; the others shorter ones, already in the cache
        s["prompts"] = [g.ints(0, V - 1, c["rows"])] + [g.ints(0, V - 1, n) for n in g.ints(5, 60, c["batch"] - 1)]
        s["next"] = g.ints(0, V - 1, c["batch"])
        return s
    M = c["rows"]
    s["table"] = g.normal(EMBED_ROWS, H)
    s["tok"] = torch.tensor(g.ints(0, EMBED_ROWS - 1, M), dtype=torch.int32, device="cuda")
    layers = c.get("layers", 1)
    s["layers"] = []
    for _ in range(layers):
        ly = {"n1": g.norm_weight(H), "n2": g.norm_weight(H)}
        if k in ("decode_attn", "batched", "prefill_attn"):
            ly["qkv"] = g.weight((Hq + 2 * Hkv) * D, H, c["int8"])
            ly["bqkv"] = g.normal((Hq + 2 * Hkv) * D, std=0.1) if bias else None
            ly["o"] = g.weight(H, Hq * D, c["int8"])
        if k in ("decode_mlp", "batched", "prefill_mlp"):
            ly["gu"] = g.weight(2 * I, H, c["int8"])
            ly["down"] = g.weight(H, I, c["int8"])
        s["layers"].append(ly)
    if k in ("decode_attn", "batched"):
        S = _round_up(c["ctx_hi"] + 1, 64)
        s["pos_list"] = g.ints(c["ctx_lo"] - 1, c["ctx_hi"] - 1, M)
        s["pos"] = torch.tensor(s["pos_list"], dtype=torch.int32, device="cuda")
        slots = M
    elif k == "prefill_attn":
        S, slots = _round_up(c["p0"] + M, 64), 1
    if k in ("decode_attn", "batched", "prefill_attn"):
        s["cs"] = _rope_table(S, D)
        for ly in s["layers"]:
            ly["kc"], ly["vc"] = g.normal(slots, Hkv, S, D), g.normal(slots, Hkv, S, D)
    return s


# ------------------------------------------------------------------ what a program keeps
def _capture(step):
    """The step as a graph: one eager pass first (it chooses the GEMM tiles), then the capture."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    return graph


def prepare(case, seed):
    s = _inputs(case, seed)
    k = case["kind"]
    half = dict(dtype=torch.float16, device="cuda")
    if k in ("gemv", "flash"):
        return s
    if k == "moe":
        s["x"] = torch.empty(case["rows"], case["hidden"], **half)
        return s
    H, Hq, Hkv, D, I, _ = MODELS[case["model"]]
    if k == "engine":
        s["engine"] = _engine(case, s)
        for name in ("embed", "nf", "lm", "layers"):
            del s[name]
        return s
    M = case["rows"]
    s["x"], s["act"] = torch.empty(M, H, **half), torch.empty(M, I, **half)
    s["xn"] = torch.empty(M, H, **half)
    s["qkv"] = torch.empty(M, (Hq + 2 * Hkv) * D, **half)
    s["q"], s["att"] = torch.empty(M, Hq * D, **half), torch.empty(M, Hq * D, **half)
    if k in ("decode_attn", "batched"):
        s["work"] = torch.zeros(hi.lib.hi_decode_work_bytes(M, Hq, Hkv, D), dtype=torch.uint8, device="cuda")
    if k == "decode_mlp":
        s["graph"] = _capture(lambda: _decode_mlp(s))
    elif k == "decode_attn":
        s["graph"] = _capture(lambda: _decode_attn(s))
    elif k == "batched":
        s["graph"] = _capture(lambda: _batched(s))
    return s


def _decode_mlp(s):
    hi.embed(s["tok"], s["table"], out=s["x"])
    for ly in s["layers"]:
        hi.gemv(s["x"], ly["gu"][0], out=s["act"], normw=ly["n2"], eps=EPS, epi=2, scales=ly["gu"][1])
        hi.gemv(s["act"], ly["down"][0], out=s["x"], epi=1, scales=ly["down"][1])


def _decode_attn(s):
    _, Hq, Hkv, _, _, _ = MODELS[s["c"]["model"]]
    hi.embed(s["tok"], s["table"], out=s["x"])
    for ly in s["layers"]:
        hi.gemv_qkv_rope(s["x"], ly["qkv"][0], ly["n1"], Hq, Hkv, s["cs"], s["pos"], ly["kc"], ly["vc"], s["q"],
                         bias=ly["bqkv"], eps=EPS, scales=ly["qkv"][1])
        hi.decode_attn(s["q"], ly["kc"], ly["vc"], s["pos"], Hq, Hkv, out=s["att"], work=s["work"])
        hi.gemv(s["att"], ly["o"][0], out=s["x"], epi=1, scales=ly["o"][1])


def _batched(s):
    _, Hq, Hkv, D, _, _ = MODELS[s["c"]["model"]]
    ly = s["layers"][0]
    hi.embed(s["tok"], s["table"], out=s["x"])
    hi.rmsnorm(s["x"], ly["n1"], EPS, out=s["xn"])
    hi.gemm(s["xn"], ly["qkv"][0], out=s["qkv"], bias=ly["bqkv"], scales=ly["qkv"][1])
    hi.rope_cache(s["qkv"], Hq, Hkv, s["cs"], ly["kc"], ly["vc"], pos=s["pos"])
    hi.decode_attn(s["qkv"][:, :Hq * D], ly["kc"], ly["vc"], s["pos"], Hq, Hkv, out=s["att"], work=s["work"])
    hi.gemm_rmsnorm(s["att"], ly["o"][0], s["x"], ly["n2"], EPS, out=s["xn"], scales=ly["o"][1])
    hi.gemm(s["xn"], ly["gu"][0], out=s["act"], epi=2, scales=ly["gu"][1])
    hi.gemm_rmsnorm(s["act"], ly["down"][0], s["x"], ly["n1"], EPS, out=s["xn"], scales=ly["down"][1])


def _prefill_attn(s):
    c = s["c"]
    _, Hq, Hkv, D, _, _ = MODELS[c["model"]]
    ly = s["layers"][0]
    hi.embed(s["tok"], s["table"], out=s["x"])
    hi.rmsnorm(s["x"], ly["n1"], EPS, out=s["xn"])
    hi.gemm(s["xn"], ly["qkv"][0], out=s["qkv"], bias=ly["bqkv"], scales=ly["qkv"][1])
    hi.rope_cache(s["qkv"], Hq, Hkv, s["cs"], ly["kc"], ly["vc"], pos_base=c["p0"])
    hi.flash_prefill(s["qkv"][:, :Hq * D], ly["kc"][0], ly["vc"][0], c["rows"], c["p0"], Hq, Hkv, out=s["att"])
    hi.gemm_rmsnorm(s["att"], ly["o"][0], s["x"], ly["n2"], EPS, out=s["xn"], scales=ly["o"][1])


def _prefill_mlp(s):
    ly = s["layers"][0]
    hi.embed(s["tok"], s["table"], out=s["x"])
    hi.rmsnorm(s["x"], ly["n2"], EPS, out=s["xn"])
    hi.gemm(s["xn"], ly["gu"][0], out=s["act"], epi=2, scales=ly["gu"][1])
    hi.gemm_rmsnorm(s["act"], ly["down"][0], s["x"], ly["n1"], EPS, out=s["xn"], scales=ly["down"][1])


def _engine(case, s):
    H, Hq, Hkv, D, I, _ = MODELS[case["model"]]
    arr = lambda t: t.cpu().numpy()
    proj = lambda w: arr(w[0]) if w[1] is None else (arr(w[0]), arr(w[1]))
    W = {"inv_freq": s["inv_freq"], "embed": arr(s["embed"]), "final_norm": arr(s["nf"]), "lm_head": proj(s["lm"]),
         "layers": [{"attn_norm": arr(l["n1"]), "wqkv": proj(l["qkv"]), "wo": proj(l["o"]), "mlp_norm": arr(l["n2"]),
                     "wgu": proj(l["gu"]), "wdown": proj(l["down"])} for l in s["layers"]]}
    cfg = dict(vocab=case["vocab"], hidden=H, inter=I, layers=case["layers"], heads=Hq, kv_heads=Hkv, head_dim=D,
               max_pos=2048, eps=EPS)
    fd, path = tempfile.mkstemp(suffix=".hipi")
    os.close(fd)
    try:
        wfile.write_weights(path, cfg, W)
        eng = hi.Engine(path, max_batch=case["batch"], max_seq=2048, max_prefill=case["chunk"])
    finally:
        os.unlink(path)
    for slot in range(1, case["batch"]):
        eng.prefill(slot, s["prompts"][slot])
    return eng


# ------------------------------------------------------------------ one pass
def run(s):
    c = s["c"]
    k = c["kind"]
    if k == "gemv":
        return hi.gemv(s["x"], s["w"][0], normw=s["nw"], eps=EPS, epi=c["epi"], scales=s["w"][1])
    if k == "decode_mlp":
        s["graph"].replay()
        return s["x"]
    if k == "decode_attn":
        s["graph"].replay()
        return [s["x"]] + [ly[n] for ly in s["layers"] for n in ("kc", "vc")]
    if k == "batched":
        s["graph"].replay()
        return [s["x"], s["xn"], s["layers"][0]["kc"], s["layers"][0]["vc"]]
    if k == "prefill_attn":
        _prefill_attn(s)
        return [s["x"], s["xn"], s["layers"][0]["kc"], s["layers"][0]["vc"]]
    if k == "prefill_mlp":
        _prefill_mlp(s)
        return [s["x"], s["xn"]]
    if k == "flash":
        _, Hq, Hkv, _, _, _ = MODELS[c["model"]]
        return hi.flash_prefill_lse(s["q"], s["kc"], s["vc"], c["rows"], c["p0"], Hq, Hkv)
    if k == "moe":
        hi.embed(s["tok"], s["x0"], out=s["x"])
        idx, w = hi.moe_route_experts(s["xn"], s["wr"], s["wgu"], s["wdown"], c["top_k"], s["x"],
                                      hi.MOE_NORM_TOPK | hi.MOE_FP16_WEIGHTS, 0.22)
        return [s["x"], idx, w]
    eng = s["engine"]
    logits = eng.prefill_logits(0, s["prompts"][0])
    eng.set_state(s["next"], [len(p) for p in s["prompts"]])
    eng.decode(c["batch"], 1)
    return [logits, eng.logits(c["batch"])]


# ------------------------------------------------------------------ what a pass cannot do without
def _proj_bytes(n, k, int8):
    return n * k + 2 * n if int8 else 2 * n * k


def work(c):
    k = c["kind"]
    by = fl = 0.0
    if k == "gemv":
        M, n, kk = c["rows"], c["n"], c["k"]
        return {"bytes": _proj_bytes(n, kk, c["int8"]) + 2 * M * (kk + (n // 2 if c["epi"] == 2 else n)),
                "flops": 2.0 * M * n * kk}
    if k == "moe":
        M, E, K, H, I = c["rows"], c["experts"], c["top_k"], c["hidden"], c["inter"]
        hit = E * (1.0 - (1.0 - K / E) ** M)  # experts that some token chooses, for even routing
        return {"bytes": hit * 6 * H * I + 2 * E * H + 2 * M * 3 * H + 8 * M * K, "flops": 2.0 * M * (K * 3 * H * I + E * H)}
    H, Hq, Hkv, D, I, _ = MODELS[c["model"]]
    qd, q = (Hq + 2 * Hkv) * D, Hq * D
    M = c["rows"]
    if k == "flash":
        T, p0 = c["rows"], c["p0"]
        return {"bytes": 4.0 * T * q + 4.0 * (p0 + T) * Hkv * D + 4.0 * Hq * T,
                "flops": 4.0 * D * Hq * (T * p0 + T * (T + 1) / 2)}
    layers = c.get("layers", 1)
    attn_by = _proj_bytes(qd, H, c["int8"]) + _proj_bytes(H, q, c["int8"])
    mlp_by = _proj_bytes(2 * I, H, c["int8"]) + _proj_bytes(H, I, c["int8"])
    attn_fl, mlp_fl = 2.0 * H * (qd + q), 2.0 * H * 3 * I  # a row
    if k in ("decode_attn", "decode_mlp", "batched"):
        if k != "decode_mlp":
            ctx = (c["ctx_lo"] + c["ctx_hi"]) / 2
            by += layers * (attn_by + M * ctx * Hkv * D * 4)
            fl += layers * M * (attn_fl + 4.0 * ctx * q)
        if k != "decode_attn":
            by += layers * mlp_by
            fl += layers * M * mlp_fl
        return {"bytes": by + 4.0 * M * H, "flops": fl}
    if k == "prefill_attn":
        T, p0 = M, c["p0"]
        return {"bytes": attn_by + 6.0 * M * H + 4.0 * (p0 + 2 * T) * Hkv * D,
                "flops": M * attn_fl + 4.0 * q * (T * p0 + T * (T + 1) / 2)}
    if k == "prefill_mlp":
        return {"bytes": mlp_by + 6.0 * M * H, "flops": M * mlp_fl}
    # engine: each chunk streams the layers' weights once, the decode step once more, and the head
    V, T, B, L = c["vocab"], c["rows"], c["batch"], c["layers"]
    chunks = -(-T // c["chunk"])
    head = _proj_bytes(V, H, c["int8"])
    return {"bytes": (chunks + 1) * (L * (attn_by + mlp_by) + head) + 2.0 * (T + B) * V + 2.0 * (T + B) * H,
            "flops": (T + B) * (L * (attn_fl + mlp_fl) + 2.0 * V * H) + L * 4.0 * q * T * (T + 1) / 2}


def tolerance(c):
    # about four times what the outputs measure from the 64-bit results: fp16 outputs (2 to 4e-4) and,
    # in the blocks, the rounding of the fp16 intermediates (to 8e-4 through one block, 1.4e-3 through
    # the MLPs of several layers, 1.1e-3 through the engine's model). `max` holds the few new rows of
    # a cache that is otherwise the input: a few ulp of fp16.
    k = c["kind"]
    if k in ("gemv", "flash"):
        return {"rel": 1.5e-3, "max": 2e-2}
    if k == "moe":
        return {"rel": 1.5e-3, "max": 2e-2, "differ": 0.002}
    if k == "decode_mlp":
        return {"rel": 6e-3, "max": 5e-2}
    if k == "engine":
        return {"rel": 5e-3, "max": 5e-2}
    return {"rel": 3e-3, "max": 2e-2}


# ------------------------------------------------------------------ 64-bit results
def _w64(w):
    W, s = w
    return W.double() if s is None else W.double() * s.double()[:, None]


def _rms64(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w.double()


def _swiglu64(y):
    """Gate and up columns interleaved in groups of 16."""
    M, n = y.shape
    y = y.view(M, n // 32, 2, 16)
    return (torch.nn.functional.silu(y[:, :, 0]) * y[:, :, 1]).reshape(M, n // 2)


def _rope64(x, cos, sin):
    """x [M, heads, D], cos / sin [M, D/2]; pairs (d, d + D/2)."""
    a, b = x.chunk(2, -1)
    c, s = cos[:, None, :], sin[:, None, :]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attend64(q, K, V, first):
    """q [T, Hq, D] at positions first.., K / V [Hkv, n, D]: causal attention, and its base-2
    log-sum-exp [Hq, T]."""
    T, Hq, D = q.shape
    G, n = Hq // K.shape[0], K.shape[1]
    hidden = torch.arange(n, device=q.device)[None, :] > first + torch.arange(T, device=q.device)[:, None]
    out, lse = torch.empty_like(q), torch.empty(Hq, T, dtype=q.dtype, device=q.device)
    for h in range(Hq):
        sc = (q[:, h] @ K[h // G].t()) / math.sqrt(D)
        sc.masked_fill_(hidden, -math.inf)
        lse[h] = torch.logsumexp(sc, -1) / math.log(2.0)
        out[:, h] = torch.softmax(sc, -1) @ V[h // G]
    return out, lse


def _mlp64(x, ly):
    return x + _swiglu64(_rms64(x, ly["n2"]) @ _w64(ly["gu"]).t()) @ _w64(ly["down"]).t()


def _qkv64(x, ly, Hq, Hkv, D, cos, sin):
    y = _rms64(x, ly["n1"]) @ _w64(ly["qkv"]).t()
    if ly.get("bqkv") is not None:
        y = y + ly["bqkv"].double()
    y = y.view(x.shape[0], Hq + 2 * Hkv, D)
    return _rope64(y[:, :Hq], cos, sin), _rope64(y[:, Hq:Hq + Hkv], cos, sin), y[:, Hq + Hkv:]


def exact(case, seed):
    s = _inputs(case, seed)
    c, k = case, case["kind"]
    if k == "gemv":
        x = s["x"].double()
        y = (x if s["nw"] is None else _rms64(x, s["nw"])) @ _w64(s["w"]).t()
        return _swiglu64(y) if c["epi"] == 2 else y
    if k == "moe":
        return _moe64(c, s)
    H, Hq, Hkv, D, I, _ = MODELS[c["model"]]
    if k == "flash":
        n = c["p0"] + c["rows"]
        o, lse = _attend64(s["q"].double().view(-1, Hq, D), s["kc"][:, :n].double(), s["vc"][:, :n].double(), c["p0"])
        return o.reshape(c["rows"], Hq * D), lse
    if k == "engine":
        return _engine64(c, s)
    x = s["table"].double()[s["tok"].long()]
    if k == "decode_mlp":
        for ly in s["layers"]:
            x = _mlp64(x, ly)
        return x
    if k == "prefill_mlp":
        ly = s["layers"][0]
        x = _mlp64(x, ly)
        return [x, _rms64(x, ly["n1"])]
    cs = s["cs"].double()
    if k == "prefill_attn":
        ly, T, p0 = s["layers"][0], c["rows"], c["p0"]
        cos, sin = cs[p0:p0 + T, :, 0], cs[p0:p0 + T, :, 1]
        q, kk, v = _qkv64(x, ly, Hq, Hkv, D, cos, sin)
        K, V = ly["kc"].double(), ly["vc"].double()
        K[0, :, p0:p0 + T], V[0, :, p0:p0 + T] = kk.transpose(0, 1), v.transpose(0, 1)
        o, _ = _attend64(q, K[0, :, :p0 + T], V[0, :, :p0 + T], p0)
        x = x + o.reshape(T, Hq * D) @ _w64(ly["o"]).t()
        return [x, _rms64(x, ly["n2"]), K, V]
    pos = s["pos"].long()
    cos, sin = cs[pos, :, 0], cs[pos, :, 1]
    caches = []
    for ly in s["layers"]:
        q, kk, v = _qkv64(x, ly, Hq, Hkv, D, cos, sin)
        K, V = ly["kc"].double(), ly["vc"].double()
        att = torch.empty_like(q)
        for b, p in enumerate(s["pos_list"]):
            K[b, :, p], V[b, :, p] = kk[b], v[b]
            att[b] = _attend64(q[b:b + 1], K[b, :, :p + 1], V[b, :, :p + 1], p)[0][0]
        x = x + att.reshape(-1, Hq * D) @ _w64(ly["o"]).t()
        caches += [K, V]
    if k == "decode_attn":
        return [x] + caches
    ly = s["layers"][0]
    x = _mlp64(x, ly)
    return [x, _rms64(x, ly["n1"])] + caches


def _moe64(c, s):
    xn, x = s["xn"].double(), s["x0"].double()[s["tok"].long()]
    # the router's logits are fp16 by definition (ties go to the lower expert)
    logits = (xn @ s["wr"].double().t()).half().double()
    best, idx = torch.sort(logits, dim=1, descending=True, stable=True)
    best, idx = best[:, :c["top_k"]], idx[:, :c["top_k"]].contiguous()
    w = torch.softmax(best, 1)
    y = torch.zeros_like(x)
    for e in range(c["experts"]):
        rows, slot = (idx == e).nonzero(as_tuple=True)
        if rows.numel():
            h = _swiglu64(xn[rows] @ s["wgu"][e].double().t()) @ s["wdown"][e].double().t()
            y.index_add_(0, rows, h * w[rows, slot][:, None])
    return [x + 0.22 * y, idx.int(), w]


def _engine64(c, s):
    H, Hq, Hkv, D, I, _ = MODELS[c["model"]]
    seqs = [p + [t] for p, t in zip(s["prompts"], s["next"])]
    prompt_logits, step_logits = None, []
    inv = torch.from_numpy(s["inv_freq"]).double().cuda()
    for i, seq in enumerate(seqs):
        ang = torch.arange(len(seq), device="cuda").double()[:, None] * inv[None, :]
        x = s["embed"].double()[torch.tensor(seq, device="cuda")]
        for ly in s["layers"]:
            q, kk, v = _qkv64(x, ly, Hq, Hkv, D, ang.cos(), ang.sin())
            o, _ = _attend64(q, kk.transpose(0, 1).contiguous(), v.transpose(0, 1).contiguous(), 0)
            x = x + o.reshape(len(seq), Hq * D) @ _w64(ly["o"]).t()
            x = _mlp64(x, ly)
        logits = _rms64(x, s["nf"]) @ _w64(s["lm"]).t()
        if i == 0:
            prompt_logits = logits[:-1]
        step_logits.append(logits[-1])
    return [prompt_logits, torch.stack(step_logits)]
