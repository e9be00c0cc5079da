"""The work a user of these decode kernels has them do, as cases that can be timed and compared.

A case is a dict of plain values. ``prepare`` makes what a user's program holds before the call (quantized weights, a
model with its captured decode step, a paged cache, buffers), ``run`` makes one pass through the public entry points
(``runtime.ext`` ops, ``runtime.model.Model``), ``exact`` gives the same outputs from plain torch in 64 bits.

Ranges (``draw`` covers them, ``listed`` has representatives):
  gemv               one W4A16 GEMV: the projections and INT4 heads of Llama shapes; N 256-32768, K 1024-16384, G 64/128
  attention          decode attention of one token over a paged cache: contexts 64-32768, head dim 64/128, 1-8 query
                     heads per kv head, pages of 16 and 32 tokens
  step               one decode step of a whole model through its captured graph: contexts 16-8192
  gemm               one prompt projection: 2-2048 tokens, with and without the SwiGLU epilogue
  attention_prefill  causal attention of a prompt: 16-4096 tokens, at the start of a sequence or behind a cached prefix
  prefill            a whole prompt through a model: 8-1024 tokens
  quantize           the INT4 producer of a model build: round-to-nearest and range-clipped, G 32-256
"""
import json
import math
import os
import sys

import torch

# the package folder's name is not an identifier: its modules are imported from inside it
_PKG = os.path.join(os.getcwd(), "llm-decode-kernels_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from runtime import ext  # noqa: E402
from runtime.model import DecodeConfig, Model, default_gemv_config  # noqa: E402
from runtime.quant import quantize_pack  # noqa: E402
from runtime.synth import LlamaShape, SyntheticLlama  # noqa: E402

DEV = "cuda"
EPS = 1e-5
# hidden, heads, kv heads, intermediate, vocabulary, RoPE base of the two model shapes
SHAPES = {"tinyllama": (2048, 32, 4, 5632, 32000, 10000.0), "llama3_8b": (4096, 32, 8, 14336, 128256, 500000.0)}


def listed():
    return [
        # the smallest call: one attention output projection of TinyLlama, through the op module
        {"name": "gemv_2048x2048", "kind": "gemv", "N": 2048, "K": 2048, "G": 128},
        # the down projection of Llama-3-8B, the widest reduction of its decode step
        {"name": "gemv_4096x14336", "kind": "gemv", "N": 4096, "K": 14336, "G": 128},
        # the headline workload: one token of TinyLlama at context 512, all layers, fp16 head
        {"name": "step_tinyllama_512", "kind": "step", "shape": "tinyllama", "layers": 22, "vocab": 32000, "head": "fp16",
         "G": 128, "ctx": 512},
        # one token of the Llama-3-8B shape at context 4096 (four of its layers, INT4 head)
        {"name": "step_llama3_8b_4096", "kind": "step", "shape": "llama3_8b", "layers": 4, "vocab": 128256, "head": "int4",
         "G": 128, "ctx": 4096},
        # decode attention far into a long conversation, Llama-3-8B heads
        {"name": "attention_16384", "kind": "attention", "n_kv": 8, "hpg": 4, "D": 128, "page": 16, "ctx": 16384},
        # a short prompt (a chat turn): the gate|up projection of 16 tokens
        {"name": "gemm_gate_up_16", "kind": "gemm", "M": 16, "N": 28672, "K": 4096, "G": 128, "epilogue": 1},
        # an ordinary prompt: the same projection of 512 tokens
        {"name": "gemm_gate_up_512", "kind": "gemm", "M": 512, "N": 28672, "K": 4096, "G": 128, "epilogue": 1},
        # a long prompt: the down projection of 2048 tokens
        {"name": "gemm_down_2048", "kind": "gemm", "M": 2048, "N": 4096, "K": 14336, "G": 128, "epilogue": 0},
        # causal attention of an ordinary TinyLlama prompt
        {"name": "attention_prefill_512", "kind": "attention_prefill", "n_kv": 4, "hpg": 8, "D": 64, "page": 16,
         "M": 512, "start": 0},
        # causal attention of a long Llama-3-8B prompt (a document)
        {"name": "attention_prefill_4096", "kind": "attention_prefill", "n_kv": 8, "hpg": 4, "D": 128, "page": 16,
         "M": 4096, "start": 0},
        # time to first token: a TinyLlama prompt of a length that fits no tile
        {"name": "prefill_tinyllama_333", "kind": "prefill", "shape": "tinyllama", "layers": 22, "vocab": 32000,
         "head": "fp16", "G": 128, "M": 333},
        # building a model: quantizing one Llama-3-8B down projection
        {"name": "quantize_4096x14336", "kind": "quantize", "N": 4096, "K": 14336, "G": 128, "clip": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "attention", "step", "gemm", "gemm", "attention_prefill", "attention_prefill", "prefill",
                       "quantize"])
    G = rng.choice([64, 128, 128])
    if kind == "gemv":
        K = 128 * _log_int(rng, 8, 128)
        return {"kind": kind, "N": min(_log_int(rng, 256, 32768), 100_000_000 // K), "K": K, "G": G}
    if kind == "attention":
        return {"kind": kind, "n_kv": rng.choice([2, 4, 8]), "hpg": rng.choice([1, 2, 4, 8]), "D": rng.choice([64, 128]),
                "page": rng.choice([16, 16, 32]), "ctx": _log_int(rng, 64, 32768)}
    if kind == "step":
        return {"kind": kind, "shape": rng.choice(sorted(SHAPES)), "layers": rng.choice([1, 2, 3]), "vocab": 32000,
                "head": rng.choice(["fp16", "int4"]), "G": G, "ctx": _log_int(rng, 16, 8192)}
    if kind == "gemm":
        N, K = rng.choice([(2560, 2048), (2048, 2048), (11264, 2048), (2048, 5632), (6144, 4096), (4096, 4096),
                           (28672, 4096), (4096, 14336), (2 * rng.randint(500, 6000), 128 * rng.randint(8, 64))])
        epilogue = int(N in (11264, 28672) or (N % 4 == 0 and rng.random() < 0.2))
        return {"kind": kind, "M": min(_log_int(rng, 2, 2048), 110_000_000_000 // (N * K)), "N": N, "K": K, "G": G,
                "epilogue": epilogue}
    if kind == "attention_prefill":
        return {"kind": kind, "n_kv": rng.choice([2, 4, 8]), "hpg": rng.choice([1, 2, 4, 8]), "D": rng.choice([64, 128]),
                "page": rng.choice([16, 16, 32]), "M": _log_int(rng, 16, 2048), "start": rng.choice([0, 0, rng.randint(1, 4096)])}
    if kind == "prefill":
        return {"kind": kind, "shape": rng.choice(sorted(SHAPES)), "layers": rng.choice([1, 2, 3]), "vocab": 32000,
                "head": rng.choice(["fp16", "int4"]), "G": G, "M": _log_int(rng, 8, 1024)}
    return {"kind": kind, "N": _log_int(rng, 256, 16384), "K": 256 * rng.randint(4, 56), "G": rng.choice([32, 64, 128, 256]),
            "clip": rng.choice([False, True])}


# ------------------------------------------------------------------------------------------------ inputs and passes
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *size, std=1.0):
    return (torch.randn(*size, generator=g, device=DEV) * std).half()


def _config_json(name):
    with open(os.path.join(_PKG, "configs", name)) as f:
        return json.load(f)


def _gemv_config(N, K, G):
    """The tuned entry of a shape, else the default rule (what a program that calls the op by hand takes)."""
    e = _config_json("autotune.json").get("best", {}).get(f"{N}x{K}_G{G}")
    return default_gemv_config(N, K) if e is None else tuple(e) if len(e) == 4 else (2, *e)


def _part_size(D, ctx):
    """Tokens per split by the attention policy table: the entry of the largest context that is not over this one."""
    pol = _config_json("attn_policy.json")
    ents = [e for e in pol.get(f"policy_d{D}", pol["policy"]) if e["max_ctx"] < (1 << 30)]
    below = [e for e in ents if e["max_ctx"] <= ctx]
    return (below[-1] if below else ents[0])["part_size"]


def _paged_cache(g, ctx, n_kv, page, D):
    pages = -(-ctx // page) + 1
    kc, vc = _randn(g, pages, n_kv, page, D), _randn(g, pages, n_kv, page, D)
    return kc, vc, torch.randperm(pages, generator=g, device=DEV).int()


def _model(case, seed, max_ctx):
    H, n_q, n_kv, inter, _, theta = SHAPES[case["shape"]]
    shape = LlamaShape(H, case["layers"], n_q, n_kv, inter, case["vocab"], EPS, theta)
    return Model(SyntheticLlama(shape, seed=seed, device=DEV, norm_std=0.1), shape,
                 DecodeConfig(lm_head=case["head"], group=case["G"], max_ctx=max_ctx, seed=seed))


def prepare(case, seed):
    kind, g = case["kind"], _gen(seed)
    s = {"case": case, "ops": ext.load()}
    if kind in ("gemv", "gemm"):
        N, K, G = case["N"], case["K"], case["G"]
        s["packed"], s["sz"] = quantize_pack(_randn(g, N, K, std=0.02), G)
        if kind == "gemv":
            s.update(x=_randn(g, K), y=torch.empty(N, dtype=torch.half, device=DEV), config=_gemv_config(N, K, G))
        else:
            M, epi = case["M"], case["epilogue"]
            s.update(x=_randn(g, M, K), y=torch.empty(M, N // (1 + epi), dtype=torch.half, device=DEV))
            need = s["ops"].gemm_workspace_bytes(M, N, K, G, epi)
            s["workspace"] = torch.empty(need, dtype=torch.uint8, device=DEV) if need else None
    elif kind == "attention":
        n_kv, D, ctx = case["n_kv"], case["D"], case["ctx"]
        n_q = n_kv * case["hpg"]
        s["kc"], s["vc"], s["bt"] = _paged_cache(g, ctx, n_kv, case["page"], D)
        s["q"], s["out"] = _randn(g, n_q, D), torch.empty(n_q, D, dtype=torch.half, device=DEV)
        s["pos"] = torch.tensor([ctx - 1], dtype=torch.int32, device=DEV)
        s["part"] = _part_size(D, ctx)
        S = -(-ctx // s["part"])
        s["parts"] = tuple(torch.empty(*z, device=DEV) for z in ((n_q, S, D), (n_q, S), (n_q, S)))
    elif kind == "attention_prefill":
        n_kv, D, M, start = case["n_kv"], case["D"], case["M"], case["start"]
        n_q = n_kv * case["hpg"]
        s["kc"], s["vc"], s["bt"] = _paged_cache(g, start + M, n_kv, case["page"], D)
        s["qkv"] = _randn(g, M, (n_q + 2 * n_kv) * D)
        s["out"] = torch.empty(M, n_q * D, dtype=torch.half, device=DEV)
        s["pos"] = torch.tensor([start], dtype=torch.int32, device=DEV)
    elif kind == "step":
        ctx = case["ctx"]
        m = s["model"] = _model(case, seed, ctx + 64)
        m.prepare(ctx + 64)
        m.kv.normal_(generator=g)
        s["token"] = torch.randint(0, m.V, (1,), generator=g, device=DEV)
    elif kind == "prefill":
        s["model"] = _model(case, seed, case["M"] + 64)
        s["tokens"] = torch.randint(0, case["vocab"], (case["M"],), generator=torch.Generator().manual_seed(seed)).tolist()
    else:
        N, K, G = case["N"], case["K"], case["G"]
        s.update(w=_randn(g, N, K, std=0.02), packed=torch.empty(N, K // 8, dtype=torch.int32, device=DEV),
                 sz=torch.empty(N, K // G, 2, dtype=torch.half, device=DEV))
    return s


def run(s):
    case, ops = s["case"], s["ops"]
    kind = case["kind"]
    if kind == "gemv":
        ops.gemv_w4a16(*s["config"], s["packed"], s["sz"], s["x"], s["y"], case["G"])
        return s["y"]
    if kind == "gemm":
        ops.gemm_w4a16(s["packed"], s["sz"], s["x"], s["y"], case["G"], case["epilogue"], s["workspace"])
        return s["y"]
    if kind == "attention":
        ops.paged_attention(s["q"], s["kc"], s["vc"], s["bt"], s["pos"], s["part"], *s["parts"], s["out"], 3)
        return s["out"]
    if kind == "attention_prefill":
        ops.attention_prefill(s["qkv"], s["pos"], s["bt"], s["kc"], s["vc"], s["kc"].size(1) * case["hpg"],
                              s["kc"].size(1), case["start"] + case["M"], s["out"])
        return s["out"]
    if kind == "quantize":
        ops.quantize_w4(s["w"], s["packed"], s["sz"], case["G"], case["clip"])
        return {"packed": s["packed"], "sz": s["sz"]}
    m = s["model"]
    if kind == "step":  # the next token of a sequence that stands at `ctx`
        m.reset(case["ctx"])
        m.tok.copy_(s["token"])
        m.run_step()
    else:
        m.reset(0)
        m.prefill(s["tokens"])
    return {"logits": m.logits, "kv": m.kv}


# ------------------------------------------------------------------------------------------------ what a pass needs
def _gemv_bytes(N, K, G):
    return N * K // 2 + 4 * N * (K // G)


def work(case):
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        M, N, K = case.get("M", 1), case["N"], case["K"]
        out = N // (1 + case.get("epilogue", 0))
        return {"bytes": _gemv_bytes(N, K, case["G"]) + 2 * M * (K + out), "flops": 2 * M * N * K}
    if kind == "quantize":
        N, K, G = case["N"], case["K"], case["G"]
        return {"bytes": 2 * N * K + _gemv_bytes(N, K, G), "flops": 0}
    if kind in ("attention", "attention_prefill"):
        n_kv, D = case["n_kv"], case["D"]
        n_q = n_kv * case["hpg"]
        if kind == "attention":
            M, ctx, pairs = 1, case["ctx"], case["ctx"]
        else:
            M, ctx = case["M"], case["start"] + case["M"]
            pairs = M * case["start"] + M * (M + 1) // 2
        return {"bytes": 4 * ctx * n_kv * D + 4 * M * n_q * D + 4 * -(-ctx // case["page"]), "flops": 4 * n_q * D * pairs}
    H, n_q, n_kv, inter, _, _ = SHAPES[case["shape"]]
    L, V, G, D = case["layers"], case["vocab"], case["G"], H // n_q
    proj = (((n_q + 2 * n_kv) * D, H), (H, n_q * D), (2 * inter, H), (H, inter))
    M, start = (1, case["ctx"]) if kind == "step" else (case["M"], 0)
    pairs = M * start + M * (M + 1) // 2
    size = L * sum(_gemv_bytes(N, K, G) for N, K in proj) + (2 * V * H if case["head"] == "fp16" else _gemv_bytes(V, H, G))
    size += L * (4 * (start + M) * n_kv * D + 4 * H) + 2 * M * H + 2 * V
    return {"bytes": size, "flops": L * (2 * M * sum(N * K for N, K in proj) + 4 * n_q * D * pairs) + 2 * V * H}


def tolerance(case):
    """About four times the relative error that each path shows against 64 bits: 2e-4 for an fp16 output of fp32 sums,
    4.3e-4 where the SwiGLU epilogue rounds gate, silu and product, 5e-3 after the 22 layers of a whole model."""
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    if kind in ("step", "prefill"):
        return {"rel": 0.02, "max": 0.3}
    if case.get("epilogue", 0):
        return {"rel": 1.7e-3, "max": 0.03}
    return {"rel": 8e-4, "max": 0.01}


# ------------------------------------------------------------------------------------------------ 64-bit references
def _dequant(packed, sz, rounded):
    """[N, K] float64 of (q - zero) * scale; `rounded`: as the fp16 value that the prompt path defines."""
    N, K = packed.size(0), packed.size(1) * 8
    shift = torch.tensor([4 * (e >> 1) + 16 * (e & 1) for e in range(8)], dtype=torch.int32, device=packed.device)
    q = (packed.unsqueeze(-1) >> shift) & 15
    s, z = sz[..., :1].double(), sz[..., 1:].double()
    w = ((q.view(N, sz.size(1), -1) - z) * s).view(N, K)
    return w.half().double() if rounded else w


def _silu(x):
    return x / (1 + torch.exp(-x))


def _gather(cache, bt, ctx):
    """Tokens [0, ctx) of a paged cache [pages, n_kv, P, D] as float64 [n_kv, ctx, D]."""
    page = cache.size(2)
    t = torch.arange(ctx, device=cache.device)
    return cache[bt.long()[t // page], :, t % page].double().transpose(0, 1).contiguous()


def _attend(q, k, v, start):
    """q [M, n_q, D] (row m at position start + m), k and v [n_kv, ctx, D], all float64: causal attention [M, n_q, D]."""
    M, n_q, D = q.shape
    hpg, ctx = n_q // k.size(0), k.size(1)
    out = torch.empty_like(q)
    for m0 in range(0, M, 1024):
        qm = q[m0:m0 + 1024]
        hidden = torch.arange(ctx, device=q.device) > start + m0 + torch.arange(qm.size(0), device=q.device)[:, None]
        for h in range(n_q):
            sc = torch.mm(qm[:, h].contiguous(), k[h // hpg].t().contiguous()) / math.sqrt(D)
            out[m0:m0 + 1024, h] = torch.mm(torch.softmax(sc.masked_fill(hidden, -math.inf), -1), v[h // hpg])
    return out


def _exact_model(case, seed):
    s = prepare(case, seed)
    m, step = s["model"], case["kind"] == "step"
    H, n_q, n_kv, inter, _, theta = SHAPES[case["shape"]]
    D = H // n_q
    start = case["ctx"] if step else 0
    toks = s["token"] if step else torch.tensor(s["tokens"], device=DEV)
    M = toks.numel()
    kv = m.kv.double()
    t = start + torch.arange(M, device=DEV)
    ang = t.double()[:, None] / theta ** (torch.arange(0, D, 2, dtype=torch.float64, device=DEV) / D)
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def norm(x, w):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w.double()

    def rope(x):
        a, b = x[..., : D // 2], x[..., D // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    def proj(x, lin, rounded=not step):
        w = _dequant(lin.packed, lin.sz, rounded) if lin.quant else lin.w.double()
        return torch.mm(x, w.t())

    x = m.emb[toks].double()
    for i, lw in enumerate(m.layers):
        qkv = proj(norm(x, lw["ln1"]), lw["qkv"]).view(M, n_q + 2 * n_kv, D)
        kv[i, 0, m.bt.long()[t // m.cfg.page], :, t % m.cfg.page] = rope(qkv[:, n_q:n_q + n_kv])
        kv[i, 1, m.bt.long()[t // m.cfg.page], :, t % m.cfg.page] = qkv[:, n_q + n_kv:]
        k, v = (_gather(kv[i, j], m.bt, start + M) for j in range(2))
        x = x + proj(_attend(rope(qkv[:, :n_q]).contiguous(), k, v, start).view(M, -1), lw["o"])
        gu = proj(norm(x, lw["ln2"]), lw["gu"])
        gate, up = (gu[:, 0::2], gu[:, 1::2]) if lw["gu"].pairs_interleaved else (gu[:, :inter], gu[:, inter:])
        x = x + proj(_silu(gate) * up, lw["down"])
    return {"logits": proj(norm(x[-1:], m.norm_f), m.lm_head, False)[0], "kv": kv}


def exact(case, seed):
    kind = case["kind"]
    if kind == "quantize":
        return None  # codes and their fp16 parameters are compared bit by bit
    if kind in ("step", "prefill"):
        return _exact_model(case, seed)
    s = prepare(case, seed)
    if kind == "gemv":
        return torch.mv(_dequant(s["packed"], s["sz"], False), s["x"].double())
    if kind == "gemm":
        y = torch.mm(s["x"].double(), _dequant(s["packed"], s["sz"], True).t())
        return _silu(y[:, 0::2]) * y[:, 1::2] if case["epilogue"] else y
    n_kv, D = case["n_kv"], case["D"]
    n_q = n_kv * case["hpg"]
    if kind == "attention":
        k, v = (_gather(s[c], s["bt"], case["ctx"]) for c in ("kc", "vc"))
        return _attend(s["q"].double().unsqueeze(0), k, v, case["ctx"] - 1)[0]
    ctx = case["start"] + case["M"]
    k, v = (_gather(s[c], s["bt"], ctx) for c in ("kc", "vc"))
    q = s["qkv"][:, : n_q * D].double().view(-1, n_q, D)
    return _attend(q.contiguous(), k, v, case["start"]).view(case["M"], -1)
