"""Per-shape W4A16 GEMV tuner for MI355X (the role of the reference's scripts/autotune.py:27-54).

For every (N, K, group) shape, sweeps the kernel family of libdk_amd (stage 2: whole-row waves, R rows per wave x
waves per workgroup x 2^pf steps in flight; stage 3: split-K, R rows per workgroup x waves x one-step prefetch;
stage 4: 2^pf row tiles of R rows over a workgroup that covers K once) with
cold weights (runtime.timing), and writes

    configs/autotune.json   {"device": ..., "best": {"NxK_G": [stage, R, warps, pf]}, "best_tile": {the best stage-4
                             entry}, "us": {"NxK_G": us}, "best_norm": {the fused residual + RMSNorm GEMV},
                             "best_gate_up": {the gate|up GEMV with the SwiGLU epilogue}, "best_f16" /
                             "best_f16_norm": {"NxK": [R, waves, pf]} of the fp16 GEMV, "us_*": times,
                             "grid": [every measurement]}

The runtime (runtime.model.Model.gemv_cfg) reads "best" ("best_tile" is informational: the fastest stage-4
configuration of a shape whose overall best is another stage); 3-element entries [R, warps, pf] of the reference's schema
are read as stage 2. Run:  python -m runtime.autotune [--shapes tinyllama,llama3_8b,baseline] [--groups 128]
With --attention it tunes the decode attention instead (kernel and split size per head dim and context) and writes
configs/attn_policy.json; with --step it chooses the decode step's GEMV configurations by the step time ("best_step").
"""
import argparse
import json
import pathlib
import sys

import torch

from . import ext
from .quant import quantize_pack
from .timing import ColdCopies, graph_time, n_copies

PKG = pathlib.Path(__file__).resolve().parents[1]
CONFIG = PKG / "configs" / "autotune.json"

SHAPE_SETS = {
    # TinyLlama-1.1B decode: qkv, o, gate|up, down, INT4 LM head
    "tinyllama": {"qkv": (2560, 2048), "o": (2048, 2048), "gate_up": (11264, 2048), "down": (2048, 5632),
                  "lm_head": (32000, 2048)},
    # Llama-3-8B decode
    "llama3_8b": {"qkv8b": (6144, 4096), "o8b": (4096, 4096), "gate_up8b": (28672, 4096), "down8b": (4096, 14336),
                  "lm_head8b": (128256, 4096)},
    # BASELINE config 1 and the standalone target shapes
    "baseline": {"cfg1": (5632, 2048), "w4096x14336": (4096, 14336), "w14336x4096": (14336, 4096)},
    # one GPU's share under tensor parallelism (qkv and gate|up split by rows, o and down by columns): Llama-3-8B over
    # 8 GPUs (one kv head each) and TinyLlama over 4 (its kv head count)
    "llama3_8b_tp8": {"qkv8b_tp8": (768, 4096), "o8b_tp8": (4096, 512), "gate_up8b_tp8": (3584, 4096),
                      "down8b_tp8": (4096, 1792)},
    "tinyllama_tp4": {"qkv_tp4": (640, 2048), "o_tp4": (2048, 512), "gate_up_tp4": (2816, 2048),
                      "down_tp4": (2048, 1408)},
}


def candidates(N, K):
    out = []
    for R in (1, 2, 4, 8):
        for w in (1, 2, 4, 8):
            for pf in range(4):
                if (1 << pf) > 16 // R or (1 << pf) > max(1, -(-K // 2048)):
                    continue
                out.append((2, R, w, pf))
    U = K // 32
    full = min(16, -(-U // 64))
    for R in (1, 2, 4, 8):
        for w in sorted({1, 2, 4, 8, full}):
            for pf in (0, 1):
                if pf and U <= 64 * w:
                    continue
                out.append((3, R, w, pf))
    if K <= 32768:
        out += tile_candidates(K)
    return [c for c in out if not (c[0] == 2 and K > 32768)]


def tile_candidates(K):
    """stage-4 configurations: one row group per workgroup over R x 2^pf, and 2 or 4 row groups of ceil(K / 2048)
    waves each (warps = groups x ceil(K / 2048) <= 16) over the smaller tiles."""
    tw = -(-K // 2048)
    out = [(4, R, 0, pf) for R in (1, 2, 4, 8) for pf in range(4)]
    out += [(4, R, g * tw, pf) for g in (2, 4) if g * tw <= 16 for R in (1, 2, 4) for pf in range(3)]
    return out


def attn_candidates(K):
    """stage-4 configurations of the o projection with the attention combine in its prologue: one thread per 8
    values of x, so at least ceil(K / 512) waves (a multiple of ceil(K / 2048)) and at most 8."""
    tw = -(-K // 2048)
    need = -(-max(-(-K // 512), tw) // tw) * tw
    return [(4, R, w, pf) for w in sorted({need, 2 * need}) if w <= 8 for R in (1, 2, 4) for pf in range(3)]


def fused_candidates(kind, K):
    """stage-4 configurations of the fused INT4 GEMVs (the gate|up SwiGLU epilogue needs an even row tile; so does
    the qkv RoPE epilogue, which takes the same candidates)."""
    return [c for c in tile_candidates(K) if kind != "gate_up" or (c[1] << c[3]) >= 2]


def f16_candidates(K):
    """(R, waves, pf) of the fp16 GEMV: R * 2^ceil(log2(ceil(K / 512))) <= 16 loads per lane per tile."""
    c = 1 << max(0, (-(-K // 512) - 1).bit_length())
    return [(R, w, pf) for R in (1, 2, 4) if R * c <= 16 for w in (1, 2, 4, 8) for pf in range(4)]


def tune_fused_shape(Kx, kind, N, K, G, reps=5, log=print):
    """Best configuration of one fused variant for one shape, cold weights:
       rmsnorm   dk_gemv_w4a16_rmsnorm (qkv, gate|up, INT4 LM head behind a residual + RMSNorm)
       gate_up   dk_gemv_w4a16_gate_up with the RMSNorm input (the MLP's gate|up + SwiGLU; N = 2I rows)
       f16       dk_gemv_f16 (fp16 LM head, G unused)
       f16_norm  dk_gemv_f16_rmsnorm (the fp16 LM head behind the final residual + RMSNorm)"""
    g = torch.Generator(device="cuda").manual_seed(N * 17 + K)
    w = (torch.randn(N, K, generator=g, device="cuda") * 0.02).half()
    x = torch.randn(K, generator=g, device="cuda").half()
    d = torch.randn(K, generator=g, device="cuda").half()
    nw = torch.ones(K, dtype=torch.half, device="cuda")
    xo = torch.empty_like(x)
    y = torch.empty(N, dtype=torch.half, device="cuda")
    act = torch.empty(N // 2, dtype=torch.half, device="cuda")
    if kind in ("f16", "f16_norm"):
        ops, nb, cands = [w], N * K * 2, f16_candidates(K)
    else:
        ops, nb, cands = list(quantize_pack(w, G)), gemv_bytes(N, K, G), fused_candidates(kind, K)
    del w
    cold = ColdCopies(ops, n_copies(nb))
    call = {
        "rmsnorm": lambda c, i: Kx.gemv_w4a16_rmsnorm(*c, *cold[i], x, None, d, nw, 1e-5, xo, y, G),
        "gate_up": lambda c, i: Kx.gemv_w4a16_gate_up(*c, *cold[i], x, None, d, nw, 1e-5, xo, act, G),
        "f16": lambda c, i: Kx.gemv_f16(*c, cold[i][0], x, y),
        "f16_norm": lambda c, i: Kx.gemv_f16_rmsnorm(*c, cold[i][0], x, d, nw, 1e-5, None, y),
    }[kind]
    recs = []
    for cfg in cands:
        _, med = graph_time(lambda i: call(cfg, i), cold.copies, reps)
        recs.append({"N": N, "K": K, "G": G, "cfg": list(cfg), "median_us": med, "variant": kind})
    best = confirm(recs, lambda c: graph_time(lambda i: call(c, i), cold.copies, reps)[1])
    for r in recs:
        r["gbps"] = nb / r["median_us"] / 1e3
    log(f"  {kind} {N}x{K}: best {best['cfg']} {best['median_us']:.2f} us {best['gbps']:.0f} GB/s; "
        f"{len(recs)} configs")
    del cold
    return best, recs


def confirm(recs, measure, top=5, rounds=3):
    """Re-time the `top` fastest candidates in `rounds` interleaved passes and keep each one's best median: a single
    pass over tens of configurations picks an outlier now and then (a 1 us slip at a 14 us shape is within one pass's
    spread), and the runtime then pays for it in every layer of every token."""
    lead = sorted(recs, key=lambda r: r["median_us"])[:top]
    for _ in range(rounds):
        for r in lead:
            r["median_us"] = min(r["median_us"], measure(tuple(r["cfg"])))
    return min(recs, key=lambda r: r["median_us"])


def gemv_bytes(N, K, G):
    return N * K // 2 + N * (K // G) * 4 + 2 * K + 2 * N


def tune_shape(Kx, N, K, G, reps=5, log=print):
    g = torch.Generator(device="cuda").manual_seed(N * 131 + K)
    packed, sz = quantize_pack((torch.randn(N, K, generator=g, device="cuda") * 0.02).half(), G)
    x = torch.randn(K, generator=g, device="cuda").half()
    y = torch.empty(N, dtype=torch.half, device="cuda")
    nb = gemv_bytes(N, K, G)
    cold = ColdCopies([packed, sz], n_copies(nb))
    recs = []
    for cfg in candidates(N, K):
        mn, med = graph_time(lambda i: Kx.gemv_w4a16(*cfg, *cold[i], x, y, G), cold.copies, reps)
        recs.append({"N": N, "K": K, "G": G, "cfg": list(cfg), "min_us": mn, "median_us": med})
    best = confirm(recs, lambda c: graph_time(lambda i: Kx.gemv_w4a16(*c, *cold[i], x, y, G), cold.copies, reps)[1])
    tiles = sorted((r for r in recs if r["cfg"][0] == 4), key=lambda r: r["median_us"])
    if tiles and tiles[0] is not best:  # the best row-tile entry is a table of its own: confirm it the same way
        confirm(tiles, lambda c: graph_time(lambda i: Kx.gemv_w4a16(*c, *cold[i], x, y, G), cold.copies, reps)[1])
    for r in recs:
        r["gbps"] = nb / r["median_us"] / 1e3
    del cold
    log(f"  {N}x{K} G{G}: best {best['cfg']} {best['median_us']:.2f} us {best['gbps']:.0f} GB/s "
        f"({best['gbps'] / 80:.1f}% of 8 TB/s); {len(recs)} configs")
    return best, recs


# Shapes of the fused variants in the decode step: INT4 GEMVs behind a residual + RMSNorm (qkv, INT4 LM head), the
# gate|up GEMV with the SwiGLU epilogue, and the fp16 LM head (plain and behind the final norm)
FUSED_SHAPES = {
    "tinyllama": {"rmsnorm": ((2560, 2048), (11264, 2048), (32000, 2048)), "gate_up": ((11264, 2048),),
                  "f16": ((32000, 2048),), "f16_norm": ((32000, 2048),)},
    "llama3_8b": {"rmsnorm": ((6144, 4096), (28672, 4096), (128256, 4096)), "gate_up": ((28672, 4096),),
                  "f16": ((128256, 4096),), "f16_norm": ((128256, 4096),)},
    "baseline": {},
}
# table name in configs/autotune.json per variant, and whether its key carries the group size
TABLES = {"rmsnorm": ("best_norm", True), "gate_up": ("best_gate_up", True), "f16": ("best_f16", False),
          "f16_norm": ("best_f16_norm", False)}


def tune(shape_sets=("tinyllama", "llama3_8b", "baseline"), groups=(128,), reps=5, path=CONFIG, log=print):
    Kx = ext.load()
    old = json.load(open(path)) if pathlib.Path(path).exists() else {}
    best, us, grid = dict(old.get("best", {})), dict(old.get("us", {})), []
    best_tile = dict(old.get("best_tile", {}))
    tables = {t: dict(old.get(t, {})) for t, _ in TABLES.values()}
    times = {t: dict(old.get("us_" + t[5:], {})) for t, _ in TABLES.values()}
    for ss in shape_sets:
        for kind, shapes in FUSED_SHAPES.get(ss, {}).items():
            table, grouped = TABLES[kind]
            for (N, K) in shapes:
                for G in (groups if grouped else (128,)):
                    b, recs = tune_fused_shape(Kx, kind, N, K, G, reps, log)
                    key = f"{N}x{K}_G{G}" if grouped else f"{N}x{K}"
                    tables[table][key], times[table][key] = b["cfg"], round(b["median_us"], 3)
                    grid += recs
    for ss in shape_sets:
        for name, (N, K) in SHAPE_SETS[ss].items():
            for G in groups:
                b, recs = tune_shape(Kx, N, K, G, reps, log)
                key = f"{N}x{K}_G{G}"
                best[key], us[key] = b["cfg"], round(b["median_us"], 3)
                tiles = [r for r in recs if r["cfg"][0] == 4]
                if tiles:
                    best_tile[key] = min(tiles, key=lambda r: r["median_us"])["cfg"]
                grid += [dict(r, shape=name) for r in recs]
    out = {"device": torch.cuda.get_device_properties(0).name, "best": best, "best_tile": best_tile, "us": us}
    for t, _ in TABLES.values():
        out[t], out["us_" + t[5:]] = tables[t], times[t]
    out["grid"] = grid
    pathlib.Path(path).parent.mkdir(exist_ok=True)
    write_table(out, path)
    return out


def write_table(out, path):
    """One line per table entry and per grid record (times rounded to ns)."""
    def compact(v):
        if isinstance(v, float):
            return round(v, 3)
        if isinstance(v, dict):
            return {k: compact(x) for k, x in v.items()}
        return v

    parts = []
    for k, v in out.items():
        if isinstance(v, dict):
            body = ",\n".join(f"  {json.dumps(kk)}: {json.dumps(compact(vv))}" for kk, vv in v.items())
            parts.append(f" {json.dumps(k)}: {{\n{body}\n }}" if v else f" {json.dumps(k)}: {{}}")
        elif isinstance(v, list):
            body = ",\n".join("  " + json.dumps(compact(r), separators=(",", ":")) for r in v)
            parts.append(f" {json.dumps(k)}: [\n{body}\n ]" if v else f" {json.dumps(k)}: []")
        else:
            parts.append(f" {json.dumps(k)}: {json.dumps(v)}")
    txt = "{\n" + ",\n".join(parts) + "\n}\n"
    assert json.loads(txt).keys() == out.keys()
    pathlib.Path(path).write_text(txt)


# ------------------------------------------------------------------------------------------ attention policy
ATTN_MODELS = {64: "TINYLLAMA", 128: "LLAMA3_8B"}   # head_dim -> the model whose decode step the policy is tuned in
ATTN_CONTEXTS = (512, 1024, 2048, 4096, 8192, 16384)
ATTN_PATH = PKG / "configs" / "attn_policy.json"


def step_time_us(model, ctx, steps=24, warmup=8):
    """Mean graph-replayed decode step time starting at context ctx."""
    model.reset(ctx)
    for _ in range(warmup):
        model.run_step()
    torch.cuda.synchronize()
    model.reset(ctx)
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    a.record()
    for _ in range(steps):
        model.run_step()
    b.record()
    torch.cuda.synchronize()
    return a.elapsed_time(b) * 1e3 / steps


def merge_policy(entries, tuned):
    """Policy entries by context, those of `tuned` in the place of earlier ones, and after them an open-ended copy of the
    last (the reference's schema ends on one; the runtime's lookup takes the entries with a context of their own)."""
    by_ctx = {e["max_ctx"]: e for e in entries if e["max_ctx"] < 1 << 30}
    by_ctx.update({e["max_ctx"]: e for e in tuned})
    ents = [by_ctx[c] for c in sorted(by_ctx)]
    return ents + [dict(ents[-1], max_ctx=1 << 30)]


SAME_STEP = 1.005   # two passes of the tuner differ by 0.2 to 0.4%


def choose_split(times, smaller):
    """(impl, part_size) of the least step time; the choice of the largest context among the entries `smaller` where it
    is no slower than that within a pass's spread (a model prepared for a long context mostly runs at shorter ones)."""
    best = min(times, key=times.get)
    if smaller:
        e = max(smaller, key=lambda e: e["max_ctx"])
        kept = (e["impl"], e["part_size"])
        if times.get(kept, float("inf")) <= SAME_STEP * times[best]:
            return kept
    return best


def tune_attention(dims=(64, 128), contexts=ATTN_CONTEXTS, path=ATTN_PATH, log=print):
    """Writes configs/attn_policy.json: per head dim, entries {max_ctx, part_size, impl} (the reference's schema,
    runtime/model.py:160-178, plus the kernel choice), the last one open-ended; entries and grid records of contexts that
    are not tuned now stay. Every candidate (impl 1 block kernel,
    2 MFMA kernel or 3 lean MFMA kernel, split size) is timed inside the decode step of the model that has this head
    dim (graph replay at context ctx): an attention kernel costs more inside the step, interleaved with the GEMVs,
    than back to back, and by different amounts per kernel, so isolated launches would choose wrongly. The three
    fastest candidates of each context are timed twice more, interleaved, and keep their best time (choose_split)."""
    from . import synth
    from .model import DecodeConfig, Model
    old = json.load(open(path)) if pathlib.Path(path).exists() else {}
    out = {"version": old.get("version", 3),
           "note": "part_size (tokens per split) and impl (1 block kernel, 3 lean MFMA kernel) by the "
                   "largest tuned context "
                   "<= the prepared cap; chosen by the decode step time of the TinyLlama (head_dim 64) and Llama-3-8B "
                   "(head_dim 128) shapes on MI355X (runtime.autotune.tune_attention). 'policy' is head_dim 64, "
                   "'policy_d128' head_dim 128."}
    key = lambda D: "policy" if D == 64 else f"policy_d{D}"
    out.update({key(D): old[key(D)] for D in sorted(ATTN_MODELS) if key(D) in old})
    grid = [r for r in old.get("grid", []) if r["D"] not in dims or r["ctx"] not in contexts]
    for D in dims:
        shape = getattr(synth, ATTN_MODELS[D])
        cap_max = max(contexts) + 64
        model = Model(synth.SyntheticLlama(shape, seed=0), shape,
                      DecodeConfig(lm_head="int4" if D == 128 else "fp16", max_ctx=cap_max))
        ents = []
        lean_max = 256 if D == 128 else 512
        for ctx in contexts:
            cands = [(1, ps) for ps in (32, 64, 128)]  # the block kernel costs about 3 us per extra 64-token block
            # every multiple of 16 is a valid lean split: sizes between the powers of two set the workgroup count
            # against the 256 CUs (Llama-3-8B ctx 4096: part 160, 26 splits x 8 kv heads, 1302 us per step against
            # 1337 at part 256)
            cands += [(3, ps) for ps in (16, 32, 48, 64, 80, 96, 112, 128, 160, 192, 224, 256, 320, 384, 448, 512)
                      if ps <= lean_max]
            times = {}
            for impl, ps in cands:
                model.prepare(ctx + 48, part_size=ps, impl=impl)
                times[(impl, ps)] = step_time_us(model, ctx)
            for _ in range(2):  # confirm the leaders
                for impl, ps in sorted(times, key=times.get)[:3]:
                    model.prepare(ctx + 48, part_size=ps, impl=impl)
                    times[(impl, ps)] = min(times[(impl, ps)], step_time_us(model, ctx))
            for (impl, ps), us in times.items():
                grid.append({"D": D, "ctx": ctx, "impl": impl, "part_size": ps, "step_us": round(us, 2)})
            impl, ps = choose_split(times, [e for e in old.get(key(D), []) + ents if e["max_ctx"] < ctx])
            best = (times[(impl, ps)], impl, ps)
            log(f"  attention D{D} ctx {ctx}: best impl {best[1]} part_size {best[2]} ({best[0]:.1f} us per step)")
            ents.append({"max_ctx": ctx, "part_size": best[2], "impl": best[1]})
        out[key(D)] = merge_policy(old.get(key(D), []), ents)
        del model
        torch.cuda.empty_cache()
    out["grid"] = sorted(grid, key=lambda r: (r["D"], r["ctx"]))
    write_table(out, path)
    return out


# ------------------------------------------------------------------------------------------ GEMVs inside the step
STEP_MODELS = {"tinyllama": ("TINYLLAMA", "fp16", 512), "llama3_8b": ("LLAMA3_8B", "int4", 4096)}


def step_slots(model):
    """The GEMV launches of one decode step that the in-step tuner varies: (table kind, projection, candidates).
    Kinds: "norm" (qkv behind the fused residual + RMSNorm), "rope" (the same qkv launch with the RoPE + append
    epilogue, whose row tile must hold a rotation pair), "attn" (o with the attention combine in its prologue),
    "plain" (o, down; the INT4 head when the norm does not pay inside it), "gate_up" (gate|up with the SwiGLU
    epilogue), "f16_norm" (the fp16 head behind the final norm)."""
    lw = model.layers[0]
    K = lambda lin: lin.K
    qkv = (("rope", lw["qkv"], fused_candidates("gate_up", K(lw["qkv"]))) if model.rope_epilogue
           else ("norm", lw["qkv"], fused_candidates("rmsnorm", K(lw["qkv"]))))
    o = (("attn", lw["o"], attn_candidates(K(lw["o"]))) if model.attn_in_o
         else ("plain", lw["o"], fused_candidates("rmsnorm", K(lw["o"]))))
    slots = [qkv, o,
             ("gate_up", lw["gu"], fused_candidates("gate_up", K(lw["gu"]))),
             ("plain", lw["down"], fused_candidates("rmsnorm", K(lw["down"])))]
    head = model.lm_head
    if head.quant:
        kind = "norm" if model.norm_fusion_pays(head) else "plain"
        slots.append((kind, head, fused_candidates("rmsnorm", head.K)))
    elif model.use_f16_gemv(head):
        slots.append(("f16_norm", head, f16_candidates(head.K)))
    return slots


def tune_step(models=("tinyllama", "llama3_8b"), path=CONFIG, rounds=2, log=print):
    """Writes "best_step" into configs/autotune.json: {"kind:NxK_G": config} for the GEMVs of the decode step, each
    chosen by the graph-replayed step time of the model it belongs to (coordinate descent over the launches, `rounds`
    passes). At batch 1 these GEMVs are latency-bound inside the step, where a configuration that keeps every row of
    a workgroup in flight at once can win although it loses in isolated cold launches; the isolated tables stay the
    fallback for shapes the step tuner has not seen."""
    from . import synth
    from .model import DecodeConfig, Model
    old = json.load(open(path)) if pathlib.Path(path).exists() else {}
    table = dict(old.get("best_step", {}))
    for name in models:
        shape_name, head, ctx = STEP_MODELS[name]
        shape = getattr(synth, shape_name)
        model = Model(synth.SyntheticLlama(shape, seed=0), shape, DecodeConfig(lm_head=head, max_ctx=ctx + 64))
        model.prepare(ctx + 48)
        base = step_time_us(model, ctx)
        log(f"  {name}: step {base:.1f} us with the isolated tables")
        for _ in range(rounds):
            for kind, lin, cands in step_slots(model):
                key = model.step_key(kind, lin)
                cur = model.step_cfg_override.pop(key, None)
                isolated = {"plain": model.gemv_cfg, "norm": model.gemv_norm_cfg, "gate_up": model.gemv_gate_up_cfg,
                            "rope": model.qkv_rope_cfg, "attn": model.gemv_attn_cfg,
                            "f16_norm": lambda l: model.gemv_f16_cfg(l, norm=True)}[kind](lin)
                cands = list(dict.fromkeys([tuple(c) for c in cands] + [tuple(isolated)]))
                times = {}
                for c in cands:
                    model.step_cfg_override[key] = tuple(c)
                    model.capture()
                    times[tuple(c)] = step_time_us(model, ctx)
                for c in sorted(times, key=times.get)[:3]:  # confirm the leaders
                    model.step_cfg_override[key] = c
                    model.capture()
                    times[c] = min(times[c], step_time_us(model, ctx))
                best = min(times, key=times.get)
                model.step_cfg_override[key] = best
                log(f"  {name} {key}: {list(best)} {times[best]:.1f} us per step (was {list(cur) if cur else None})")
        model.capture()
        log(f"  {name}: step {step_time_us(model, ctx):.1f} us with the in-step choices (from {base:.1f})")
        # only this model's slots: its override map also holds the other models' entries read from the old table
        tuned = {model.step_key(kind, lin) for kind, lin, _ in step_slots(model)}
        table.update({k: list(v) for k, v in model.step_cfg_override.items() if k in tuned})
        del model
        torch.cuda.empty_cache()
    out = dict(old, best_step=table)
    write_table(out, path)
    return out


def main(argv=None):
    ap = argparse.ArgumentParser()
    ap.add_argument("--shapes", default="tinyllama,llama3_8b,baseline")
    ap.add_argument("--groups", default="128")
    ap.add_argument("--reps", type=int, default=5)
    ap.add_argument("--out", default=None)
    ap.add_argument("--attention", action="store_true", help="tune the attention policy instead of the GEMVs")
    ap.add_argument("--contexts", default=None, help="with --attention: the contexts to tune (default: all)")
    ap.add_argument("--step", action="store_true", help="tune the decode step's GEMV launches inside the step")
    a = ap.parse_args(argv)
    log = lambda *s: print(*s, flush=True)
    if a.attention:
        ctxs = tuple(int(c) for c in a.contexts.split(",")) if a.contexts else ATTN_CONTEXTS
        tune_attention(contexts=ctxs, path=a.out or ATTN_PATH, log=log)
        return
    if a.step:
        tune_step(path=a.out or CONFIG, log=log)
        return
    tune(a.shapes.split(","), tuple(int(g) for g in a.groups.split(",")), a.reps, a.out or CONFIG, log=log)


if __name__ == "__main__":
    sys.exit(main())
