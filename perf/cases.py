"""The work a serving program has this framework do, as cases that can be timed and compared.

Decode attention, varlen prefill attention, the fused norm / RoPE / cache-write kernels, the
decode step's MLP projections, a whole captured decode step and a whole mixed step, each
through the package's public entry points. ``listed()`` holds the named cases; ``draw(rng)``
gives more of the same ranges. The sequence lengths of a case follow from its own ``lens``
field (a seed), so that its work does not depend on the inputs' seed.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from tinyserve_amd import hip_attention, hip_fused, hip_prefill, hip_rows
from tinyserve_amd.decode_step import DecodeGraph, DecodeStep, KVPool, ModelShape
from tinyserve_amd.step_inputs import DecodeInputs, PagedTable, build_batch, fill_decode_inputs

DEVICE = "cuda"
DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"fp32": 4, "fp16": 2, "bf16": 2}
EPS = 1e-6
THETA = 1.0e6
HIDDEN, INTER, VOCAB = 1024, 3072, 151936
HQ, HKV, D = 16, 8, 128
QKV = (HQ + 2 * HKV) * D


def listed() -> list[dict]:
    return [
        # The smallest batch: four short sequences in fp32, two launches' latency.
        decode("decode_fp32_4_short", 4, 17, 200, dtype="fp32", lens=3),
        # A short-context decode batch, as an engine's step at 128 prompt + 128 new tokens.
        decode("decode_fp16_32x256", 32, 256, 256),
        # A ragged long-context batch in bf16 with four query heads per kv head.
        decode("decode_bf16_gqa4_48_ragged", 48, 100, 5000, dtype="bf16", hq=32, lens=1),
        # The largest: 64 sequences of 4096 tokens, bound by the cache's bytes.
        decode("decode_fp16_64x4096", 64, 4096, 4096),
        # One 2048-token prompt: the time to first token of a lone request.
        prefill("prefill_fp16_1x2048", 1, 2048, 2048),
        # A packed batch of 32 prompts of 16 to 2048 tokens.
        prefill("prefill_fp16_32_varlen", 32, 16, 2048, lens=0),
        # Eight prompts of odd lengths in bf16.
        prefill("prefill_bf16_8_mixed", 8, 200, 3000, dtype="bf16", lens=4),
        # Prefix-cache hits: long cached prefixes, short new chunks.
        prefill("prefill_fp16_16_prefix", 16, 20, 128, cached_lo=500, cached_hi=5000, lens=2),
        # The kernels around attention on a 4096-token prefill step: RoPE tables, RMSNorm,
        # q/k norm + RoPE + cache write.
        {"name": "norms_fp16_4096", "kind": "norms", "dtype": "fp16", "tokens": 4096},
        # The MLP half of eight decoder layers on 64 decode rows, captured as an engine does.
        {"name": "mlp_bf16_64x8", "kind": "mlp", "dtype": "bf16", "rows": 64, "layers": 8},
        # A whole 28-layer decode step in a captured graph, 32 sequences at short contexts.
        {"name": "step_fp16_32", "kind": "step", "dtype": "fp16", "rows": 32, "lo": 192, "hi": 320,
         "layers": 28, "lens": 7},
        # A whole mixed step: six prompts and 16 decoding sequences in one flat batch.
        {"name": "mixed_fp16_6p_16d", "kind": "mixed", "dtype": "fp16", "prompts": 6, "plo": 40, "phi": 600,
         "rows": 16, "lo": 100, "hi": 1000, "layers": 28, "lens": 5},
    ]  # fmt: skip


def decode(name: str | None, batch: int, lo: int, hi: int, dtype: str = "fp16", hq: int = HQ, hkv: int = HKV,
           d: int = D, bs: int = 16, splits: int = 0, lens: int = 0) -> dict:  # fmt: skip
    c = {"kind": "decode", "batch": batch, "lo": lo, "hi": hi, "dtype": dtype, "hq": hq, "hkv": hkv, "d": d,
         "bs": bs, "splits": splits, "lens": lens}  # fmt: skip
    return {"name": name, **c} if name else c


def prefill(name: str | None, seqs: int, lo: int, hi: int, dtype: str = "fp16", hq: int = HQ, hkv: int = HKV,
            d: int = D, bs: int = 16, cached_lo: int = 0, cached_hi: int = 0, lens: int = 0) -> dict:  # fmt: skip
    c = {"kind": "prefill", "seqs": seqs, "lo": lo, "hi": hi, "dtype": dtype, "hq": hq, "hkv": hkv, "d": d,
         "bs": bs, "cached_lo": cached_lo, "cached_hi": cached_hi, "lens": lens}  # fmt: skip
    return {"name": name, **c} if name else c


def draw(rng) -> dict:  # noqa: ANN001
    def log(lo: int, hi: int) -> int:
        return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))

    kind = rng.choice(["decode", "decode", "prefill", "prefill", "norms", "mlp", "step", "mixed"])
    half = rng.choice(["fp16", "bf16"])
    seed = rng.randrange(1 << 20)
    hq, hkv, d = rng.choice([(16, 8, 128), (16, 8, 128), (32, 8, 128), (8, 2, 64), (16, 8, 64)])
    bs = rng.choice([16, 16, 32])
    if kind == "decode":
        batch = log(1, 128)
        # At most the K/V bytes of the largest listed case: 64 sequences of 4096 tokens.
        most = min(32768, 64 * 4096 // batch)
        hi = log(16, most)
        lo = rng.choice([hi, max(1, hi // 4), 1])
        return decode(None, batch, lo, hi, rng.choice([half, half, half, "fp32"]) if hi <= 2048 else half, hq, hkv,
                      d, bs, rng.choice([0, 0, 0, 4, 16]), seed)  # fmt: skip
    if kind == "prefill":
        seqs = log(1, 64)
        if rng.random() < 0.3:
            hi = log(2, 256)
            ch = log(64, max(64, min(16384, 65536 // seqs)))
            return prefill(None, seqs, max(1, hi // 3), hi, half, hq, hkv, d, bs, max(1, ch // 4), ch, seed)
        hi = log(16, min(8192, int(math.sqrt(1.0e8 / seqs))))
        return prefill(None, seqs, rng.choice([hi, max(1, hi // 2), min(hi, 16)]), hi, half, hq, hkv, d, bs, 0, 0, seed)
    if kind == "norms":
        return {"kind": "norms", "dtype": half, "tokens": log(1, 16384)}
    if kind == "mlp":
        return {"kind": "mlp", "dtype": half, "rows": log(1, 256), "layers": 8}
    if kind == "step":
        rows = log(1, 128)
        hi = log(16, min(4096, 16384 // rows))
        return {"kind": "step", "dtype": half, "rows": rows, "lo": max(1, hi // 2), "hi": hi,
                "layers": rng.choice([8, 16, 28]), "lens": seed}  # fmt: skip
    prompts = rng.randint(1, 6)
    phi = log(32, min(2000, 3600 // prompts))  # about the listed step's tokens at most
    return {"kind": "mixed", "dtype": half, "prompts": prompts, "plo": max(2, phi // 8), "phi": phi,
            "rows": rng.choice([0, 1, 5, 24]), "lo": 16, "hi": log(32, 1500), "layers": rng.choice([4, 12, 28]),
            "lens": seed}  # fmt: skip


# ---- sizes -------------------------------------------------------------------------------
def _between(seed: int, n: int, lo: int, hi: int) -> list[int]:
    g = torch.Generator().manual_seed(seed)
    return torch.randint(lo, hi + 1, (n,), generator=g).tolist()


def _decode_lens(c: dict) -> list[int]:
    return _between(c["lens"], c["batch"], c["lo"], c["hi"])


def _prefill_lens(c: dict) -> tuple[list[int], list[int]]:
    """(cached, new) tokens of each sequence."""
    new = _between(c["lens"], c["seqs"], c["lo"], c["hi"])
    cached = _between(c["lens"] + 1, c["seqs"], c["cached_lo"], c["cached_hi"])
    return cached, new


def _step_lens(c: dict) -> tuple[list[int], list[int]]:
    """(context, new) tokens of each sequence of a step: prompts first, then decodes."""
    ctx = _between(c["lens"], c["rows"], c["lo"], c["hi"]) if c["rows"] else []
    new = [1] * c["rows"]
    if c["kind"] == "mixed":
        p = _between(c["lens"] + 1, c["prompts"], c["plo"], c["phi"])
        ctx, new = p + ctx, p + new
    return ctx, new


def work(c: dict) -> dict:
    e = BYTES[c["dtype"]]
    kind = c["kind"]
    if kind == "decode":
        n, b = sum(_decode_lens(c)), c["batch"]
        return {"bytes": 2 * n * c["hkv"] * c["d"] * e + 2 * b * c["hq"] * c["d"] * e,
                "flops": 4 * n * c["hq"] * c["d"]}  # fmt: skip
    if kind == "prefill":
        cached, new = _prefill_lens(c)
        pairs = sum(n * p + n * (n + 1) // 2 for p, n in zip(cached, new))
        return {"bytes": 2 * (sum(cached) + sum(new)) * c["hkv"] * c["d"] * e + 2 * sum(new) * c["hq"] * c["d"] * e,
                "flops": 4 * pairs * c["hq"] * c["d"]}  # fmt: skip
    if kind == "norms":
        t = c["tokens"]
        # x and its norm, q in and out, k and v in and out, positions and slots, cos and sin.
        return {"bytes": t * (2 * HIDDEN * e + 2 * QKV * e + 16 + 2 * D * 4), "flops": 0}
    if kind == "mlp":
        w = 3 * HIDDEN * INTER
        return {"bytes": c["layers"] * (w * e) + 3 * c["rows"] * HIDDEN * e, "flops": 2 * c["rows"] * c["layers"] * w}
    ctx, new = _step_lens(c)
    t = sum(new)
    w = HIDDEN * QKV + HQ * D * HIDDEN + 3 * HIDDEN * INTER
    pairs = sum(n * (s - n) + n * (n + 1) // 2 for s, n in zip(ctx, new))
    kv = 2 * HKV * D * e
    heads = len(new)  # rows through the output head
    return {"bytes": c["layers"] * (w * e + sum(ctx) * kv + t * kv) + VOCAB * HIDDEN * e + heads * VOCAB * 4,
            "flops": c["layers"] * (2 * t * w + 4 * pairs * HQ * D) + 2 * heads * VOCAB * HIDDEN}  # fmt: skip


# About four times what each kind's outputs differ by from the same computation in 64 bits:
# what the roundings of its types give (measured relative errors: decode 1.5e-7 fp32, 2.1e-4
# fp16, 1.7e-3 bf16; prefill 2.9e-4 fp16, 1.6e-3 bf16; norms 3.6e-4 fp16; MLP layers 6.8e-3
# bf16; whole steps 5e-3 fp16, 1.6e-2 bf16, the last stated at the most that says anything).
TOLERANCE = {
    ("decode", "fp32"): {"rel": 1e-6, "max": 4e-5},
    ("decode", "fp16"): {"rel": 8e-4, "max": 6e-3},
    ("decode", "bf16"): {"rel": 7e-3, "max": 5e-2},
    ("prefill", "fp16"): {"rel": 1.2e-3, "max": 1.5e-2},
    ("prefill", "bf16"): {"rel": 6.5e-3, "max": 6e-2},
    ("norms", "fp16"): {"rel": 1.5e-3, "max": 8e-3},
    ("norms", "bf16"): {"rel": 1.2e-2, "max": 6e-2},
    ("mlp", "fp16"): {"rel": 3.5e-3, "max": 3e-2},
    ("mlp", "bf16"): {"rel": 2.7e-2, "max": 0.2},
    ("step", "fp16"): {"rel": 2e-2, "max": 0.12},
    ("step", "bf16"): {"rel": 3e-2, "max": 0.4},
    ("mixed", "fp16"): {"rel": 2e-2, "max": 0.12},
    ("mixed", "bf16"): {"rel": 3e-2, "max": 0.4},
}


def tolerance(c: dict) -> dict:
    return TOLERANCE[c["kind"], c["dtype"]]


# ---- inputs ------------------------------------------------------------------------------
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _randn(g: torch.Generator, *shape: int, dtype: torch.dtype, scale: float = 1.0) -> torch.Tensor:
    x = torch.randn(shape, generator=g, device=DEVICE, dtype=dtype)
    return x if scale == 1.0 else x.mul_(scale)


def _norm_weight(g: torch.Generator, n: int, dtype: torch.dtype) -> torch.Tensor:
    return (1.0 + 0.1 * torch.randn(n, generator=g, device=DEVICE)).to(dtype)


def _blocks(seed: int, lens: list[int], bs: int) -> tuple[list[list[int]], int]:
    """Each sequence's cache blocks, scattered at random over the pool, and their count."""
    need = [-(-n // bs) for n in lens]
    perm = torch.randperm(sum(need), generator=torch.Generator().manual_seed(seed)).tolist()
    out, at = [], 0
    for k in need:
        out.append(perm[at : at + k])
        at += k
    return out, sum(need)


def _table(blocks: list[list[int]]) -> torch.Tensor:
    width = max(len(b) for b in blocks)
    return torch.tensor([b + [0] * (width - len(b)) for b in blocks], dtype=torch.int32, device=DEVICE)


def _i32(xs: list[int]) -> torch.Tensor:
    return torch.tensor(xs, dtype=torch.int32, device=DEVICE)


def _decode_inputs(c: dict, seed: int) -> dict:
    g, dt, lens = _gen(seed), DTYPES[c["dtype"]], _decode_lens(c)
    blocks, nb = _blocks(seed, lens, c["bs"])
    shape = (nb * c["bs"], c["hkv"], c["d"])
    return {"q": _randn(g, c["batch"], c["hq"], c["d"], dtype=dt), "k": _randn(g, *shape, dtype=dt),
            "v": _randn(g, *shape, dtype=dt), "blocks": blocks, "lens": lens}  # fmt: skip


def _prefill_inputs(c: dict, seed: int) -> dict:
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    cached, new = _prefill_lens(c)
    ctx = [p + n for p, n in zip(cached, new)]
    blocks, nb = _blocks(seed, ctx, c["bs"])
    shape = (nb * c["bs"], c["hkv"], c["d"])
    return {"q": _randn(g, sum(new), c["hq"], c["d"], dtype=dt), "k": _randn(g, *shape, dtype=dt),
            "v": _randn(g, *shape, dtype=dt), "blocks": blocks, "new": new, "ctx": ctx}  # fmt: skip


def _norms_inputs(c: dict, seed: int) -> dict:
    g, dt, t = _gen(seed), DTYPES[c["dtype"]], c["tokens"]
    slots = -(-max(t, 16) // 16) * 32  # a pool of about twice the step's tokens
    return {"x": _randn(g, t, HIDDEN, dtype=dt), "w": _norm_weight(g, HIDDEN, dt), "qkv": _randn(g, t, QKV, dtype=dt),
            "qw": _norm_weight(g, D, dt), "kw": _norm_weight(g, D, dt),
            "pos": torch.randint(0, 4096, (t,), generator=g, device=DEVICE),
            "slots": torch.randperm(slots, generator=g, device=DEVICE)[:t],
            "k": _randn(g, slots, HKV, D, dtype=dt), "v": _randn(g, slots, HKV, D, dtype=dt)}  # fmt: skip


def _mlp_inputs(c: dict, seed: int) -> dict:
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    return {"rows": _randn(g, c["rows"], HIDDEN, dtype=dt), "norm": _norm_weight(g, HIDDEN, dt),
            "layers": [(_norm_weight(g, HIDDEN, dt), _randn(g, 2 * INTER, HIDDEN, dtype=dt, scale=0.02),
                        _randn(g, HIDDEN, INTER, dtype=dt, scale=0.02)) for _ in range(c["layers"])]}  # fmt: skip


def _model_inputs(c: dict, seed: int) -> dict:
    """A random-weight model, its cache (earlier tokens' k and v) and the step's tokens."""
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    ctx, new = _step_lens(c)
    w = {"model.embed_tokens.weight": _randn(g, VOCAB, HIDDEN, dtype=dt, scale=0.02),
         "model.norm.weight": _norm_weight(g, HIDDEN, dt)}  # fmt: skip
    for i in range(c["layers"]):
        p = f"model.layers.{i}."
        w[p + "input_layernorm.weight"] = _norm_weight(g, HIDDEN, dt)
        w[p + "post_attention_layernorm.weight"] = _norm_weight(g, HIDDEN, dt)
        w[p + "self_attn.qkv_proj.weight"] = _randn(g, QKV, HIDDEN, dtype=dt, scale=0.02)
        w[p + "self_attn.o_proj.weight"] = _randn(g, HIDDEN, HQ * D, dtype=dt, scale=0.02)
        w[p + "self_attn.q_norm.weight"] = _norm_weight(g, D, dt)
        w[p + "self_attn.k_norm.weight"] = _norm_weight(g, D, dt)
        w[p + "mlp.gate_up_proj.weight"] = _randn(g, 2 * INTER, HIDDEN, dtype=dt, scale=0.02)
        w[p + "mlp.down_proj.weight"] = _randn(g, HIDDEN, INTER, dtype=dt, scale=0.02)
    blocks, nb = _blocks(seed, ctx, 16)
    slots = (nb + 1) * 16  # the last block takes padding rows
    k = _randn(g, c["layers"], slots, HKV, D, dtype=dt)
    v = _randn(g, c["layers"], slots, HKV, D, dtype=dt)
    tokens = torch.randint(0, VOCAB, (sum(new),), generator=torch.Generator().manual_seed(seed)).tolist()
    return {"w": w, "k": k, "v": v, "blocks": blocks, "nb": nb, "ctx": ctx, "new": new, "tokens": tokens}


def _model(c: dict, m: dict) -> tuple[DecodeStep, KVPool, list[PagedTable]]:
    shape = ModelShape(hidden=HIDDEN, num_heads=HQ, num_kv_heads=HKV, head_dim=D, intermediate=INTER, vocab=VOCAB,
                       num_layers=c["layers"], rms_norm_eps=EPS, rope_theta=THETA)  # fmt: skip
    pool = KVPool(shape, m["nb"], 16, DTYPES[c["dtype"]], DEVICE)
    pool.k, pool.v = m["k"], m["v"]
    tables = [PagedTable(b, 16, n) for b, n in zip(m["blocks"], m["ctx"])]
    return DecodeStep(shape, m["w"], pool), pool, tables


def _mlp_pass(m: dict, ids: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    x, pending = m["rows"][ids], None
    for norm, gate_up, down in m["layers"]:
        h = hip_rows.add_rms_norm(x, pending, norm, EPS)
        act = hip_rows.rows_silu_gate_up(h, gate_up)
        pending, _ = hip_rows.rows_linear_partials(act, down)
    h = hip_rows.add_rms_norm(x, pending, m["norm"], EPS, tiled=False)
    return h, x


def prepare(c: dict, seed: int) -> dict:
    kind = c["kind"]
    if kind == "decode":
        m = _decode_inputs(c, seed)
        args = (m["q"], m["k"], m["v"], _table(m["blocks"]), _i32(m["lens"]), c["d"] ** -0.5, c["bs"])
        return {"kind": kind, "args": args, "splits": c["splits"] or None}
    if kind == "prefill":
        m = _prefill_inputs(c, seed)
        starts = [sum(m["new"][:i]) for i in range(len(m["new"]))]
        return {"kind": kind, "args": (m["q"], m["k"], m["v"], _table(m["blocks"]), _i32(starts), _i32(m["new"]),
                                       _i32(m["ctx"]), c["d"] ** -0.5, c["bs"], max(m["new"]))}  # fmt: skip
    if kind == "norms":
        m, t = _norms_inputs(c, seed), c["tokens"]
        q, k, v = torch.split(m["qkv"], [HQ * D, HKV * D, HKV * D], dim=1)
        return {"kind": kind, "x": m["x"], "w": m["w"], "pos": m["pos"],
                "qkv": (q.view(t, HQ, D), k.view(t, HKV, D), v.view(t, HKV, D), m["qw"], m["kw"]),
                "cache": (m["slots"], m["k"], m["v"])}  # fmt: skip
    if kind == "mlp":
        m = _mlp_inputs(c, seed)
        inputs = DecodeInputs.empty(c["rows"], 1, DEVICE)
        inputs.token_ids.copy_(torch.arange(c["rows"]))
        return {"kind": kind, "graph": DecodeGraph(lambda inp: _mlp_pass(m, inp.token_ids), inputs),
                "keep": (m, inputs)}  # a graph reads the buffers it was captured on  # fmt: skip
    m = _model_inputs(c, seed)
    step, pool, tables = _model(c, m)
    if kind == "step":
        inputs = DecodeInputs.empty(c["rows"], max(len(b) for b in m["blocks"]), DEVICE)
        fill_decode_inputs(inputs, list(zip(m["tokens"], tables)), pool.pad_block)
        return {"kind": kind, "graph": DecodeGraph(step.forward, inputs), "pool": pool, "keep": (step, inputs)}
    items, at = [], 0
    for n, table in zip(m["new"], tables):
        items.append((m["tokens"][at : at + n], table))
        at += n
    return {"kind": kind, "step": step, "batch": build_batch(items, DEVICE), "pool": pool}


def run(s: dict):  # noqa: ANN201
    kind = s["kind"]
    if kind == "decode":
        return hip_attention.launch_paged_decode_split(*s["args"], num_splits=s["splits"])
    if kind == "prefill":
        return hip_prefill.paged_prefill_attention(*s["args"])
    if kind == "norms":
        cos, sin = hip_fused.rope_cos_sin(D, THETA, s["pos"])
        h = hip_fused.rms_norm_rows(s["x"], s["w"], EPS)
        q = hip_fused.qk_norm_rope_store(*s["qkv"], cos, sin, *s["cache"], EPS)
        return {"cos": cos, "sin": sin, "h": h, "q": q, "k": s["cache"][1], "v": s["cache"][2]}
    if kind == "mlp":
        h, x = s["graph"].replay()
        return {"h": h, "x": x}
    if kind == "step":
        return {"logits": s["graph"].replay(), "k": s["pool"].k, "v": s["pool"].v}
    return {"logits": s["step"].forward_batch(s["batch"]), "k": s["pool"].k, "v": s["pool"].v}


# ---- the same results in 64 bits ---------------------------------------------------------
def _slots(blocks: list[int], n: int, bs: int) -> torch.Tensor:
    pos = torch.arange(n, device=DEVICE)
    return torch.tensor(blocks, device=DEVICE)[pos // bs] * bs + pos % bs


def _attend64(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, past: int) -> torch.Tensor:
    """Causal attention of q [n, Hq, D] at positions past .. past + n - 1 over k, v [S, Hkv, D]."""
    group = q.shape[1] // k.shape[1]
    q, k, v = q.double(), k.double(), v.double()
    out = torch.empty_like(q)
    keys = torch.arange(k.shape[0], device=DEVICE)
    for h in range(q.shape[1]):
        for at in range(0, q.shape[0], 2048):
            rows = torch.arange(at, min(at + 2048, q.shape[0]), device=DEVICE)
            s = q[rows, h].contiguous() @ k[:, h // group].t().contiguous() * q.shape[2] ** -0.5
            s.masked_fill_(keys[None, :] > past + rows[:, None], -math.inf)
            out[rows, h] = torch.softmax(s, -1) @ v[:, h // group].contiguous()
    return out


def _decode64(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
    """One query [Hq, D] over k, v [S, Hkv, D]."""
    q = q.double().view(k.shape[1], -1, q.shape[1])
    s = (q * q.shape[2] ** -0.5) @ k.double().permute(1, 2, 0).contiguous()
    return (torch.softmax(s, -1) @ v.double().permute(1, 0, 2).contiguous()).reshape(-1, k.shape[2])


def _norm64(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(pos: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    freq = THETA ** (-torch.arange(0, D, 2, dtype=torch.float64, device=DEVICE) / D)
    a = pos.double()[:, None] * freq[None, :]
    a = torch.cat([a, a], -1)
    return a.cos(), a.sin()


def _rotate64(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    a, b = x.chunk(2, -1)
    return x * cos[:, None] + torch.cat([-b, a], -1) * sin[:, None]


def _mlp64(h: torch.Tensor, gate_up: torch.Tensor, down: torch.Tensor) -> torch.Tensor:
    gate, up = (h @ gate_up.double().t()).chunk(2, -1)
    return (F.silu(gate) * up) @ down.double().t()


def exact(c: dict, seed: int):  # noqa: ANN201
    kind = c["kind"]
    if kind == "decode":
        m = _decode_inputs(c, seed)
        rows = []
        for b, n in enumerate(m["lens"]):
            sl = _slots(m["blocks"][b], n, c["bs"])
            rows.append(_decode64(m["q"][b], m["k"][sl], m["v"][sl]))
        return torch.stack(rows)
    if kind == "prefill":
        m = _prefill_inputs(c, seed)
        out, at = [], 0
        for b, (n, s) in enumerate(zip(m["new"], m["ctx"])):
            sl = _slots(m["blocks"][b], s, c["bs"])
            out.append(_attend64(m["q"][at : at + n], m["k"][sl], m["v"][sl], s - n))
            at += n
        return torch.cat(out)
    if kind == "norms":
        m, t = _norms_inputs(c, seed), c["tokens"]
        cos, sin = _rope64(m["pos"])
        q, k, v = (x.double() for x in torch.split(m["qkv"], [HQ * D, HKV * D, HKV * D], dim=1))
        kc, vc = m["k"].double(), m["v"].double()
        kc[m["slots"]] = _rotate64(_norm64(k.view(t, HKV, D), m["kw"]), cos, sin)
        vc[m["slots"]] = v.view(t, HKV, D)
        return {"cos": cos, "sin": sin, "h": _norm64(m["x"].double(), m["w"]),
                "q": _rotate64(_norm64(q.view(t, HQ, D), m["qw"]), cos, sin), "k": kc, "v": vc}  # fmt: skip
    if kind == "mlp":
        m = _mlp_inputs(c, seed)
        x = m["rows"].double()
        for norm, gate_up, down in m["layers"]:
            x = x + _mlp64(_norm64(x, norm), gate_up, down)
        return {"h": _norm64(x, m["norm"]), "x": x}
    m = _model_inputs(c, seed)
    w, kc, vc = m["w"], m["k"].double(), m["v"].double()
    pos = torch.cat([torch.arange(s - n, s, device=DEVICE) for s, n in zip(m["ctx"], m["new"])])
    seqs = [_slots(b, s, 16) for b, s in zip(m["blocks"], m["ctx"])]
    new = torch.cat([sl[len(sl) - n :] for sl, n in zip(seqs, m["new"])])
    cos, sin = _rope64(pos)
    x = w["model.embed_tokens.weight"][torch.tensor(m["tokens"], device=DEVICE)].double()
    t = x.shape[0]
    for i in range(c["layers"]):
        p = f"model.layers.{i}."
        h = _norm64(x, w[p + "input_layernorm.weight"])
        q, k, v = torch.split(h @ w[p + "self_attn.qkv_proj.weight"].double().t(), [HQ * D, HKV * D, HKV * D], 1)
        q = _rotate64(_norm64(q.reshape(t, HQ, D), w[p + "self_attn.q_norm.weight"]), cos, sin)
        kc[i, new] = _rotate64(_norm64(k.reshape(t, HKV, D), w[p + "self_attn.k_norm.weight"]), cos, sin)
        vc[i, new] = v.reshape(t, HKV, D)
        out, at = [], 0
        for sl, n in zip(seqs, m["new"]):
            ks, vs = kc[i, sl], vc[i, sl]
            out.append(_decode64(q[at], ks, vs)[None] if n == 1 else _attend64(q[at : at + n], ks, vs, len(sl) - n))
            at += n
        x = x + torch.cat(out).reshape(t, HQ * D) @ w[p + "self_attn.o_proj.weight"].double().t()
        x = x + _mlp64(_norm64(x, w[p + "post_attention_layernorm.weight"]), w[p + "mlp.gate_up_proj.weight"],
                       w[p + "mlp.down_proj.weight"])  # fmt: skip
    last = torch.tensor(m["new"], device=DEVICE).cumsum(0) - 1
    logits = _norm64(x[last], w["model.norm.weight"]) @ w["model.embed_tokens.weight"].double().t()
    return {"logits": logits, "k": kc, "v": vc}
