"""The decode step through the HIP kernels (``tinyserve_amd.decode_step``) on the GPU.

Mirrors the reference's tests/test_decode_inputs.py:80-130, tests/test_cuda_graphs.py and
tests/test_batched_forward.py: the step's logits and cache writes against a reference step
composed from the oracle (``rms_norm``, ``rope_cos_sin``, ``qk_norm_rope_store_ref``,
``decode_ref`` / ``prefill_ref``) and plain fp32 matrix products on the CPU, on a tiny
random Qwen3 in fp32; padding rows leave real rows unchanged; a captured graph gives the
eager result on every replay, with other work between replays; a mixed prefill + decode
step (``forward_batch``) gives the oracle's logits and the same logits as each sequence
run alone.
"""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from oracle import ref
from tinyserve_amd.decode_step import (DecodeGraph, DecodeStep, KVPool, ModelShape, random_context_tables,
                                       random_weights, rope_tables)  # fmt: skip
from tinyserve_amd.hip_fused import rms_norm_rows
from tinyserve_amd.step_inputs import Batch, DecodeInputs, PagedTable, build_batch, fill_decode_inputs

pytestmark = pytest.mark.gpu
DEVICE = "cuda"
# Bound on the config-5 logits of the fp16 step against the all-fp32 oracle composition:
# fp16 activations and GEMM outputs over 28 layers drift from float32 by ~0.02 (measured
# 0.019 at 16 splits and 0.021 with the policy, logits up to 3.2 in magnitude); the bound
# leaves 2.5x that.
LOGITS_ATOL = 0.05
# bf16 (8 significant bits) drifts further: measured 0.157 with the row-batch projections
# and the policy; 2.5x that, as for fp16.
CONFIG5_LOGITS_ATOL = {torch.float16: LOGITS_ATOL, torch.bfloat16: 0.4}
# The 2-layer tiny model's 16-bit logits against the fp32 composition: measured 0.0010-0.0012
# (fp16) and 0.0077-0.0080 (bf16) on both projection paths; the bounds leave ~4x that.
TINY_LOGITS_ATOL = {torch.float16: 5e-3, torch.bfloat16: 3e-2}
TINY = ModelShape(hidden=256, num_heads=4, num_kv_heads=2, head_dim=64, intermediate=512, vocab=1000,
                  num_layers=2)  # fmt: skip


def setup(lens: list[int], rows: int, dtype: torch.dtype = torch.float32, shape: ModelShape = TINY,
          block_size: int = 4, seed: int = 0):  # fmt: skip
    w = random_weights(shape, dtype, DEVICE, seed)
    blocks, nb = random_context_tables(lens, block_size, seed=seed)
    pool = KVPool(shape, nb + 3, block_size, dtype, DEVICE)  # blocks nb .. nb + 2 are spare
    g = torch.Generator(device="cpu").manual_seed(seed + 1)
    pool.k.copy_(torch.randn(pool.k.shape, generator=g).to(dtype))  # stands in for earlier steps
    pool.v.copy_(torch.randn(pool.v.shape, generator=g).to(dtype))
    tabs = [PagedTable(b, block_size, n) for b, n in zip(blocks, lens)]
    inp = DecodeInputs.empty(rows, max(len(b) for b in blocks) + 1, DEVICE)
    tokens = [(7 * i + 3) % shape.vocab for i in range(len(lens))]
    fill_decode_inputs(inp, list(zip(tokens, tabs)), pool.pad_block)
    return w, pool, tabs, inp


def reference_step(shape: ModelShape, w: dict, k: torch.Tensor, v: torch.Tensor, inp: DecodeInputs | Batch,
                   block_size: int, device: str = "cpu") -> torch.Tensor:  # fmt: skip
    """The reference's forward_decode (a ``DecodeInputs``) or forward_batch (a ``Batch``:
    every sequence through the per-sequence prefill reference) composed from the oracle,
    fp32 on ``device`` (``k``, ``v``: float32 caches there); logits of every row; writes
    k, v."""
    cw = {n: t.float().to(device) for n, t in w.items()}
    bt, lens = inp.block_tables.cpu(), inp.context_lens.cpu()
    if isinstance(inp, Batch):
        tok, pos, slots = inp.token_ids.cpu(), inp.positions.cpu(), inp.new_slots.cpu()
        qs, ql = inp.q_starts.cpu(), inp.q_lens.cpu()

        def attend(q: torch.Tensor, kc: torch.Tensor, vc: torch.Tensor) -> torch.Tensor:
            return ref.prefill_ref(q, kc, vc, bt, qs, ql, lens, shape.head_dim**-0.5, block_size)
    else:
        tok, pos, slots = inp.token_ids.cpu(), inp.positions.cpu(), inp.slots.cpu()

        def attend(q: torch.Tensor, kc: torch.Tensor, vc: torch.Tensor) -> torch.Tensor:
            return ref.decode_ref(q, kc, vc, bt, lens, shape.head_dim**-0.5, block_size)

    cos, sin = ref.rope_cos_sin(shape.head_dim, shape.rope_theta, pos)
    tok, slots = tok.to(device), slots.to(device)
    x = cw["model.embed_tokens.weight"][tok]
    n, s = x.shape[0], shape
    for i in range(s.num_layers):
        p = f"model.layers.{i}."
        h = ref.rms_norm(x, cw[p + "input_layernorm.weight"], s.rms_norm_eps)
        q, kk, vv = torch.split(h @ cw[p + "self_attn.qkv_proj.weight"].T, [s.q_size, s.kv_size, s.kv_size], 1)
        q = ref.qk_norm_rope_store_ref(
            q.reshape(n, s.num_heads, s.head_dim), kk.reshape(n, s.num_kv_heads, s.head_dim),
            vv.reshape(n, s.num_kv_heads, s.head_dim), cw[p + "self_attn.q_norm.weight"],
            cw[p + "self_attn.k_norm.weight"], cos, sin, slots, k[i], v[i], s.rms_norm_eps)  # fmt: skip
        attn = attend(q, k[i], v[i])
        x = x + attn.reshape(n, s.q_size) @ cw[p + "self_attn.o_proj.weight"].T
        h = ref.rms_norm(x, cw[p + "post_attention_layernorm.weight"], s.rms_norm_eps)
        gate, up = (h @ cw[p + "mlp.gate_up_proj.weight"].T).chunk(2, dim=1)
        x = x + (F.silu(gate) * up) @ cw[p + "mlp.down_proj.weight"].T
    x = ref.rms_norm(x, cw["model.norm.weight"], s.rms_norm_eps)
    return x @ cw["model.embed_tokens.weight"].T


@pytest.mark.parametrize("rows", [4, 8])  # no padding; 4 padding rows
@pytest.mark.parametrize("splits", [None, 1, 3])
def test_step_matches_the_reference_step(rows: int, splits: int | None) -> None:
    lens = [6, 1, 13, 4]
    w, pool, tabs, inp = setup(lens, rows)
    k0, v0 = pool.k.cpu(), pool.v.cpu()
    kr, vr = k0.clone(), v0.clone()
    want = reference_step(TINY, w, kr, vr, inp, pool.block_size)
    got = DecodeStep(TINY, w, pool, splits).forward(inp).cpu()
    assert got.shape == (rows, TINY.vocab) and got.dtype == torch.float32
    torch.testing.assert_close(got[: len(lens)], want[: len(lens)], atol=1e-4, rtol=1e-4)
    # The cache changed at the new tokens' slots (and the padding block) only, to the
    # reference's values.
    new = set(inp.slots.cpu().tolist())
    changed = ((pool.k.cpu() != k0) | (pool.v.cpu() != v0)).flatten(2).any(-1).any(0)
    assert set(changed.nonzero().flatten().tolist()) <= new
    real = inp.slots.cpu()[: len(lens)]
    torch.testing.assert_close(pool.k.cpu()[:, real], kr[:, real], atol=1e-5, rtol=1e-5)
    # v is the QKV product copied as is: only the GEMMs' rounding (GPU vs CPU) differs.
    torch.testing.assert_close(pool.v.cpu()[:, real], vr[:, real], atol=1e-5, rtol=1e-5)


def test_padding_rows_do_not_change_real_rows() -> None:
    outs = []
    for rows in (2, 8):
        w, pool, tabs, inp = setup([5, 2], rows, seed=4)
        outs.append(DecodeStep(TINY, w, pool).forward(inp)[:2].cpu())
    torch.testing.assert_close(outs[1], outs[0], atol=1e-5, rtol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_graph_replays_equal_the_eager_step(dtype: torch.dtype) -> None:
    lens = [9, 30, 2, 17, 5]
    w, pool, tabs, inp = setup(lens, 8, dtype, seed=7)
    step = DecodeStep(TINY, w, pool)
    graph = DecodeGraph(step.forward, inp)
    spare = iter(range(pool.pad_block - 3, pool.pad_block))
    for it in range(3):
        # A new step: every sequence grows by one token (the new token's block may be new).
        for t in tabs:
            t.num_tokens += 1
            if len(t.blocks) * t.block_size < t.num_tokens:
                t.blocks.append(next(spare))
        fill_decode_inputs(inp, [((it * 5 + j) % TINY.vocab, t) for j, t in enumerate(tabs)], pool.pad_block)
        k_before, v_before = pool.k.clone(), pool.v.clone()
        got = graph.replay().clone()
        torch.cuda.synchronize()
        k_after, v_after = pool.k.clone(), pool.v.clone()
        pool.k.copy_(k_before)
        pool.v.copy_(v_before)
        want = step.forward(inp)  # eager, on the same cache state
        torch.cuda.synchronize()
        torch.testing.assert_close(got, want, atol=0, rtol=0)
        assert torch.equal(pool.k, k_after) and torch.equal(pool.v, v_after)
        torch.randn(1 << 20, device=DEVICE).sum().item()  # unrelated eager work between replays


def mixed_setup(cached: list[int], new: list[int], seed: int, block_size: int = 4):
    """A tiny fp32 model, a filled pool and a ``Batch`` of ``new[b]`` tokens per sequence
    after ``cached[b]`` earlier ones (whose k/v the random pool stands in for)."""
    w, pool, tabs, _ = setup([c + n for c, n in zip(cached, new)], len(cached), seed=seed, block_size=block_size)
    g = torch.Generator(device="cpu").manual_seed(seed + 2)
    items = [(torch.randint(0, TINY.vocab, (n,), generator=g).tolist(), t) for n, t in zip(new, tabs)]
    return w, pool, tabs, items


@pytest.mark.parametrize(
    "cached,new",
    [
        ([5, 0, 9, 2, 0], [3, 7, 1, 1, 1]),  # prefill and decode sequences interleaved
        ([0, 3], [17, 40]),  # prefill only, one from scratch
        ([6, 1, 13], [1, 1, 1]),  # decode only
        ([30], [1]),
    ],
)
def test_mixed_step_matches_the_reference_step(cached: list[int], new: list[int]) -> None:
    w, pool, tabs, items = mixed_setup(cached, new, seed=11)
    batch = build_batch(items, DEVICE)
    kr, vr = pool.k.cpu(), pool.v.cpu()
    want = reference_step(TINY, w, kr, vr, batch, pool.block_size)[batch.last_rows.cpu()]
    got = DecodeStep(TINY, w, pool).forward_batch(batch).cpu()
    assert got.shape == (len(new), TINY.vocab) and got.dtype == torch.float32
    torch.testing.assert_close(got, want, atol=1e-4, rtol=1e-4)
    slots = batch.new_slots.cpu()
    torch.testing.assert_close(pool.k.cpu()[:, slots], kr[:, slots], atol=1e-5, rtol=1e-5)
    torch.testing.assert_close(pool.v.cpu()[:, slots], vr[:, slots], atol=1e-5, rtol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_mixed_step_row_projections_match_the_reference_step(dtype: torch.dtype) -> None:
    # forward_batch (prefill and decode sequences in one step) in 16-bit types: the
    # row-batch projection kernels (up to 256 rows) and library GEMMs, each against the
    # oracle-composed fp32 step.
    cached, new = [5, 0, 9, 2, 0], [3, 7, 1, 1, 40]
    outs = {}
    for projections in ("rows", "library"):
        w, pool, tabs, _ = setup([c + n for c, n in zip(cached, new)], len(cached), dtype, seed=17)
        g = torch.Generator(device="cpu").manual_seed(19)
        items = [(torch.randint(0, TINY.vocab, (n,), generator=g).tolist(), t) for n, t in zip(new, tabs)]
        batch = build_batch(items, DEVICE)
        kr, vr = pool.k.float().cpu(), pool.v.float().cpu()
        want = reference_step(TINY, w, kr, vr, batch, pool.block_size)[batch.last_rows.cpu()]
        step = DecodeStep(TINY, w, pool, None, projections)
        outs[projections] = step.forward_batch(batch).cpu()
        err = (outs[projections] - want).abs().max().item()
        print(f"[mixed {dtype}] {projections}: logits max-abs {err:.3g} vs fp32")
        torch.testing.assert_close(outs[projections], want, atol=TINY_LOGITS_ATOL[dtype], rtol=0)
    torch.testing.assert_close(outs["rows"], outs["library"], atol=TINY_LOGITS_ATOL[dtype], rtol=0)


def test_mixed_step_equals_each_sequence_alone() -> None:
    # test_batched_forward.py: a sequence's logits do not depend on what else is batched.
    cached, new = [4, 0, 11, 7], [1, 9, 1, 5]
    w, pool, tabs, items = mixed_setup(cached, new, seed=3)
    k0, v0 = pool.k.clone(), pool.v.clone()
    step = DecodeStep(TINY, w, pool)
    together = step.forward_batch(build_batch(items, DEVICE))
    for b, item in enumerate(items):
        pool.k.copy_(k0)
        pool.v.copy_(v0)
        alone = step.forward_batch(build_batch([item], DEVICE))
        torch.testing.assert_close(alone[0], together[b], atol=1e-5, rtol=1e-5)


def test_decode_only_batch_equals_the_decode_step() -> None:
    # Same rows, same table width (so the same split policy): bit-identical logits.
    lens = [6, 1, 13, 4]
    w, pool, tabs, _ = setup(lens, len(lens), seed=5)
    items = [((7 * i + 3) % TINY.vocab, t) for i, t in enumerate(tabs)]
    batch = build_batch([([tok], tab) for tok, tab in items], DEVICE)
    inp = DecodeInputs.empty(len(lens), batch.block_tables.shape[1], DEVICE)
    fill_decode_inputs(inp, items, pool.pad_block)
    k0, v0 = pool.k.clone(), pool.v.clone()
    step = DecodeStep(TINY, w, pool)
    want = step.forward(inp)
    pool.k.copy_(k0)
    pool.v.copy_(v0)
    got = step.forward_batch(batch)
    torch.testing.assert_close(got, want, atol=0, rtol=0)


CONFIG5 = ModelShape()  # Qwen3-0.6B: hidden 1024, 16/8 heads of 128, inter 3072, vocab 151936, 28 layers
CHECKED_LAYERS = (0, 13, 27)


@pytest.mark.parametrize(("splits", "projections", "dtype"),
                         [(16, "rows", torch.float16), (None, "rows", torch.float16),
                          (None, "library", torch.float16), (None, "rows", torch.bfloat16)])  # fmt: skip
def test_config_5_step_at_full_shape(splits: int | None, projections: str, dtype: torch.dtype,
                                     monkeypatch: pytest.MonkeyPatch) -> None:  # fmt: skip
    # BASELINE config 5 at its real shape, as bench.py runs it: the random-init
    # Qwen3-0.6B-shaped model in fp16 (and once in bf16), B=64, contexts ~ U[1024, 4096], 16-token blocks
    # scattered over the pool; the reference's 16 splits (HBM partials + combine) and
    # this library's policy; the projections on the row-batch kernels (the default) and
    # on library GEMMs. Layers 0, 13 and 27: the fused kernel's q and cache writes
    # and the attention output against the oracle on the same fp16 inputs, at the
    # contract's bounds. Then the logits of the whole 28-layer step against the
    # oracle-composed step in float32 (run on the GPU as the checker).
    from tests.helpers import ULP, assert_contract
    from tinyserve_amd import hip_attention, hip_fused

    s, bs, batch, seed = CONFIG5, 16, 64, 5
    w = random_weights(s, dtype, DEVICE, seed)
    g = torch.Generator().manual_seed(seed)
    lens = torch.randint(1024, 4097, (batch,), generator=g).tolist()
    blocks, nb = random_context_tables(lens, bs, seed=seed)
    pool = KVPool(s, nb, bs, dtype, DEVICE)
    gd = torch.Generator(device=DEVICE).manual_seed(seed)
    pool.k.normal_(generator=gd)
    pool.v.normal_(generator=gd)
    k32, v32 = pool.k.float(), pool.v.float()  # the caches before the step, for the reference
    tabs = [PagedTable(b, bs, n) for b, n in zip(blocks, lens)]
    inp = DecodeInputs.empty(batch, max(len(b) for b in blocks), DEVICE)
    fill_decode_inputs(inp, [((97 * i) % s.vocab, t) for i, t in enumerate(tabs)], pool.pad_block)

    seen: dict[str, list] = {"qk": [], "attn": []}
    qk_kernel, attn_kernel = hip_fused.qk_norm_rope_store, hip_attention.launch_paged_decode_split

    def qk(q, k, v, qw, kw, cos, sin, slots, kc, vc, eps):  # noqa: ANN001, ANN202
        out = qk_kernel(q, k, v, qw, kw, cos, sin, slots, kc, vc, eps)
        seen["qk"].append((q.clone(), k.clone(), v.clone(), qw, kw, cos, sin, slots, out.clone()))
        return out

    def attn(q, kc, vc, bt, cl, scale, block_size, num_splits=None, tile=None):  # noqa: ANN001, ANN202
        out = attn_kernel(q, kc, vc, bt, cl, scale, block_size, num_splits, tile)
        seen["attn"].append((q.clone(), out.clone()))
        return out

    monkeypatch.setattr(hip_fused, "qk_norm_rope_store", qk)
    monkeypatch.setattr(hip_attention, "launch_paged_decode_split", attn)
    step = DecodeStep(s, w, pool, splits, projections)
    assert step.projections == projections
    logits = step.forward(inp)
    torch.cuda.synchronize()
    assert len(seen["qk"]) == len(seen["attn"]) == s.num_layers
    new = inp.slots[:batch]
    for i in CHECKED_LAYERS:
        q, k, v, qw, kw, cos, sin, slots, q_out = seen["qk"][i]
        assert torch.equal(slots, new)
        for name, x, wt, got in (("q", q, qw, q_out), ("k cache", k, kw, pool.k[i][new])):
            # The oracle's rms_norm rounds x/rms to fp16 and multiplies by the fp16 weight
            # (layers.py:34-38); RoPE then rotates in float32, compared before its final
            # rounding. One fp16 ulp of the normalised intermediate per rotate-half pair
            # is allowed on top of the contract (a near-tie rounded the other way).
            n = ref.rms_norm(x, wt, s.rms_norm_eps).float()
            h = s.head_dim // 2
            e = ULP[dtype] * (n[..., :h].abs() + n[..., h:].abs())
            want = ref.apply_rope(n, cos, sin)
            assert_contract(got, want, dtype, f"layer {i} {name}", torch.cat([e, e], -1))
        assert torch.equal(pool.v[i][new], v), f"layer {i}: the v scatter is an exact copy"
        q_att, out = seen["attn"][i]
        want = ref.decode_ref(q_att.float(), pool.k[i].float(), pool.v[i].float(), inp.block_tables,
                              inp.context_lens, s.head_dim**-0.5, bs)  # fmt: skip
        assert_contract(out, want, dtype, f"layer {i} attention (splits={splits})")
    want_logits = reference_step(s, w, k32, v32, inp, bs, device=DEVICE)
    err = (logits.float() - want_logits).abs().max().item()
    scale = want_logits.abs().max().item()
    print(f"[config 5] splits={splits} {projections} {dtype}: logits max-abs {err:.3g} (max |logit| {scale:.3g})")
    # fp16 activations over 28 layers against an all-fp32 composition: stated bound.
    torch.testing.assert_close(logits.float(), want_logits, atol=CONFIG5_LOGITS_ATOL[dtype], rtol=0)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows", [5, 8])
def test_row_projections_match_the_reference_step(dtype: torch.dtype, rows: int) -> None:
    # The tiny model in 16-bit types through both projection paths: each against the
    # oracle-composed fp32 step, and the two against each other (same kernels elsewhere).
    lens = [9, 30, 2, 17, 5]
    outs = {}
    for projections in ("rows", "library"):
        w, pool, tabs, inp = setup(lens, rows, dtype, seed=13)
        kr, vr = pool.k.float().cpu(), pool.v.float().cpu()
        want = reference_step(TINY, w, kr, vr, inp, pool.block_size)[: len(lens)]
        step = DecodeStep(TINY, w, pool, None, projections)
        assert step.projections == projections
        outs[projections] = step.forward(inp)[: len(lens)].cpu()
        err = (outs[projections] - want).abs().max().item()
        print(f"[tiny {dtype}] {projections}: logits max-abs {err:.3g} vs fp32")
        torch.testing.assert_close(outs[projections], want, atol=TINY_LOGITS_ATOL[dtype], rtol=0)
        # The new tokens' k/v went to the cache (the v copy through the fused kernel).
        real = inp.slots.cpu()[: len(lens)]
        torch.testing.assert_close(pool.v.float().cpu()[:, real], vr[:, real],
                                   atol=2e-3 if dtype == torch.float16 else 2e-2, rtol=2e-2)  # fmt: skip
    torch.testing.assert_close(outs["rows"], outs["library"], atol=TINY_LOGITS_ATOL[dtype], rtol=0)


def test_projection_choice() -> None:
    w, pool, _, _ = setup([3], 1, torch.float32)
    assert DecodeStep(TINY, w, pool).projections == "library"  # fp32: no MFMA projection kernels
    with pytest.raises(ValueError, match="row-batch"):
        DecodeStep(TINY, w, pool, projections="rows")
    with pytest.raises(ValueError, match="projections"):
        DecodeStep(TINY, w, pool, projections="fast")
    w16, pool16, _, _ = setup([3], 1, torch.float16)
    assert DecodeStep(TINY, w16, pool16).projections == "rows"


# bf16 config 5 through the row-batch projections at the stated 16 splits against the
# library projections at the policy's split count. Both round every projection, residual
# add, norm and activation to bf16 where model.py:137-179 rounds, so the two differ only by
# fp32 summation order (a rare one-ulp flip of a rounded value, carried through 28 layers):
# measured 0.117 at max |logit| 3.3 (the fp16 paths differ by 0.017); the library GEMM's
# summation order may change with its kernel choice, so the bound leaves 2x.
CONFIG5_BF16_PATHS_ATOL = 0.25


def test_config_5_bf16_rows_at_16_splits_against_library_projections() -> None:
    s, bs, batch, seed = CONFIG5, 16, 64, 7
    dtype = torch.bfloat16
    w = random_weights(s, dtype, DEVICE, seed)
    g = torch.Generator().manual_seed(seed)
    lens = torch.randint(1024, 4097, (batch,), generator=g).tolist()
    blocks, nb = random_context_tables(lens, bs, seed=seed)
    pool = KVPool(s, nb, bs, dtype, DEVICE)
    gd = torch.Generator(device=DEVICE).manual_seed(seed)
    pool.k.normal_(generator=gd)
    pool.v.normal_(generator=gd)
    k0, v0 = pool.k.clone(), pool.v.clone()
    tabs = [PagedTable(b, bs, n) for b, n in zip(blocks, lens)]
    inp = DecodeInputs.empty(batch, max(len(b) for b in blocks), DEVICE)
    fill_decode_inputs(inp, [((89 * i) % s.vocab, t) for i, t in enumerate(tabs)], pool.pad_block)
    rows = DecodeStep(s, w, pool, 16, "rows").forward(inp)
    pool.k.copy_(k0)
    pool.v.copy_(v0)
    lib = DecodeStep(s, w, pool, None, "library").forward(inp)
    torch.cuda.synchronize()
    err = (rows.float() - lib.float()).abs().max().item()
    print(f"[config 5 bf16] rows/16 splits vs library/policy: logits max-abs {err:.3g} "
          f"(max |logit| {lib.float().abs().max().item():.3g})")
    torch.testing.assert_close(rows.float(), lib.float(), atol=CONFIG5_BF16_PATHS_ATOL, rtol=0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_layers_one_by_one_give_the_step(dtype: torch.dtype) -> None:
    # ``layer`` adds its last residual itself, where the step leaves it to the next norm: the
    # same sums, bit for bit.
    w, pool, _, inp = setup([3, 17, 40, 9, 1, 22, 5, 13], 8, dtype)
    step = DecodeStep(TINY, w, pool, projections="library")
    want = step.forward(inp)
    cos, sin = rope_tables(TINY.head_dim, TINY.rope_theta, inp.positions)
    x = w["model.embed_tokens.weight"][inp.token_ids]
    for i in range(TINY.num_layers):
        x = step.layer(i, x, cos, sin, inp.slots, lambda i, q: step._attention(i, q, inp))
    h = rms_norm_rows(x, w["model.norm.weight"], TINY.rms_norm_eps)
    assert torch.equal(F.linear(h, w["model.embed_tokens.weight"]).float(), want)
