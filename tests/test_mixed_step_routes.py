"""Which launches a mixed step makes (``DecodeStep.forward_batch``), on the CPU: the tables and
lengths that reach the attention kernels, with the kernels themselves replaced."""

from __future__ import annotations

import pytest
import torch

from tinyserve_amd import hip_attention, hip_prefill
from tinyserve_amd.decode_step import DecodeStep, KVPool, ModelShape, random_weights
from tinyserve_amd.step_inputs import PagedTable, build_batch

BS = 16
SHAPE = ModelShape(hidden=64, num_heads=16, num_kv_heads=8, head_dim=128, intermediate=64, vocab=32, num_layers=1)


@pytest.mark.parametrize(("prompt", "cached", "cuts"), [(100, 0, False), (40, 0, False), (100, 3000, True)])
def test_prefill_width_is_the_prompts_own(prompt: int, cached: int, cuts: bool, monkeypatch) -> None:  # noqa: ANN001
    # A prompt beside decodes of 4096 tokens: the prefill launch gets the prompt's blocks
    # only, so a fresh one does not get the key cut's plan, merge and workspace; a chunk
    # behind a long cached prefix does.
    shapes = [(prompt, prompt + cached)] + [(1, 4096)] * 16
    items, at = [], 0
    for new, total in shapes:
        n = -(-total // BS)
        items.append(([1] * new, PagedTable(list(range(at, at + n)), BS, total)))
        at += n
    batch = build_batch(items)
    step = DecodeStep(SHAPE, random_weights(SHAPE, torch.float16, "cpu", 0), KVPool(SHAPE, 1, BS, torch.float16, "cpu"))
    seen = {}

    def prefill(q, k, v, tables, starts, qlens, lens, scale, bs, max_q, out):  # noqa: ANN001, ANN202
        seen.update(tables=tables, lens=lens, max_q=max_q)

    monkeypatch.setattr(hip_prefill, "paged_prefill_attention", prefill)
    monkeypatch.setattr(hip_attention, "launch_paged_decode_split_into", lambda *a: None)
    monkeypatch.setattr(step, "_run", lambda ids, pos, slots, attend, rows: attend(
        0, torch.zeros(len(ids), 16, 128, dtype=torch.float16)))  # fmt: skip
    step.forward_batch(batch)
    width = -(-(prompt + cached) // BS)
    assert torch.equal(seen["tables"], batch.block_tables[:1, :width]) and seen["lens"].tolist() == [prompt + cached]
    floats = hip_prefill._workspace_floats(-1, 1, 16, 8, 128, BS, seen["max_q"], seen["tables"].shape[1] * BS,
                                           torch.float16)  # fmt: skip
    assert (floats > 0) == cuts
