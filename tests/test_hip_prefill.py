"""The HIP varlen prefill kernel must match the oracle (GPU).

Mirrors the reference's tests/test_triton_prefill.py: the reference result is the
oracle's ``prefill_ref`` (``paged_gqa_attention`` one sequence at a time); every cache
slot no sequence owns is NaN and block-table padding points at a NaN block. fp32 runs
the exact-fp32 path; fp16 / bf16 at head_dim 64 / 128 run the MFMA kernel, whose P is
rounded to the input dtype before P.V as in the reference kernel. Tolerances:
tests/helpers.py.
"""

from __future__ import annotations

from dataclasses import replace

import pytest
import torch
from hypothesis import given, settings
from hypothesis import strategies as st

from oracle import ref
from tests.helpers import assert_contract, assert_matches
from tinyserve_amd import hip_prefill
from tinyserve_amd.hip_prefill import paged_prefill_attention
from tinyserve_amd.workloads import PrefillCase, prefill_case, prefill_lengths

pytestmark = pytest.mark.gpu
DEVICE = "cuda"


def on_gpu(c: PrefillCase) -> PrefillCase:
    return PrefillCase(c.q.to(DEVICE), c.k.to(DEVICE), c.v.to(DEVICE), c.tables.to(DEVICE),
                       c.starts.to(DEVICE), c.q_lens.to(DEVICE), c.ctx_lens.to(DEVICE),
                       c.block_size, c.max_q_len)  # fmt: skip


def oracle32(c: PrefillCase) -> torch.Tensor:
    return ref.prefill_ref(c.q.float(), c.k.float(), c.v.float(), c.tables, c.starts, c.q_lens,
                           c.ctx_lens, c.scale, c.block_size)  # fmt: skip


def run(c: PrefillCase, out: torch.Tensor | None = None, **kw: int) -> torch.Tensor:
    g = on_gpu(c)
    return paged_prefill_attention(*g.args(), out=out, **kw)


def check(c: PrefillCase, out: torch.Tensor) -> None:
    want = oracle32(c)
    for r in range(c.tables.shape[0]):
        s, n = int(c.starts[r]), int(c.q_lens[r])
        assert torch.isfinite(out[s : s + n]).all(), f"sequence {r} read an unowned slot"
        assert_matches(out[s : s + n], want[s : s + n], c.q.dtype, f"sequence {r}")


def widened(c: PrefillCase, tokens: int) -> PrefillCase:
    """``c`` under a table of ``tokens`` keys (padding repeats the NaN block)."""
    pad = c.tables[:, -1:].expand(-1, max(tokens // c.block_size - c.tables.shape[1], 0))
    return replace(c, tables=torch.cat([c.tables, pad], dim=1).contiguous())


def shape_of(c: PrefillCase) -> str:
    """The workgroup shape the launch of ``c`` runs."""
    return hip_prefill.prefill_plan(c.tables.shape[0], c.q.shape[1], c.k.shape[1], c.q.shape[2], c.block_size,
                                    c.max_q_len, c.q.shape[0], c.tables.shape[1] * c.block_size,
                                    c.q.dtype)  # fmt: skip


SHAPES = [(4, 4, 8), (4, 2, 8), (4, 1, 8), (16, 8, 128), (8, 2, 64), (16, 2, 128)]
SPECS = [
    [(0, 5)],
    [(0, 37), (0, 1), (0, 9)],
    [(12, 4), (40, 7), (3, 1)],
    [(0, 130), (70, 66), (5, 200)],  # several 64-key tiles, partial tiles, prefix hits
]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("specs", SPECS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_matches_the_reference(shape: tuple[int, int, int], specs: list[tuple[int, int]],
                               dtype: torch.dtype) -> None:  # fmt: skip
    hq, hkv, d = shape
    if d * (4 if dtype == torch.float32 else 2) < 16:
        pytest.skip("rows under 16 bytes are not a kernel shape")
    c = prefill_case(specs, hq, hkv, d, block_size=16 if d >= 64 else 4, dtype=dtype)
    check(c, run(c))


@pytest.mark.parametrize("block_size", [1, 2, 4, 16, 32])
@pytest.mark.parametrize(("rows_per_tile", "block_n"), [(16, 16), (64, 32), (32, 64)])
def test_any_block_size_and_tile_shape(block_size: int, rows_per_tile: int, block_n: int) -> None:
    c = prefill_case([(9, 21), (0, 3), (30, 2)], block_size=block_size, seed=block_size)
    check(c, run(c, rows_per_tile=rows_per_tile, block_n=block_n))


@pytest.mark.parametrize("block_size", [1, 2, 4, 8, 32])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_mfma_kernel_at_any_block_size(block_size: int, dtype: torch.dtype) -> None:
    c = prefill_case([(9, 71), (0, 3), (100, 2), (0, 65)], 16, 8, 128, block_size, dtype,
                     seed=block_size)  # fmt: skip
    check(c, run(c))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_dtypes(dtype: torch.dtype) -> None:
    c = prefill_case(SPECS[2], 16, 8, 128, block_size=16, dtype=dtype)
    out = run(c)
    assert out.dtype == dtype
    check(c, out)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_rows_of_other_sequences_are_left_alone(dtype: torch.dtype) -> None:
    shape = (4, 2, 8) if dtype == torch.float32 else (16, 8, 128)
    c = prefill_case(SPECS[2], *shape, block_size=4, dtype=dtype, gap=2)
    out = torch.full_like(c.q, 7.0).to(DEVICE)
    run(c, out=out)
    check(c, out)
    mine = torch.zeros(c.q.shape[0], dtype=torch.bool)
    for s, n in zip(c.starts.tolist(), c.q_lens.tolist()):
        mine[s : s + n] = True
    assert bool((out.cpu()[~mine] == 7.0).all())


@settings(max_examples=40, deadline=None)
@given(
    specs=st.lists(st.tuples(st.integers(0, 40), st.integers(1, 40)), min_size=1, max_size=4),
    shape=st.sampled_from(SHAPES[:3]),
    block_size=st.sampled_from([1, 2, 4, 8]),
    seed=st.integers(0, 2**16),
)
def test_random_batches(specs: list[tuple[int, int]], shape: tuple[int, int, int], block_size: int,
                        seed: int) -> None:  # fmt: skip
    c = prefill_case(specs, *shape, block_size=block_size, seed=seed)
    check(c, run(c, rows_per_tile=16, block_n=16))


@settings(max_examples=60, deadline=None)
@given(
    specs=st.lists(st.tuples(st.integers(0, 150), st.integers(1, 150)), min_size=1, max_size=4),
    heads=st.sampled_from([(8, 8), (8, 4), (8, 2), (8, 1)]),
    head_dim=st.sampled_from([64, 128]),
    # The gather has three paths by block size: ids staged in LDS (a load's rows span
    # blocks: 1, 2, and 4 at head_dim 64), a scalar id per load, and one scalar id per
    # wave and tile (8 and up at the 32-key shape, 16 and up at the 4-wave 64-key shape).
    block_size=st.sampled_from([1, 2, 4, 8, 16, 32]),
    dtype=st.sampled_from([torch.float16, torch.bfloat16]),
    seed=st.integers(0, 2**16),
)
def test_random_batches_on_mfma(specs: list[tuple[int, int]], heads: tuple[int, int], head_dim: int,
                                block_size: int, dtype: torch.dtype, seed: int) -> None:  # fmt: skip
    c = prefill_case(specs, *heads, head_dim, block_size, dtype, seed=seed)
    check(c, run(c))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32, torch.bfloat16])
def test_qwen3_shapes_with_prefix_hits(dtype: torch.dtype) -> None:
    # test_triton_prefill.py:246-252: 1,024 cached + 64 new tokens, next to a 128-token prompt.
    c = prefill_case([(1024, 64)] * 4 + [(0, 128)], 16, 8, 128, 16, dtype)
    check(c, run(c))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_baseline_config_3(dtype: torch.dtype) -> None:
    # 32 fresh prompts, L ~ U[16, 2048], packed by cu_seqlens; every
    # row within the contract's max-abs bound against the per-sequence oracle (fp16: 2e-3
    # including P's rounding to fp16 before P.V, as triton_prefill.py:118 rounds it).
    lens = prefill_lengths(32, seed=0)
    c = prefill_case([(0, n) for n in lens], 16, 8, 128, 16, dtype, seed=3)
    out = run(c)
    check(c, out)
    assert_contract(out, oracle32(c), dtype, "config 3")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_baseline_config_3_against_the_batched_path(dtype: torch.dtype) -> None:
    # The reference's other prefill path, prefill_plan + batched_prefill_attention
    # (attention.py:144-220): every sequence padded into one rectangle and attended by one
    # masked float32 SDPA call, run here on the GPU on config 3's inputs. Its padding keys
    # read slot 0 under the mask (as the reference's plan pads them), so the pool holds no
    # NaN sentinels here: 0 x NaN would poison the masked sum.
    lens = prefill_lengths(32, seed=0)
    c = prefill_case([(0, n) for n in lens], 16, 8, 128, 16, dtype, seed=3, sentinel=False)
    g = on_gpu(c)
    out = run(c)
    want = ref.batched_prefill_ref(g.q, g.k, g.v, g.tables, g.starts, g.q_lens, g.ctx_lens, g.scale,
                                   g.block_size, out=torch.empty_like(g.q, dtype=torch.float32))  # fmt: skip
    assert_contract(out, want, dtype, "config 3 vs the batched SDPA path")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_both_workgroup_shapes(dtype: torch.dtype) -> None:
    # The library picks the workgroup shape from the grids and the walk, at Qwen3 shapes on 256
    # CUs: one prompt of 2048 tokens makes one round of the key-split shape; 3 and 4 prompts
    # of up to 2048 and 16 of up to 512 make up to 8 8-wave workgroups per CU (4 waves, 32-key
    # tiles, three per CU); 24 prompts of up to 1408 tokens make 2112, over 8 per CU with a mean
    # above 1280 new tokens (8 waves, 64-key tiles, many query tiles per sequence).
    for lens, shape in (([2048], "key_split"), ([2048, 1999, 1100, 700], "short_tiles"),
                        ([2048, 1500, 64], "short_tiles"), ([512] * 15 + [77], "short_tiles"),
                        ([1300 + (37 * i) % 109 for i in range(23)] + [1408], "eight_wave")):  # fmt: skip
        c = prefill_case([(0, n) for n in lens], 16, 8, 128, 16, dtype, seed=len(lens))
        assert shape_of(c) == shape, lens
        check(c, run(c))


@pytest.mark.parametrize("block_size", [1, 2, 4, 8, 16, 32, 64])
@pytest.mark.parametrize("shape", [(16, 8, 128), (8, 2, 64)])
def test_every_gather_path_on_every_workgroup_shape(block_size: int, shape: tuple[int, int, int]) -> None:
    # Each launch below runs one of the three workgroup shapes (one prompt: two key halves, or
    # 4 waves over 64-key tiles below the halves' block size; 16 prompts of 512: 4 waves,
    # 32-key tiles; 4 chunks of 128 new tokens: 8 waves), with prefix hits so that tiles start
    # mid-block, at every block size; the last cuts its keys where the block size allows.
    cut = "cut_eight_wave" if block_size * shape[2] >= 512 else "eight_wave"
    for specs, want in (([(70, 300)], "key_split"), ([(33, 512)] * 15 + [(5, 77)], "short_tiles"),
                        ([(100 + 200 * i, 128) for i in range(4)], "eight_wave"),
                        ([(1000 + 300 * i, 128) for i in range(4)], cut)):  # fmt: skip
        c = prefill_case(specs, *shape, block_size, torch.float16, seed=block_size)
        assert shape_of(c) == want, specs
        check(c, run(c))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("heads", [(16, 8, 128), (32, 8, 128), (8, 2, 64)])
def test_key_split_workgroups(dtype: torch.dtype, heads: tuple[int, int, int]) -> None:
    # One or two prompts run workgroups whose waves split the key tiles in two halves
    # and merge at the end: one key tile (the upper half empty) and a few, under tables of 512
    # keys (under tight ones such prompts run the 32-key shape), odd and even tile
    # counts, a query block whose keys end before the upper half, prefix hits (the
    # halves split the cached keys too; chunks of at most 64 new tokens in small launches
    # run this shape as well, or the cut of longer keys), and block sizes below the scalar-id
    # gather's (the unsplit 4-wave kernel).
    for specs, bs, tokens in (([(0, 1)], 16, 512), ([(0, 64)], 16, 512), ([(0, 60), (130, 1)], 16, 512),
                              ([(0, 200)], 16, 512), ([(0, 1000)], 32, 0), ([(300, 37)], 16, 0),
                              ([(100, 2048)], 16, 0), ([(1024, 64)] * 4, 16, 0), ([(8000, 50)], 16, 0),
                              ([(0, 500), (9, 700)], 64, 0), ([(0, 500)], 2, 0), ([(33, 400)], 1, 0),
                              ([(0, 1)], 16, 0), ([(0, 64)], 16, 0), ([(0, 65)], 16, 0), ([(0, 200)], 16, 0),
                              ([(0, 700), (9, 1300)], 64, 0)):  # fmt: skip
        c = widened(prefill_case(specs, *heads, bs, dtype, seed=bs + len(specs)), tokens)
        if tokens or max(n for _, n in specs) not in (1, 64, 65, 200, 1300):
            assert shape_of(c) == ("cut_key_split" if specs[0][0] == 8000 else "key_split"), specs
        check(c, run(c))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("heads", [(16, 8, 128), (8, 2, 64)])
def test_output_rows_off_16_bytes(dtype: torch.dtype, heads: tuple[int, int, int]) -> None:
    # Output strides that are not whole 16-byte vectors: every shape stores its lanes' pieces of
    # 8 bytes directly, whole and cut items alike.
    for specs, want in (([(0, 70), (9, 3)], "short_tiles"), ([(0, 300)], "key_split"),
                        ([(300, 100), (5, 33)], "eight_wave"), ([(5000, 40), (3, 9)], "cut_key_split"),
                        ([(3000, 100), (0, 7)], "cut_eight_wave")):  # fmt: skip
        c = prefill_case(specs, *heads, 16, dtype, seed=len(want))
        assert shape_of(c) == want, specs
        wide = torch.full((*c.q.shape[:2], heads[2] + 4), 7.0, dtype=dtype, device=DEVICE)
        out = wide[:, :, : heads[2]]
        run(c, out=out)
        check(c, out)
        assert bool((wide[:, :, heads[2] :] == 7.0).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_length_ranked_sequence_groups(dtype: torch.dtype) -> None:
    # Batches of 8-16 prompts, of short ones (up to 64), of 32-64 with equal new-token
    # counts, or of 17-64 mixed ones are dispatched in groups of sequences ranked by
    # context length: 64 short prompts with ties, 12 mixed ones with prefix hits, 9 whose
    # longest is not first, 33 chunks of 600 new tokens after prefixes of different
    # lengths, 21 mixed prompts in pairs (an odd count: the last pair is one), and two
    # batches already in rank order (no ranking loop), one with ties.
    for specs in ([(0, 1 + (53 * i) % 200) for i in range(64)],
                  [((37 * i) % 300, 1 + (211 * i) % 700) for i in range(12)],
                  [(0, 40)] * 4 + [(5, 900)] + [(0, 40)] * 4,
                  [((37 * i) % 500, 600) for i in range(33)],
                  [((29 * i) % 90, 300 + (397 * i) % 1100) for i in range(21)],
                  [(0, 900 - 60 * i) for i in range(12)],
                  [(0, 500)] * 3 + [(0, 300)] * 6):  # fmt: skip
        c = prefill_case(specs, 16, 8, 128, 16, dtype, seed=len(specs), gap=1)
        out = torch.full_like(c.q, 7.0).to(DEVICE)
        run(c, out=out)
        check(c, out)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("heads", [(16, 8, 128), (32, 8, 128), (8, 2, 64), (8, 1, 128)])
def test_long_keys_cut_over_workgroups(dtype: torch.dtype, heads: tuple[int, int, int]) -> None:
    # Chunks behind long cached prefixes: few query tiles, so each one's key tiles are
    # divided over several workgroups whose states are merged. One and 64 new tokens (the
    # key-split shape), 65 and 128 (one 8-wave tile), 300 (several tiles, a partial one);
    # lengths from one key to thousands in one launch (whole and cut items together, an
    # empty sequence, prompts ending on and off a tile); parts whose first tile lies past
    # some rows' positions.
    hq, hkv, d = heads
    cases = [([(3000, 1)], 16), ([(4000, 64), (0, 1), (700, 33)], 16), ([(1985, 65)], 32),
             ([(40, 128), (3100, 100), (0, 128), (1000, 24)], 16)]  # fmt: skip
    if hq // hkv <= 4:  # longer chunks at head groups of 8 keep whole items
        cases.append(([(7000, 300)], 8))
    for specs, bs in cases:
        c = prefill_case(specs, hq, hkv, d, bs, dtype, seed=bs + len(specs), gap=1)
        assert hip_prefill._workspace_floats(0, len(specs), hq, hkv, d, bs, c.max_q_len,
                                             c.tables.shape[1] * bs, dtype) > 0  # fmt: skip
        out = torch.full_like(c.q, 7.0).to(DEVICE)
        run(c, out=out)
        check(c, out)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("heads", [(16, 8, 128), (32, 8, 128), (8, 2, 64), (8, 1, 128)])
def test_short_contexts_under_wide_tables(dtype: torch.dtype, heads: tuple[int, int, int]) -> None:
    # The table's width is the launch's bound on its keys: short contexts under a wide one run
    # the key cut with every item whole, unpriced up to 640 keys and priced from there on (700
    # cached tokens), in the key-split and the 8-wave shape, some sequences shorter than the
    # longest's tiles; 60 sequences fill most of a wave's lanes.
    cases = [[(0, 100)], [(0, 128), (0, 1), (300, 40), (0, 128)], [(0, 40)] * 3, [(0, 250), (3, 17)],
             [(700, 20), (0, 30)]]  # fmt: skip
    if heads[1] == 1:
        cases = [*cases[:3], [(i, 1 + (5 * i) % 32) for i in range(60)]]
    for specs in cases:
        c = widened(prefill_case(specs, *heads, 16, dtype, seed=len(specs), gap=1), 16384)
        assert shape_of(c).startswith("cut"), specs
        out = torch.full_like(c.q, 7.0).to(DEVICE)
        run(c, out=out)
        check(c, out)


@pytest.mark.parametrize("specs", [[(3000, 20)], [(3000, 100), (0, 9)], [(700, 60)], [(0, 500)]])
def test_scores_far_below_zero(specs: list[tuple[int, int]]) -> None:
    # Every score -2^110 (exact, so every weight is equal): key parts and halves that start
    # past the first key must take their own maximum, whatever it is.
    c = prefill_case(specs, 16, 8, 128, 16, torch.bfloat16, seed=len(specs), sentinel=False)
    c = replace(c, q=torch.full_like(c.q, 2.0**50), k=torch.full_like(c.k, -(2.0**53)))
    assert "key_split" in shape_of(c) or "cut" in shape_of(c)
    check(c, run(c))


def test_cut_launch_replays_in_a_graph() -> None:
    c = on_gpu(prefill_case([(2500, 90), (100, 20)], 16, 8, 128, 16, torch.float16, seed=5))
    want = paged_prefill_attention(*c.args())
    out = torch.empty_like(want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        paged_prefill_attention(*c.args(), out=out)
    for _ in range(3):
        out.fill_(9.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
