"""The batched prefill's GEMM plans (tile height, K ranges) on the GPU.

* products whose planned tiles are 128, 192 and 256 rows high, at heights that
  leave a partial last tile, against the CPU product: integer operands, so fp32
  sums are exact in any order and the store and residual epilogues must agree
  bit for bit (as in test_gpu_gemm.py, whose shapes take the 64-row tile;
  test_gpu_gemm_tiled.py checks every height whatever the planner chooses);
* split K: two Qwen2.5-7B layers (the second layer's keys and values go
  through the first one's qkv, o and down partial sums) at token counts
  around the tile edges, against the engine's own single-row prefill at the
  model tolerance (test_gpu_prefill_exact.py: exactly);
* the no-allocation entry point chooses the same K ranges: equal bits.
"""
from __future__ import annotations

from dataclasses import replace

import numpy as np
import pytest
import torch

from oracle.weights import generate_weights
from oracle.workloads import C2, C2_DIMS, random_tables
from parity import engine_snapshot, make_runtime
from test_gpu_gemm import BF16, lib, one, operands, within_two_steps  # noqa: F401
from test_gpu_prefill import check_caches, read_caches, reset, written_slots

pytestmark = pytest.mark.gpu


# 75 column tiles: 250, 520 and 750 rows take the 128-, 192- and 256-row tile
@pytest.mark.parametrize("M", [250, 520, 750])
@pytest.mark.parametrize("epilogue", [0, 1, 2])
def test_tile_heights_integer_operands(lib, M, epilogue):  # noqa: F811
    N, K = (9480 if epilogue == 2 else 18952), 128
    got, ref = one(lib, M, N, K, BF16, epilogue, True, seed=M + epilogue)
    if epilogue < 2:
        assert torch.equal(got, ref), f"{(got != ref).sum().item()} of {ref.numel()} outputs differ"
    else:
        A, W, W2, _, _ = operands(M, N, K, BF16, True, M + epilogue)
        within_two_steps(got, ref, A, W, W2)


@pytest.fixture(scope="module")
def two_layers():
    W = replace(C2, name="qwen7b-2layer", dims=replace(C2_DIMS, num_layers=2), seed=C2.seed + 2)
    rt = make_runtime(W, generate_weights(W.dims, W.seed, device="cuda"))
    yield W, rt
    rt.close()


def inputs(W, lengths, seed):
    rng = np.random.default_rng(seed)
    table = random_tables(rng, W.geometry.batch, W.geometry.blocks_per_row, W.geometry.physical_blocks)
    return table, [list(map(int, rng.integers(0, W.dims.vocab, size=n))) for n in lengths]


# tokens: 1, 16, 64, 65, 129, 193, 577 (a row's last token is not prefilled)
@pytest.mark.parametrize("lengths", [[2, 1, 1, 1], [17, 1, 1, 1], [30, 34, 1, 3], [60, 3, 4, 2], [128, 2, 2, 1],
                                     [190, 2, 4, 1], [250, 250, 79, 2]])
def test_split_prefill_matches_single_row_prefill(two_layers, lengths):
    W, rt = two_layers
    B = W.geometry.batch
    table, prompts = inputs(W, lengths, 5200 + sum(lengths))
    reset(rt, torch.bfloat16, B)
    for r in range(B):
        rt.prefill(r, 20 + r, prompts[r], table[r])
    k_ref, v_ref = read_caches(rt, torch.bfloat16)
    rows_ref = rt.resident_rows().copy()
    reset(rt, torch.bfloat16, B)
    rt.prefill_batch(list(range(B)), [20 + r for r in range(B)], prompts, table)
    k, v = read_caches(rt, torch.bfloat16)
    slots = written_slots(table, prompts, W.geometry.block_size)
    check_caches(W, k, k_ref, slots, "keys")
    check_caches(W, v, v_ref, slots, "values")
    np.testing.assert_array_equal(rt.resident_rows(), rows_ref)


def test_noalloc_takes_the_same_ranges(two_layers):
    W, rt = two_layers
    B = W.geometry.batch
    table, prompts = inputs(W, [250, 250, 250, 79], 5301)
    snaps = []
    for noalloc in (False, True):
        reset(rt, torch.bfloat16, B)
        rt.prefill_batch(list(range(B)), [1, 2, 3, 4], prompts, table, noalloc=noalloc)
        snaps.append(engine_snapshot(rt, torch.bfloat16))
    for a, b in zip(snaps[0][:2], snaps[1][:2]):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
