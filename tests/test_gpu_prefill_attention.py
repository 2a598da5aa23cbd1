"""The batched prefill's attention at the edges of its kernels: pass 1 keeps its
scores for prompts of up to 1, 4 and 16 key tiles of 64 (the pass's longest
prompt decides), longer ones compute them twice.  Two Qwen2.5-7B layers (the
second layer's keys and values come from the first one's attention), with
longest prompts around each edge and shorter rows beside them, against the
engine's own single-row prefill at the model tolerance;
and in either order of the rows (other tiles beside each other), bit for bit."""
from __future__ import annotations

from dataclasses import replace

import numpy as np
import pytest
import torch

from oracle.decoder import PagedGeometry
from oracle.weights import generate_weights
from oracle.workloads import C2, C2_DIMS, random_tables
from parity import make_runtime
from test_gpu_prefill import check_caches, read_caches, reset, written_slots

pytestmark = pytest.mark.gpu

GEOMETRY = PagedGeometry(batch=2, physical_blocks=24, block_size=128, blocks_per_row=9, window=1152)
SHORT = 41


@pytest.fixture(scope="module")
def two_layers():
    W = replace(C2, name="qwen7b-2layer-w1152", dims=replace(C2_DIMS, num_layers=2), geometry=GEOMETRY, seed=C2.seed + 3)
    rt = make_runtime(W, generate_weights(W.dims, W.seed, device="cuda"))
    yield W, rt
    rt.close()


def inputs(W, longest):
    rng = np.random.default_rng(5600)
    table = random_tables(rng, 2, W.geometry.blocks_per_row, W.geometry.physical_blocks)
    short = list(map(int, rng.integers(0, W.dims.vocab, size=SHORT)))
    return table, [short, list(map(int, np.random.default_rng(longest).integers(0, W.dims.vocab, size=longest + 1)))]


# prefilled tokens of the longer row (its last token is not prefilled)
@pytest.mark.parametrize("longest", [1, 63, 64, 65, 128, 256, 257, 1023, 1024, 1025])
def test_prefill_matches_single_row_prefill(two_layers, longest):
    W, rt = two_layers
    table, prompts = inputs(W, longest)
    reset(rt, torch.bfloat16, 2)
    for r in range(2):
        rt.prefill(r, 30 + r, prompts[r], table[r])
    k_ref, v_ref = read_caches(rt, torch.bfloat16)
    reset(rt, torch.bfloat16, 2)
    rt.prefill_batch([0, 1], [30, 31], prompts, table)
    k, v = read_caches(rt, torch.bfloat16)
    slots = written_slots(table, prompts, W.geometry.block_size)
    check_caches(W, k, k_ref, slots, "keys")
    check_caches(W, v, v_ref, slots, "values")


def test_order_of_rows_changes_nothing(two_layers):
    W, rt = two_layers
    table, _ = inputs(W, 1)
    d = W.dims
    for longest in (40, 200, 900, 1100):
        _, (short, long) = inputs(W, longest)
        seen = []
        for order in ((0, 1), (1, 0)):
            reset(rt, torch.bfloat16, 2)
            rows = [(0, short, table[0]), (1, long, table[1])]
            pick = [rows[i] for i in order]
            rt.prefill_batch([p[0] for p in pick], [9, 9], [p[1] for p in pick], np.stack([p[2] for p in pick]))
            seen.append([c.view(torch.int16).reshape(d.num_layers, -1) for c in read_caches(rt, torch.bfloat16)])
        for a, b in zip(*seen):
            assert torch.equal(a, b), f"longest {longest}: the rows' order changed their keys or values"
