"""The matrix-core decode projections (re_mfma.hip) at 5 to 63 rows: one
16-row batch tile to four, whole and partial, against the row-tiled kernels
("tuning": {"mfma": 0}), which the oracle tests pin.  Two Qwen2.5-7B layers, so
the down projection's partial sums reach the next layer's norm; some rows
inactive; one decoder step: logits and the written keys and values at the
model tolerance (the fp32 sums run in another order), every other slot
untouched.  Windows cover each attention that writes the packed layout: one
workgroup per (row, head), its window split, and the grouped kernels.

An engine without the room for the packed weights is planned and allocated
again for the row-tiled kernels: the bits of "mfma": 0.
"""
from __future__ import annotations

from dataclasses import replace

import numpy as np
import pytest
import torch

from oracle.decoder import PagedGeometry
from oracle.weights import generate_weights, seeded_cache
from oracle.workloads import C2, C2_DIMS, random_tables, slot_of
from parity import assert_close_rel, make_runtime, rel_tol

pytestmark = pytest.mark.gpu

DIMS = replace(C2_DIMS, num_layers=2)
BS = 128


@pytest.fixture(scope="module")
def weights():
    return generate_weights(DIMS, C2.seed + 5, device="cuda")


def step(W, weights, args, caches, tuning, mfma=None):
    B = W.geometry.batch
    rt = make_runtime(W, weights, tuning=tuning)
    try:
        assert bool(rt.info("mfma")) == (tuning is None if mfma is None else mfma)
        k, v = caches[0].clone().cuda(), caches[1].clone().cuda()
        logits = torch.zeros(B, DIMS.vocab, dtype=torch.float32, device="cuda")
        nxt = torch.zeros(B, dtype=torch.int64, device="cuda")
        tok, pos, length, slot, active, table = args
        rt.decoder_step(tok, pos, length, k, slot, active, table, v, logits, nxt)
        torch.cuda.synchronize()
        return logits.cpu(), k.cpu(), v.cpu(), nxt.cpu()
    finally:
        rt.close()


def inputs(B, window):
    """A workload of B rows, its step arguments and its caches; some rows inactive."""
    bpr = window // BS
    geo = PagedGeometry(batch=B, physical_blocks=B * bpr, block_size=BS, blocks_per_row=bpr, window=window)
    W = replace(C2, name=f"qwen7b-2layer-b{B}", dims=DIMS, geometry=geo)
    rng = np.random.default_rng(6500 + B)
    table = random_tables(rng, B, bpr, B * bpr)
    pos = rng.integers(0, window - 1, size=B).astype(np.int64)
    pos[0], pos[-1] = window - 1, 0
    active = np.ones(B, dtype=np.int32)
    active[1::4] = 0
    slot = np.array([slot_of(table, r, int(pos[r]), BS) for r in range(B)], dtype=np.int32)
    args = (rng.integers(0, DIMS.vocab, size=(B, 1)).astype(np.int64), pos, (pos + 1).astype(np.int32).reshape(B, 1), slot,
            active, table)
    shape = (DIMS.num_layers, B * bpr, BS, DIMS.num_kv_heads, DIMS.head_dim)
    return W, args, seeded_cache(shape, 6600 + B, torch.bfloat16)


@pytest.mark.parametrize("B,window", [(5, 256), (8, 1280), (15, 128), (16, 512), (17, 256), (32, 256), (33, 256),
                                      (48, 256), (49, 256), (63, 256)])
def test_rows_match_row_tiled_kernels(weights, B, window):
    W, args, caches = inputs(B, window)
    slot, active, slots = args[3], args[4], W.geometry.physical_blocks * BS
    got, ref = step(W, weights, args, caches, None), step(W, weights, args, caches, {"mfma": 0})
    assert torch.equal(got[3], ref[3])
    assert_close_rel(got[0], ref[0], rel_tol(DIMS), "logits")
    flat = lambda t: t.reshape(DIMS.num_layers, -1, DIMS.num_kv_heads, DIMS.head_dim)
    written = [int(slot[r]) for r in range(B) if active[r]]
    mask = torch.ones(slots, dtype=torch.bool)
    mask[written] = False
    for i, what in ((1, "keys"), (2, "values")):
        assert torch.equal(flat(got[i])[:, mask], flat(caches[i - 1])[:, mask]), f"unaddressed {what} changed"
        assert_close_rel(flat(got[i])[:, written], flat(ref[i])[:, written], rel_tol(DIMS), f"written {what}")


@pytest.mark.parametrize("B,window", [(5, 256), (41, 1024)])
def test_engine_without_room_for_packed_weights(weights, B, window):
    W, args, caches = inputs(B, window)
    packed = 2 * sum(int(t.numel()) for n, t in weights.items() if n == "lm_head" or n.endswith("_weight"))
    got = step(W, weights, args, caches, {"packed_limit": packed - 1}, mfma=False)
    ref = step(W, weights, args, caches, {"mfma": 0})
    for a, b in zip(got, ref):
        assert torch.equal(a, b)
    step(W, weights, args, caches, {"packed_limit": packed}, mfma=True)
