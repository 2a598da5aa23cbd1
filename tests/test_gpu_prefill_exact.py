"""The batched prefill with split K, exact: weights chosen so that every value
on the way is a small integer in whatever order the sums run, so that the keys
and values come out bit for bit and a K step lost, doubled or added to the wrong
column, range or row shows, which the model tolerance would hide.

Two layers of Qwen2.5-7B's width.  Every embedding is sign * scale * s for one
fixed vector s of +-1, so each RMSNorm returns sign * s exactly; every row has
one prefilled token, so its attention returns its value row exactly, and position
0's rotation is the identity.  First layer, for every output: value = sign (its
weights are random in {-2 .. 2} with the sum over s fixed), o = 2 sign s, gate =
32 and up = 1 (silu(32) = 32; for sign -1 it vanishes next to the residual),
down = 32 s.  Each RMSNorm thus sees a constant magnitude again, unless a sum is
wrong.  Second layer: random integers.  Checked: keys (with a bias) of both
layers, values of both.
"""
from __future__ import annotations

from dataclasses import replace

import numpy as np
import pytest
import torch

from oracle.decoder import PagedGeometry
from oracle.workloads import C2, C2_DIMS
from parity import make_runtime
from test_gpu_prefill import read_caches

pytestmark = pytest.mark.gpu

ROWS, BS, VOCAB = 200, 16, 1024
DIMS = replace(C2_DIMS, num_layers=2, vocab=VOCAB)
BF16 = torch.bfloat16


def integers(n, k, gen):
    return torch.randint(-1, 2, (n, k), generator=gen, device="cuda", dtype=torch.int32)


def with_row_sums(w, s, target, gen):
    """w with +-1 added to some elements of each row so that w @ s == target."""
    n, k = w.shape
    delta = target - (w * s).sum(1)
    assert int(delta.abs().max()) <= k
    start = torch.randint(0, k, (n, 1), generator=gen, device="cuda")
    place = (torch.arange(k, device="cuda") - start) % k
    return w + (place < delta.abs()[:, None]) * delta.sign()[:, None] * s


@pytest.fixture(scope="module")
def model():
    gen = torch.Generator(device="cuda").manual_seed(77)
    H, I = DIMS.hidden, DIMS.intermediate
    q, kv = DIMS.num_heads * DIMS.head_dim, DIMS.num_kv_heads * DIMS.head_dim
    s = torch.randint(0, 2, (H,), generator=gen, device="cuda", dtype=torch.int32) * 2 - 1
    ones = lambda n: torch.ones(n, device="cuda", dtype=torch.int32)
    token = torch.arange(VOCAB, device="cuda")
    sign, scale = 1 - 2 * (token % 2), 2 ** (token // 2 % 3)
    w = {"embedding": (sign * scale)[:, None] * s}
    for i in range(2):
        p = f"layers_{i}_"
        w[p + "input_norm"], w[p + "post_norm"] = ones(H), ones(H)
        w[p + "q_weight"], w[p + "q_bias"] = integers(q, H, gen), 0 * ones(q)
        w[p + "k_weight"], w[p + "k_bias"] = integers(kv, H, gen), integers(1, kv, gen)[0] * 5
        v = integers(kv, H, gen)
        w[p + "v_weight"] = with_row_sums(v, s, ones(kv), gen) if i == 0 else v
        w[p + "v_bias"] = 0 * ones(kv) if i == 0 else integers(1, kv, gen)[0] * 3
        w[p + "o_weight"] = with_row_sums(integers(H, q, gen), ones(q), 2 * s, gen)
        w[p + "gate_weight"] = with_row_sums(integers(I, H, gen), s, 32 * ones(I), gen)
        w[p + "up_weight"] = with_row_sums(integers(I, H, gen), s, ones(I), gen)
        w[p + "down_weight"] = with_row_sums(integers(H, I, gen), ones(I), s, gen)
    w["final_norm"], w["lm_head"] = ones(H), integers(VOCAB, H, gen)
    W = replace(C2, name="exact-2layer", dims=DIMS,
                geometry=PagedGeometry(batch=ROWS, physical_blocks=ROWS, block_size=BS, blocks_per_row=1, window=BS))
    weights = {n: t.to(BF16) for n, t in w.items()}
    rt = make_runtime(W, weights)
    want = {}  # (sign, layer) -> key row, value row
    for sg in (1, -1):
        for i in range(2):
            p = f"layers_{i}_"
            dot = lambda n: (sg * (w[p + n + "_weight"] * s).sum(1) + w[p + n + "_bias"]).to(BF16).cpu()
            want[sg, i] = dot("k"), dot("v")
    del w
    torch.cuda.empty_cache()
    yield rt, want, weights
    rt.close()


def mismatches(rt, want, M, noalloc=False):
    """Elements of the keys and values of each layer that are not the exact ones."""
    rng = np.random.default_rng(M)
    rows, tokens = rng.permutation(ROWS)[:M], rng.integers(0, VOCAB, size=M)
    rt.prefill_batch([int(r) for r in rows], list(range(1, M + 1)), [[int(t), 0] for t in tokens],
                     rows.astype(np.int32)[:, None], noalloc=noalloc)
    caches, out = [c.view(2, ROWS, BS, -1) for c in read_caches(rt, BF16)], {}
    for i in range(2):
        for c, what in enumerate(("keys", "values")):
            ref = torch.stack([want[1 - 2 * int(t % 2), i][c] for t in tokens])
            out[i, what] = int((caches[c][i][rows, 0] != ref).sum())
    return out


@pytest.mark.parametrize("M", [1, 4, 16, 63, 64, 65, 128, 129, 200])
@pytest.mark.parametrize("noalloc", [False, True])
def test_split_prefill_exact(model, M, noalloc):
    rt, want, _ = model
    found = mismatches(rt, want, M, noalloc)
    assert not any(found.values()), found


@pytest.mark.parametrize("name,layer", [("k_weight", 0), ("v_weight", 0), ("o_weight", 1), ("down_weight", 1), ("v_weight", 1)])
def test_a_missing_k_step_shows(model, name, layer):
    """The expectation is sharp: without one 64-element step of one matrix (taken
    out of the weights) the results differ in the layer that it reaches."""
    rt, want, weights = model
    key = f"layers_{0 if name[0] in 'od' else layer}_{name}"  # o and down reach the next layer
    full = weights[key]
    steps = full.shape[1] // 64
    try:
        for step in (0, 1, steps // 2, steps - 1):
            short = full.clone()
            short[:, 64 * step:64 * (step + 1)] = 0
            rt.write_state(key, short)
            found = mismatches(rt, want, 16)
            assert found[layer, "keys" if name == "k_weight" else "values"] > 0, (step, found)
    finally:
        rt.write_state(key, full)
