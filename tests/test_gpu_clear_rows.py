"""Row and block clears in chunks of 1,024 16-byte words: a batch past one
64-row flag word, blocks of less than one chunk and of one and a bit, some rows
of a new generation and some resumed.  Every block of a cleared row must be
zero but for the step's own slot, and every other block keep its bytes."""
from __future__ import annotations

from dataclasses import replace

import numpy as np
import pytest
import torch

from cruise_amd.runtime import pack_feed, tiling_bytes
from oracle.controller import control_input_elements
from oracle.decoder import PagedGeometry
from oracle.weights import generate_weights
from oracle.workloads import C1, C1_DIMS
from parity import make_runtime

pytestmark = pytest.mark.gpu


# fp32 (2 heads of 64): 512 bytes a position; 33 positions are 1,056 words, one chunk and 32
@pytest.mark.parametrize("batch,dtype,block", [(4, "fp32", 16), (4, "fp32", 33), (130, "bf16", 8)])
def test_only_new_rows_are_cleared(batch, dtype, block):
    dims = replace(C1_DIMS, dtype=dtype)
    g = PagedGeometry(batch=batch, physical_blocks=2 * batch + 3, block_size=block, blocks_per_row=2, window=2 * block)
    W = replace(C1, dims=dims, geometry=g)
    rt = make_runtime(W, generate_weights(dims, W.seed))
    try:
        rng = np.random.default_rng(5700)
        table = rng.permutation(g.physical_blocks)[: 2 * batch].reshape(batch, 2).astype(np.int32)
        new = np.arange(batch) % 3 == 1
        pos = np.where(new, 0, 3).astype(np.int64)
        tok = rng.integers(0, dims.vocab, size=batch).astype(np.int64)
        gens = np.arange(1, batch + 1)
        T = dims.torch_dtype
        shape = (dims.num_layers, g.physical_blocks, block, dims.num_kv_heads, dims.head_dim)
        caches = [torch.randn(shape, generator=torch.Generator().manual_seed(5701 + i)).to(T) for i in range(2)]
        for name, c in zip(("key_cache", "value_cache"), caches):
            rt.write_state(name, c.cuda())
        rt.write_state("resident_rows", np.stack([np.where(new, 0, gens), tok, pos, pos + 1, np.ones(batch)]).astype(np.int64))
        control = np.zeros(control_input_elements(batch), dtype=np.int32)
        control[0], control[1 : 1 + batch], control[3 + batch :] = 1, W.eos, gens
        slot = table[np.arange(batch), pos // block] * block + pos % block
        _, ctrl = rt.proc(pack_feed(tok, pos, (pos + 1).astype(np.int32), slot.astype(np.int32),
                                    np.ones(batch, dtype=np.int32), table, tiling_bytes(), control))
        assert ctrl[3] == 0
        for name, c in zip(("key_cache", "value_cache"), caches):
            want, got = c.clone(), torch.zeros_like(c)
            rt.read_state(name, got)
            want[:, table[new].reshape(-1)] = 0
            flat = lambda t: t.view(dims.num_layers, -1, dims.num_kv_heads, dims.head_dim)
            keep = torch.ones(flat(want).shape[1], dtype=torch.bool)
            keep[torch.from_numpy(slot.astype(np.int64))] = False
            assert torch.equal(flat(got)[:, keep], flat(want)[:, keep]), name
            assert (flat(got)[:, ~keep] != 0).any(-1).all(), f"{name}: a step's slot was not written"
    finally:
        rt.close()
