"""Where the decoder step's buffers may live (resident_decoder_step): caches in
device memory are used in place, others (host memory, device memory that is not
16-byte aligned) go through the engine's own pair, and inputs in host memory
share one upload.  The same kernels run on the same values, so logits, caches
and next positions must be equal bit for bit however the buffers are given."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle.weights import generate_weights
from oracle.workloads import C1, random_tables, slot_of
from parity import make_runtime

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    rt = make_runtime(C1, generate_weights(C1.dims, C1.seed))
    yield rt
    rt.close()


def case():
    rng = np.random.default_rng(5501)
    g, d = C1.geometry, C1.dims
    B = g.batch
    table = random_tables(rng, B, g.blocks_per_row, g.physical_blocks)
    pos = np.array([0, 5, 17, 31], dtype=np.int64)
    active = np.array([1, 1, 0, 1], dtype=np.int32)
    slot = np.array([slot_of(table, r, int(pos[r]), g.block_size) for r in range(B)], dtype=np.int32)
    gen = torch.Generator().manual_seed(5502)
    shape = (d.num_layers, g.physical_blocks, g.block_size, d.num_kv_heads, d.head_dim)
    caches = [torch.randn(shape, generator=gen) for _ in range(2)]
    inputs = [rng.integers(0, d.vocab, size=B), pos, (pos + 1).astype(np.int32), slot, active, table.astype(np.int32)]
    return inputs, caches, np.where(active != 0, pos + 1, pos)


def step(rt, inputs, caches, out_device):
    tok, pos, length, slot, active, table = inputs
    logits = torch.zeros(C1.geometry.batch, C1.dims.vocab, device=out_device)
    nxt = torch.zeros(C1.geometry.batch, dtype=torch.int64, device=out_device)
    torch.cuda.synchronize()
    rt.decoder_step(tok, pos, length, caches[0], slot, active, table, caches[1], logits, nxt)
    return [t.cpu() for t in (logits, *caches, nxt)]


def device_copy(t, shift):
    """t on the GPU, starting shift elements past an aligned address."""
    return torch.cat([torch.zeros(shift), t.flatten()]).cuda()[shift:].view(t.shape)


@pytest.mark.parametrize("where", ["host", "unaligned", "one allocation", "device inputs", "mixed inputs"])
def test_buffers_give_equal_bits(rt, where):
    inputs, caches, want_next = case()
    ref = step(rt, inputs, [c.cuda() for c in caches], "cuda")
    np.testing.assert_array_equal(ref[3].numpy(), want_next)
    assert not torch.equal(ref[1], caches[0]) and not torch.equal(ref[2], caches[1])  # written in place
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in inputs]
    if where == "host":
        got = step(rt, inputs, [c.clone() for c in caches], "cpu")
    elif where == "unaligned":
        got = step(rt, inputs, [device_copy(caches[0], 1), device_copy(caches[1], 3)], "cuda")
    elif where == "one allocation":
        both = torch.stack(caches).cuda()
        got = step(rt, inputs, [both[1].copy_(caches[0]), both[0].copy_(caches[1])], "cuda")
    elif where == "device inputs":
        got = step(rt, dev, [c.cuda() for c in caches], "cuda")
    else:
        got = step(rt, [inputs[0], dev[1], inputs[2], dev[3], inputs[4], dev[5]], [caches[0].cuda(), caches[1].clone()], "cpu")
    for a, b in zip(got, ref):
        assert torch.equal(a, b)
