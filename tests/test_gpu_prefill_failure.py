"""A batched prefill that fails after its first launches returns only when what
it queued has finished: the queued work reads the call's own host tables and
the scratch that the call's locks guard.

The failure is a shape the bf16 GEMM does not take (hidden size 200, not a
multiple of 64), refused on the host after the tables' upload and the clear of
the rows' blocks, which here are gigabytes and take milliseconds.  The call
lasts as long as they do, and nothing is left for the device to finish."""
from __future__ import annotations

import time

import numpy as np
import pytest
import torch

from cruise_amd.runtime import EngineConfig, EngineSpec, ModelSpec, ResidentEpochRuntime, WeightSpec

pytestmark = pytest.mark.gpu

B, BPR = 4, 32


@pytest.mark.parametrize("noalloc", [False, True])
def test_failed_prefill_waits_for_its_queued_work(noalloc):
    model = ModelSpec(num_layers=56, hidden=200, num_heads=8, num_kv_heads=8, head_dim=256, intermediate=256, vocab=512)
    engine = EngineSpec(batch=B, physical_blocks=B * BPR, block_size=128, blocks_per_row=BPR, logical_capacity=BPR * 128,
                        configured_eos=1)
    table = np.arange(B * BPR, dtype=np.int32).reshape(B, BPR)
    with ResidentEpochRuntime(EngineConfig(model=model, engine=engine, weights=WeightSpec("upload"))) as rt:
        assert rt.cache_bytes > 3 << 30
        for _ in range(2):  # the first call also prepares the kernels and the scratch
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            with pytest.raises(RuntimeError, match="failed: -2"):
                rt.prefill_batch(list(range(B)), [1, 2, 3, 4], [[1, 2, 3]] * B, table, noalloc=noalloc)
            t1 = time.perf_counter()
            torch.cuda.synchronize()
            t2 = time.perf_counter()
        call, left = t1 - t0, t2 - t1
        assert call > 5e-4, f"the clear of {2 * rt.cache_bytes >> 20} MiB cannot have finished in {call * 1e6:.0f} us"
        assert left < call / 4, f"{left * 1e6:.0f} us of work left after a call of {call * 1e6:.0f} us"
