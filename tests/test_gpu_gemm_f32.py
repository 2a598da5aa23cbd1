"""The fp32 prefill GEMM on the GPU: fp32 MFMA on 16 x 16 and 32 x 32 tiles, K
split over four waves, and 64 x 64 tiles through LDS for large products.

* Edges of the tiles, of the 16-element K chunks and of the four waves' turns,
  every tile size (32 x 32 from 512 tiles on; 64 x 64 from 768 on, unaligned
  from 257 on), aligned and unaligned rows, against the product in 64 bits.  Each output is K products and K + 2 sums in
  fp32 (the bias or residual one of them), so it is within
  (K + 3) 2^-24 (sum |a| |w| + |bias or residual|) of it in any order.
* More tiles than a grid dimension holds.
* The SwiGLU epilogue at both tile sizes: prompts of a small fp32 model
  prefilled together (2,036 tokens: 32 x 32 tiles; 20 tokens: 16 x 16) against
  the engine's own single-row prefill at the model tolerance.
"""
from __future__ import annotations

from dataclasses import replace

import numpy as np
import pytest
import torch

from oracle.decoder import PagedGeometry
from oracle.weights import generate_weights
from oracle.workloads import C1, random_tables
from parity import make_runtime
from test_gpu_gemm import lib, operands, ptr, run  # noqa: F401
from test_gpu_prefill import check_caches, read_caches, reset, written_slots

pytestmark = pytest.mark.gpu

SMALL = [(1, 1, 1), (15, 17, 3), (16, 16, 64), (17, 33, 68), (66, 256, 688), (31, 48, 272), (5, 7, 1000)]
LARGE = [(512, 1024, 16), (496, 1024, 40), (1030, 1041, 33), (2032, 688, 256), (1024, 1024, 20), (1025, 1024, 7),
         (2048, 1472, 36), (2048, 1536, 36), (2048, 2048, 36), (1985, 2047, 12), (1984, 2112, 64)]


@pytest.mark.parametrize("M,N,K", SMALL + LARGE)
@pytest.mark.parametrize("epilogue", [0, 1])
@pytest.mark.parametrize("shift", [0, 1])
def test_fp32_gemm_against_64_bits(lib, M, N, K, epilogue, shift):  # noqa: F811
    A, W, _, bias, out0 = operands(M, N, K, torch.float32, False, M + N + K + epilogue)
    # shift 1: operands one element past 16-byte alignment
    at = lambda t: torch.cat([torch.zeros(shift), t.flatten()]).cuda()[shift:].view(t.shape)
    out, add = at(out0), bias if epilogue == 0 else out0
    assert run(lib, at(A), at(W), None, at(bias), out, epilogue) == 0
    ref = A.double() @ W.double().T + add.double()
    bound = (K + 3) * 2.0 ** -24 * (A.double().abs() @ W.double().abs().T + add.double().abs())
    bad = (out.cpu().double() - ref).abs() > bound
    assert not bad.any(), f"{bad.sum().item()} of {bad.numel()} outputs past the bound"


@pytest.mark.parametrize("length", [510, 6])
def test_fp32_swiglu_prefill_matches_single_row_prefill(length):
    W = replace(C1, geometry=PagedGeometry(batch=4, physical_blocks=128, block_size=16, blocks_per_row=32, window=512))
    rng = np.random.default_rng(5400 + length)
    table = random_tables(rng, 4, 32, 128)
    prompts = [list(map(int, rng.integers(0, W.dims.vocab, size=length))) for _ in range(4)]
    rt = make_runtime(W, generate_weights(W.dims, W.seed))
    try:
        reset(rt, torch.float32, 4)
        for r in range(4):
            rt.prefill(r, 1 + r, prompts[r], table[r])
        k_ref, v_ref = read_caches(rt, torch.float32)
        reset(rt, torch.float32, 4)
        rt.prefill_batch(list(range(4)), [1 + r for r in range(4)], prompts, table)
        k, v = read_caches(rt, torch.float32)
        slots = written_slots(table, prompts, 16)
        check_caches(W, k, k_ref, slots, "keys")
        check_caches(W, v, v_ref, slots, "values")
    finally:
        rt.close()


@pytest.mark.parametrize("M,N", [(131_080, 131_080), (4_194_330, 70), (70, 4_194_330)])
def test_fp32_gemm_of_many_tiles(lib, M, N):  # noqa: F811
    """69 GB of output: 2^24 tiles of 32 x 32, at 256 threads each more than one
    grid dimension holds; and more tiles along M or N than a grid's second
    dimension holds.  Integer operands: the sums are exact."""
    gen = torch.Generator(device="cuda").manual_seed(11)
    mk = lambda *s: torch.randint(-8, 9, s, generator=gen, device="cuda").float()
    A, W = mk(M, 4), mk(N, 4)
    out = torch.empty(M, N, device="cuda")
    out[-64:] = -1.0
    torch.cuda.synchronize()
    assert run(lib, A, W, None, None, out, 0) == 0
    for r0 in (0, 64, 4096, 65504, 131_008, 4_194_250, M - 40):
        if r0 < M:
            assert torch.equal(out[r0:r0 + 40], A[r0:r0 + 40] @ W.T), f"rows from {r0}"
    del out
    torch.cuda.empty_cache()


def test_fp32_swiglu_is_refused_and_no_rows_are_not(lib):  # noqa: F811
    A, W = torch.zeros(1, 8, device="cuda"), torch.zeros(8, 8, device="cuda")
    out = torch.full((1, 8), 7.0, device="cuda")
    assert run(lib, A, W, W, None, out, 2) == -1
    assert lib.resident_epoch_gemm(ptr(A), ptr(W), ptr(W), None, ptr(out), 0, 8, 8, 2, 4) == 0
    assert bool((out == 7.0).all())
