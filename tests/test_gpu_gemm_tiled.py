"""The prefill GEMM on given tiles (resident_epoch_gemm_tiled), so that every
tile height and every split of K is checked whatever the planner chooses.

* bf16, integer operands (|a|, |w| <= 2, so fp32 sums are exact in any order):
  the three epilogues at every tile height, and the fp32 partial sums of each K
  range against the product over that range's columns, bit for bit: ranges of
  one step, of fewer and of more steps than a tile keeps in flight, uneven
  ones, one range and as many as steps, partial tiles in M and N.
* fp32 SwiGLU at every tile size, against 64 bits.
"""
from __future__ import annotations

import pytest
import torch

from test_gpu_gemm import BF16, lib, operands, ptr, reference, within_two_steps  # noqa: F401

pytestmark = pytest.mark.gpu

HEIGHTS = [64, 128, 192, 256]
SHAPES = [(1, 8), (64, 256), (65, 264), (200, 520), (257, 248)]


def tiled(lib, A, W, W2, bias, out, epilogue, tile_rows, ranges):  # noqa: F811
    (M, K), N = A.shape, W.shape[0]
    return lib.resident_epoch_gemm_tiled(ptr(A), ptr(W), ptr(W2), ptr(bias), ptr(out), M, N, K, epilogue,
                                         A.element_size(), tile_rows, ranges)


@pytest.mark.parametrize("rows", HEIGHTS)
@pytest.mark.parametrize("epilogue", [0, 1, 2])
def test_epilogues_at_every_tile_height(lib, rows, epilogue):  # noqa: F811
    for M, N in SHAPES:
        for K in (64, 128, 192, 320):
            A, W, W2, bias, out0 = operands(M, N, K, BF16, True, M + N + K)
            out = out0.cuda()
            assert tiled(lib, A.cuda(), W.cuda(), W2.cuda(), bias.cuda(), out, epilogue, rows, 1) == 0
            ref = reference(A, W, W2, bias, out0, epilogue)
            if epilogue < 2:
                assert torch.equal(out.cpu(), ref), (M, N, K)
            else:
                within_two_steps(out.cpu(), ref, A, W, W2)


# one step a range; 1 and 2; 1 to 3; 3 and 4; 5, 8 and 9; the down projection's 296 in 18
@pytest.mark.parametrize("rows", HEIGHTS)
@pytest.mark.parametrize("steps,ranges", [(1, 1), (5, 5), (5, 3), (7, 3), (5, 1), (11, 3), (10, 2), (16, 2), (18, 2), (296, 18)])
def test_partial_sums_of_every_range(lib, rows, steps, ranges):  # noqa: F811
    for M, N in SHAPES:
        K = 64 * steps
        A, W, _, _, _ = operands(M, N, K, BF16, True, 3 * M + N + K)
        out = torch.full((ranges + 1, M, N), float("nan"), device="cuda")
        assert tiled(lib, A.cuda(), W.cuda(), None, None, out, 3, rows, ranges) == 0
        got = out.cpu()
        for r in range(ranges):
            k = slice(64 * (r * steps // ranges), 64 * ((r + 1) * steps // ranges))
            assert torch.equal(got[r], A[:, k].float() @ W[:, k].float().T), (M, N, r)
        assert bool(got[ranges].isnan().all()), "written past the last range"


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (17, 33, 68), (66, 688, 256), (31, 47, 100), (1030, 1041, 33), (2032, 688, 256), (2048, 2048, 36), (1985, 2047, 12)])
def test_fp32_swiglu_against_64_bits(lib, M, N, K):  # noqa: F811
    """Gate and up are within e = (K + 2) 2^-24 sum |a| |w| of the product each (K
    products, K + 1 sums); |silu'| < 1.1; and silu * up, an exponential, a sum, a
    quotient and a product, rounds by at most 8 x 2^-24 of its value."""
    A, W, W2, _, _ = operands(M, N, K, torch.float32, False, M + N + K)
    out = torch.zeros(M, N, device="cuda")
    assert tiled(lib, A.cuda(), W.cuda(), W2.cuda(), None, out, 2, 0, 1) == 0
    g, u = A.double() @ W.double().T, A.double() @ W2.double().T
    e_g, e_u = ((K + 2) * 2.0 ** -24 * (A.double().abs() @ w.double().abs().T) for w in (W, W2))
    ref = torch.nn.functional.silu(g) * u
    bound = 1.1 * e_g * (u.abs() + e_u) + torch.nn.functional.silu(g).abs() * e_u + 8 * 2.0 ** -24 * (ref.abs() + 1.1 * e_g * u.abs())
    bad = (out.cpu().double() - ref).abs() > bound
    assert not bad.any(), f"{bad.sum().item()} of {bad.numel()} outputs past the bound"


def test_tiles_that_do_not_exist_are_refused(lib):  # noqa: F811
    A, W = torch.zeros(8, 128, dtype=BF16, device="cuda"), torch.zeros(8, 128, dtype=BF16, device="cuda")
    out = torch.zeros(2, 8, 8, device="cuda")
    assert tiled(lib, A, W, None, None, out, 3, 64, 3) == -1  # more ranges than steps
    assert tiled(lib, A[:, :96].contiguous(), W[:, :96].contiguous(), None, None, out, 3, 64, 1) == -1  # K % 64
