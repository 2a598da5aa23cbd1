"""The SwiGLU GEMM's 96-column tiles (up to 192 rows; 256 tiles at most) on
the GPU, against the CPU product with the kernel's rounding points: 64-, 128- and
192-row tiles at their edges, partial last column tiles, the last
size with 96-column tiles and the first without.  Integer operands, so the
fp32 products are exact; within two bf16 steps for the device's exp."""
from __future__ import annotations

import pytest

from test_gpu_gemm import BF16, lib, one, operands, within_two_steps  # noqa: F401


pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 16, 63, 64, 65, 127, 128, 129, 192, 193])
@pytest.mark.parametrize("N,K", [(8, 64), (96, 128), (104, 192), (18944, 256), (24576, 64), (24584, 64)])
def test_narrow_swiglu_tiles(lib, M, N, K):  # noqa: F811
    seed = M + N + K
    got, ref = one(lib, M, N, K, BF16, 2, True, seed=seed)
    A, W, W2, _, _ = operands(M, N, K, BF16, True, seed)
    within_two_steps(got, ref, A, W, W2)
