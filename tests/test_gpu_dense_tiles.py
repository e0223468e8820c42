"""The dense-bf16 GEMM's three tiles (64 x 64, 64 x 128, 128 x 128) on both sides
of the sizes at which they change, with partial row and column tiles, one to
many K stages and output widths that do not vectorise."""
import numpy as np
import pytest

from glypr_amd import ops
from glypr_amd.ops import BF16Weight
from test_gpu_int8_fma import dev, host, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n", [(1, 64, 1), (65, 128, 63), (300, 1152, 768), (2560, 64, 1024),
                                   (2561, 192, 1025), (3001, 768, 1280), (5100, 128, 2050),
                                   (4097, 320, 130)])
def test_dense_tiles_within_bound(ctx, oracle, m, k, n):
    """|y - y64| <= (k + 2) 2^-24 |x|.|w| against the float64 product of the same
    bf16 operands: k f32 accumulations, in any order."""
    say(f"dense bf16 tiles m={m} k={k} n={n}")
    x = oracle.normal(m * k, seed=700 + m).reshape(m, k)
    wb = ops.f32_to_bf16_bits(oracle.normal(n * k, seed=800 + n, std=0.02).reshape(n, k))
    w = BF16Weight.from_bf16(ctx, wb)
    x64 = (ops.f32_to_bf16_bits(x).astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    w64 = (wb.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    y = host(ops.bf16_matmul(ctx, w, dev(x))).astype(np.float64)
    err = np.abs(y - x64 @ w64.T)
    lim = (k + 2) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T)
    assert np.all(err <= lim), (err / lim).max()
