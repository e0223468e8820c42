"""The plain int8 GEMM's three large-M tiles (128 x 128, 64 x 64, 64 x 128) and
the sizes at which they change, bit for bit against the oracle: partial row and
column tiles, one K stage, long K, and rows that small-M kernels used to take."""
import numpy as np
import pytest

from glypr_amd import ops
from glypr_amd.ops import INT8_EXACT, INT8_FMA, Q8Weight
from test_gpu_int8_fma import assert_bits_equal, dev, host, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n", [(1213, 768, 1280), (1901, 640, 1001), (2048, 512, 3072),
                                   (2049, 128, 65), (2500, 768, 768), (3333, 896, 333),
                                   (3001, 768, 1280), (4801, 768, 767), (4097, 2048, 511),
                                   (6017, 768, 1153)])
def test_matmul_tiles_bit_exact(ctx, oracle, m, k, n):
    """Output rows depend on their own x row only, so the oracle runs the rows
    around every 64-row boundary it meets first and last, and a spread of others."""
    say(f"matmul tiles m={m} k={k} n={n}")
    x = oracle.normal(m * k, seed=500 + m).reshape(m, k)
    wb = oracle.q8_0_weight(n, k, seed=600 + n)
    w = Q8Weight.from_gguf(ctx, wb, n, k)
    rows = np.unique(np.r_[0:66, 126:130, m // 2:m // 2 + 33, m - 130:m,
                           np.linspace(0, m - 1, 40).astype(int)])
    rows = rows[(rows >= 0) & (rows < m)]
    y = host(ops.q8_0_matmul(ctx, w, dev(x), INT8_EXACT))
    assert_bits_equal(y[rows], oracle.matmul(x[rows], wb, n), f"{m}x{k}x{n}")
    f = host(ops.q8_0_matmul(ctx, w, dev(x), INT8_FMA))
    assert_bits_equal(f[rows], oracle.matmul_fma(x[rows], wb, n), f"fma {m}x{k}x{n}")
