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


@pytest.mark.parametrize("m,H,F,scale", [(2049, 128, 32, 1.0), (2113, 256, 96, 8.0),
                                         (2177, 128, 160, 64.0), (2307, 256, 64, 1e-3)])
def test_geglu_tile_epilogue_bit_exact(ctx, oracle, m, H, F, scale):
    """The 128 x 128 tile's GeGLU epilogue: one h block to a partial pair, gates
    from the tanh's linear range to its saturation, rows of zeros, of single
    values, and of infinities and NaN."""
    say(f"geglu epilogue m={m} H={H} F={F} scale={scale}")
    x = (oracle.normal(m * H, seed=700 + m).reshape(m, H) * scale).astype(np.float32)
    x[5] = 0
    x[40] = 0
    x[40, 7] = 3 * scale
    x[66] *= np.float32(1e30)
    x[67] *= np.float32(1e-30)
    x[90, 3] = np.inf
    x[91, 3] = np.nan
    gb, ub, db = (oracle.q8_0_weight(F, H, seed=701), oracle.q8_0_weight(F, H, seed=702),
                  oracle.q8_0_weight(H, F, seed=703))
    gu, _ = Q8Weight.concat(ctx, [Q8Weight.from_gguf(ctx, gb, F, H),
                                  Q8Weight.from_gguf(ctx, ub, F, H)])
    y = host(ops.mlp(ctx, gu, Q8Weight.from_gguf(ctx, db, H, F), dev(x), INT8_EXACT))
    h = oracle.geglu(oracle.matmul(x, gb, F), oracle.matmul(x, ub, F))
    ref, odd = oracle.matmul(h, db, H), [66, 90, 91]
    np.testing.assert_array_equal(y[odd], ref[odd])    # a NaN's payload is not defined
    assert_bits_equal(np.delete(y, odd, 0), np.delete(ref, odd, 0), "geglu epilogue")


@pytest.mark.parametrize("m,k,n", [(1, 1024, 33), (17, 2048, 64), (333, 2048, 512),
                                   (1025, 1024, 31)])
def test_padded_scale_rows_bit_exact(ctx, oracle, m, k, n):
    """Small-M kernels at K % 1024 == 0, whose LDS scale rows carry one chunk of
    padding: plain and RMSNorm matmul, and the gate/up tile of an MLP."""
    say(f"padded scale rows m={m} k={k} n={n}")
    x = oracle.normal(m * k, seed=800 + m).reshape(m, k)
    nw = 1 + 0.1 * oracle.normal(k, seed=801)
    wb = oracle.q8_0_weight(n, k, seed=802)
    w = Q8Weight.from_gguf(ctx, wb, n, k)
    assert_bits_equal(host(ops.q8_0_matmul(ctx, w, dev(x), INT8_EXACT)), oracle.matmul(x, wb, n),
                      "matmul")
    assert_bits_equal(host(ops.rmsnorm_q8_0_matmul(ctx, w, dev(x), dev(nw), 1e-6, INT8_EXACT)),
                      oracle.matmul(oracle.rmsnorm(x, nw, 1e-6), wb, n), "rmsnorm matmul")
    F = 64
    gb, ub, db = (oracle.q8_0_weight(F, k, seed=803), oracle.q8_0_weight(F, k, seed=804),
                  oracle.q8_0_weight(k, F, seed=805))
    gu, _ = Q8Weight.concat(ctx, [Q8Weight.from_gguf(ctx, gb, F, k),
                                  Q8Weight.from_gguf(ctx, ub, F, k)])
    y = host(ops.mlp(ctx, gu, Q8Weight.from_gguf(ctx, db, k, F), dev(x), INT8_EXACT))
    h = oracle.geglu(oracle.matmul(x, gb, F), oracle.matmul(x, ub, F))
    assert_bits_equal(y, oracle.matmul(h, db, k), "mlp")
