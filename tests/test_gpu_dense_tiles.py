"""The bf16 GEMMs' tiles on both sides of the sizes at which they change: the
dense-weight kernel's 64 x 64, 64 x 128 and 128 x 128, the dequantizing kernel's
32, 64 and 128 rows, with partial row and column tiles, one to many K stages and
output widths that do not vectorise."""
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


@pytest.mark.parametrize("m,k,n", [(1, 64, 1), (33, 128, 129), (350, 768, 1280), (1025, 192, 1025),
                                   (2048, 768, 1280), (2049, 2048, 511), (3072, 64, 1024),
                                   (3073, 128, 1025)])
def test_bf16_dequant_rows_within_bound(ctx, oracle, m, k, n):
    """The dequantizing kernel in 32-, 64- and 128-row workgroups: both operands
    rounded to bf16 (2^-8 each), k f32 accumulations (at most 2^-13 of the terms'
    sum here)."""
    say(f"BF16_DEQUANT rows m={m} k={k} n={n}")
    x = oracle.normal(m * k, seed=900 + m).reshape(m, k)
    wb = oracle.q8_0_weight(n, k, seed=950 + n)
    w = ops.Q8Weight.from_gguf(ctx, wb, n, k)
    y = host(ops.q8_0_matmul(ctx, w, dev(x), ops.BF16_DEQUANT)).astype(np.float64)
    wd = oracle.dequantize_rows(wb, k).reshape(n, k).astype(np.float64)
    lim = (2.0 ** -7 + 2.0 ** -16 + 2.0 ** -13) * (np.abs(x).astype(np.float64) @ np.abs(wd).T)
    assert np.all(np.abs(y - x.astype(np.float64) @ wd.T) <= lim)


@pytest.mark.parametrize("m,H,F", [(1, 64, 32), (100, 768, 1152), (513, 256, 96), (1000, 512, 2048)])
def test_bf16_dequant_mlp_rows(ctx, oracle, m, H, F):
    """The gate/up form of the same workgroups, through the MLP: per-row cosine to
    the float64 dequant oracle as in test_mlp_bf16_dequant."""
    say(f"BF16_DEQUANT MLP rows m={m} H={H} F={F}")
    x = oracle.normal(m * H, seed=970).reshape(m, H)
    gb, ub = oracle.q8_0_weight(F, H, seed=971), oracle.q8_0_weight(F, H, seed=972)
    db = oracle.q8_0_weight(H, F, seed=973)
    gu, _ = ops.Q8Weight.concat(ctx, [ops.Q8Weight.from_gguf(ctx, gb, F, H),
                                      ops.Q8Weight.from_gguf(ctx, ub, F, H)])
    d = ops.Q8Weight.from_gguf(ctx, db, H, F)
    y = host(ops.mlp(ctx, gu, d, dev(x), ops.BF16_DEQUANT)).astype(np.float64)
    gate = oracle.matmul_dequant_f64(x, gb, F).astype(np.float32)
    up = oracle.matmul_dequant_f64(x, ub, F).astype(np.float32)
    ref = oracle.matmul_dequant_f64(oracle.geglu(gate, up), db, H)
    cos = (y * ref).sum(1) / np.linalg.norm(y, axis=1) / np.linalg.norm(ref, axis=1)
    assert cos.min() > 0.999, cos.min()
