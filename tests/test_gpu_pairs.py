"""The all-pairs int8 kernel that keeps its queries in LDS (rows of 64 to 1024
bytes), at the edges of its tiles: 16-query tiles, 64-query passes, 16-row
database tiles and databases that take several walks per workgroup."""
import numpy as np
import pytest

from glypr_amd import ops
from test_gpu_vec import dev, host, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,nb,dim", [(1, 1, 64), (16, 15, 128), (17, 65, 256), (33, 16, 512),
                                       (65, 4097, 768), (130, 63, 1024), (3, 70001, 768),
                                       (32, 33000, 64)])
def test_int8_pairs_lds(ctx, na, nb, dim):
    """Integer sums against numpy's int32 product; the cosine's float32 steps
    (correctly rounded roots, product, quotient) restated in numpy, bit for bit."""
    say(f"int8 pairs in LDS na={na} nb={nb} dim={dim}")
    rng = np.random.default_rng(na + nb + dim)
    a = rng.integers(-128, 128, size=(na, dim), dtype=np.int8)
    b = rng.integers(-128, 128, size=(nb, dim), dtype=np.int8)
    b[nb // 2] = 0
    a[-1] = -128
    a32, b32 = a.astype(np.int32), b.astype(np.int32)
    # exact in float64: |sums| <= 1024 x 2^14
    dot = (a32.astype(np.float64) @ b32.astype(np.float64).T).astype(np.int32)
    assert np.array_equal(host(ops.int8_dot(ctx, dev(a), dev(b))), dot)
    ra = np.sqrt((a32 * a32).sum(1).astype(np.float32))
    rb = np.sqrt((b32 * b32).sum(1).astype(np.float32))
    den = ra[:, None] * rb[None, :]
    with np.errstate(divide="ignore", invalid="ignore"):
        ref = np.clip(dot.astype(np.float32) / den, np.float32(-1), np.float32(1))
    ref[den == 0] = 0
    got = host(ops.int8_cosine(ctx, dev(a), dev(b)))
    assert np.array_equal(got.view(np.uint32), ref.astype(np.float32).view(np.uint32))
