"""The 32 x 32-tile attention (k_attn32.hip) on inputs whose softmax is known in
closed form, where an f32 sum or an exponent's reference that is rounded too
early shows: cos = 1 and sin = 0 leave the normalised heads unrotated, rows of
+-1 have RMS 1 (the epsilon is below an ulp), and the norm weights are powers of two, so every score is exact."""
import numpy as np
import pytest
import torch

from attn_plan_util import plan
from glypr_amd import ops
from test_gpu_backbone import say

pytestmark = pytest.mark.gpu


def constructed(ctx, t, nq, nkv, hd, scores, base, v_sign):
    """Attention whose key r scores base + scores[r] / 128 (odd |scores| < 2048)
    for every query and whose value rows are v_sign[r] * ones."""
    qw, kw, ks = torch.zeros(hd), torch.zeros(hd), torch.ones(t, hd)
    qw[0] = kw[0] = base ** 0.5
    m = (scores + 2047) // 2   # scores = sum of +-2^j over the bits of m
    for j in range(11):
        qw[1 + j], kw[1 + j] = 2.0 ** -4, 2.0 ** (j - 3)
        ks[:, 1 + j] = torch.where((m >> j) & 1 == 1, 1.0, -1.0)
    qkv = torch.cat([torch.ones(t, nq * hd), ks.repeat(1, nkv),
                     v_sign[:, None].expand(t, nkv * hd)], 1).cuda()
    out = ops.attention(ctx, qkv, qw.cuda(), kw.cuda(), 1e-12, torch.ones(t, hd, device="cuda"),
                        torch.zeros(t, hd, device="cuda"), nq, nkv, hd, 0)
    return out.double().cpu()


@pytest.mark.parametrize("t,nq,nkv,hd", [(2048, 3, 1, 256), (3500, 3, 1, 256), (1024, 4, 1, 512)])
def test_partitions_share_their_reference(ctx, t, nq, nkv, hd):
    """Scores near 2^16 in two halves of the keys, a little apart.  The weights of
    the halves are e^{difference}, whatever the size of the scores: 2^-11 (one
    rounding of a probability to f16) and 2^-18 for the f32 steps."""
    say(f"attention partitions t={t} nq={nq} nkv={nkv} hd={hd}")
    p = plan(t, nq, nkv, hd)
    assert p.kind == "tile" and p.kparts > 1, p
    first = torch.arange(t) < t // 2
    v = torch.where(first, 1.0, -1.0)
    for d in range(3, 400, 28):
        n = torch.where(first, d, 1)
        p = torch.exp(n.double() / 128)
        want = float((p * v).sum() / p.sum())
        got = constructed(ctx, t, nq, nkv, hd, n, 65536.0, v)
        assert float((got - want).abs().max()) <= 2 ** -11 + 2 ** -18, d


@pytest.mark.parametrize("t,nq,nkv,hd", [(32768, 1, 1, 256), (32768, 4, 1, 512)])
def test_long_sums_of_one_value(ctx, t, nq, nkv, hd):
    """One probability for all keys but the first tile's and values of 1: the
    output is 1, and additions that round the same way every time do not average
    out.  The probability is within 2^-18 of an f16; the products' chain of 2 per
    tile is held to half an ulp of its end value each, 2^-25 x 2048 = 2^-14."""
    say(f"attention long sums t={t} nq={nq} nkv={nkv} hd={hd}")
    p = plan(t, nq, nkv, hd)
    assert p.kind == "tile" and p.kparts == 1, p
    p = np.exp(-np.arange(2, 1024, 2) / 128.0)
    d = 2 + 2 * int(np.argmin(np.abs(p.astype(np.float16) / p - 1)))
    n = torch.full((t,), 1 - d, dtype=torch.int64)
    n[:32] = 1
    got = constructed(ctx, t, nq, nkv, hd, n, 0.0, torch.ones(t))
    assert float((got - 1).abs().max()) <= 2 ** -14 + 2 ** -18
