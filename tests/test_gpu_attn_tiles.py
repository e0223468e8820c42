"""GPU parity of the 32 x 32-tile attention (k_attn32.hip) where its blocks can
go wrong: last column groups that do not fill a workgroup, key counts around a
tile, bands narrower than a block, one to four q heads per kv head, both head
dims, and several sequences per forward."""
import numpy as np
import pytest
import torch

from glypr_amd import ops
from glypr_amd.ops import Model
from test_gpu_backbone import attention_ref, dev, host, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,window,nq,nkv,hd,qk", [
    (1025, 0, 1, 1, 256, 0.25), (1089, 31, 3, 1, 256, 1.0), (1153, 0, 4, 1, 256, 1.0),
    (1281, 100, 6, 2, 256, 0.25), (833, 512, 4, 2, 256, 0.25), (1375, 64, 3, 1, 256, 0.25),
    (705, 0, 4, 1, 512, 1.0), (799, 0, 3, 1, 512, 0.25), (1217, 33, 2, 1, 512, 0.25),
    (961, 0, 1, 1, 512, 1.0), (1057, 64, 8, 2, 512, 0.25)])
def test_tile_attention_vs_oracle(ctx, oracle, t, window, nq, nkv, hd, qk):
    """5e-4 of the largest value against the oracle fed the same f16 Q, K and V
    (the f16 probabilities' 2^-11 remains): test_attention_core_vs_oracle's
    bound.  qk = 1 spreads the logits over tens of units, so that the running
    maximum moves after the first tile."""
    say(f"tile attention t={t} window={window} nq={nq} nkv={nkv} hd={hd} qk={qk}")
    qkv = oracle.normal(t * (nq + 2 * nkv) * hd, seed=t + 21).reshape(t, -1) * np.float32(0.7)
    qnw = (1 + 0.1 * oracle.normal(hd, seed=7)) * np.float32(qk)
    knw = (1 + 0.1 * oracle.normal(hd, seed=8)) * np.float32(qk)
    ref16, c, s = attention_ref(oracle, qkv, qnw, knw, 1e-6, 1e4, nq, nkv, hd, window, True)
    args = (dev(qkv), dev(qnw), dev(knw), 1e-6, dev(c), dev(s), nq, nkv, hd, window)
    got = host(ops.attention(ctx, *args))
    assert np.abs(got - ref16).max() <= 5e-4 * np.abs(ref16).max()
    assert np.array_equal(got, host(ops.attention(ctx, *args)))


@pytest.mark.parametrize("nq,nkv,lens", [(1, 1, [700, 65, 1000, 640, 33, 900]),
                                         (2, 2, [512, 1, 700, 64, 1000, 300]),
                                         (3, 1, [1000, 64, 31, 700, 900]),
                                         (4, 1, [65, 800, 700, 1])])
def test_tile_attention_batch_vs_single(ctx, oracle, nq, nkv, lens):
    """Sequences that share one forward (workgroups of two to four waves) keep
    their single-sequence embeddings, to test_embed_batch_vs_single_and_oracle's
    cosines."""
    say(f"tile attention batch nq={nq} nkv={nkv} lens={lens}")
    H, F, vocab, L = 256, 256, 500, 2
    m = Model(ctx, hidden=H, ffn=F, n_heads=nq, n_kv_heads=nkv, n_layers=L, vocab=vocab,
              sliding_window=200, max_seq_len=1024, max_batch_tokens=8192, layer_types=[0, 1])
    seed = 400

    def q8(name, n, k):
        nonlocal seed
        m.set_tensor(name, oracle.q8_0_weight(n, k, seed=seed), n, k, True)
        seed += 1

    def f32(name, n, scale=1.0):
        nonlocal seed
        m.set_tensor(name, (1 + 0.1 * oracle.normal(n, seed=seed)) * np.float32(scale), 1, n, False)
        seed += 1

    q8("token_embd.weight", vocab, H)
    f32("output_norm.weight", H)
    for i in range(L):
        for name, n, k in [("attn_q", nq * 256, H), ("attn_k", nkv * 256, H),
                           ("attn_v", nkv * 256, H), ("attn_output", H, nq * 256),
                           ("ffn_gate", F, H), ("ffn_up", F, H), ("ffn_down", H, F)]:
            q8(f"blk.{i}.{name}.weight", n, k)
        for name in ("attn_norm", "post_attention_norm", "ffn_norm", "post_ffw_norm"):
            f32(f"blk.{i}.{name}.weight", H)
        f32(f"blk.{i}.attn_q_norm.weight", 256, 0.25)
        f32(f"blk.{i}.attn_k_norm.weight", 256, 0.25)
    m.finalize()
    seqs = [oracle.uniform_ids(n, seed=50 + i, vocab=vocab) for i, n in enumerate(lens)]
    got = host(m.embed_batch(seqs))
    assert np.isfinite(got).all()
    for i, q in enumerate(seqs):
        one = host(m.embed(q))
        cos = float(got[i].astype(np.float64) @ one / np.linalg.norm(got[i]) / np.linalg.norm(one))
        assert cos >= (0.99999 if lens[i] >= 256 else 0.9999), (i, lens[i], cos)
    m.close()
