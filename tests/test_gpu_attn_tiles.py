"""GPU parity of the 32 x 32-tile attention (k_attn32.hip) where its blocks can
go wrong: last column groups that do not fill a workgroup, key counts around a
tile, bands narrower than a block, one to four q heads per kv head, both head
dims, and several sequences per forward on workgroups of two, three and four
waves.  The tests that name a plan ask the planner for it, so that a change of
its costs cannot move them to another kernel unseen; the others run whatever the
plan picks for lengths near its lines."""
import numpy as np
import pytest
import torch

from glypr_amd import ops
from glypr_amd.ops import Model
from attn_plan_util import plan
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


@pytest.mark.parametrize("t,window,nq,nkv,hd,split", [
    # bands of at most a wave's 32 queries, with partial tiles and column groups
    (4161, 31, 3, 1, 256, False), (4225, 1, 2, 1, 256, False), (2113, 33, 8, 2, 256, False),
    (4225, 31, 4, 4, 256, False), (4161, 33, 2, 1, 512, False), (4225, 31, 3, 1, 512, False),
    (2113, 1, 8, 2, 512, False), (1301, 31, 4, 4, 512, False), (2113, 64, 2, 2, 512, True),
    # one to four q heads per kv head, one partition and several
    (2081, 0, 1, 1, 256, True), (2113, 0, 2, 1, 256, True), (1089, 512, 3, 1, 256, True),
    (1153, 0, 4, 1, 256, True), (3500, 512, 6, 2, 256, False), (2113, 512, 8, 2, 256, False),
    (577, 0, 1, 1, 512, True), (643, 0, 2, 1, 512, True), (671, 0, 3, 1, 512, True),
    (705, 512, 8, 2, 512, True), (2689, 512, 6, 2, 512, False)])
def test_planned_tiles_vs_oracle(ctx, oracle, t, window, nq, nkv, hd, split):
    """test_tile_attention_vs_oracle's comparison at lengths that plan onto the
    tile kernel, written directly (split False) or merged from partitions."""
    p = plan(t, nq, nkv, hd, window)
    assert p.kind == "tile" and p.waves == 4 and (p.kparts > 1) == split, p
    test_tile_attention_vs_oracle(ctx, oracle, t, window, nq, nkv, hd, 0.5)


@pytest.mark.parametrize("nq,nkv,hd,window,lens,waves,split", [
    (1, 1, 256, 0, [2000, 1900, 64, 1, 1700, 31], 2, True),
    (2, 2, 256, 0, [1500, 2, 63, 1700, 65, 1024, 333], 2, True),
    (2, 2, 256, 200, [1000, 65, 999, 64, 1000, 960, 1, 900, 1000, 800, 31, 930], 2, False),
    (2, 1, 256, 200, [1500, 2, 63, 1700, 65, 1024, 333], 4, True),
    (3, 1, 256, 0, [2000, 64, 1, 333], 3, True),
    (3, 1, 256, 200, [1500, 2, 63, 1700, 65, 1024, 333], 3, False),
    (4, 1, 256, 200, [2000, 1900, 64, 1, 1700, 31], 4, False),
    (1, 1, 512, 0, [400, 5, 128, 300, 33, 1, 500, 257], 2, True),
    (2, 2, 512, 0, [2000, 1900, 64, 1, 1700, 31], 2, False),
    (2, 1, 512, 0, [1000, 64, 31, 700, 900, 1, 130], 4, True),
    (3, 1, 512, 0, [1000, 64, 31, 700, 900, 1, 130], 3, True),
    (6, 2, 512, 0, [1000, 64, 31, 700, 900, 1, 130], 3, False),
    (4, 1, 512, 0, [600, 64, 1, 550, 33, 500, 31], 4, True),
    (4, 2, 512, 0, [1500, 2, 63, 1700, 65, 1024, 333], 4, False)])
def test_planned_tiles_batch_vs_single(ctx, oracle, nq, nkv, hd, window, lens, waves, split):
    """One attention layer with its feed-forward block silenced (ffn_down = 0), so
    that the embedding of a sequence is the mean over its tokens of the normalised
    embedding plus attention output, against the same sequence alone.  Probabilities
    rounded to f16 against other maxima move a context value by 2^-12, so 127 2^-12 =
    3 % of its Q8_0 codes by one step of at most 1 / 127 of the block's largest: 1.4e-3
    of a token, twice that is the bound for the mean (measured: up to 6.6e-4).  One
    wrong 32-row column group is 2e-2 of 1500 tokens, one wrong row 1e-2 of 65."""
    say(f"planned tile batch nq={nq} nkv={nkv} hd={hd} window={window} lens={lens}")
    rows = sum(-(-n // 64) * 64 for n in lens)
    p = plan(max(lens), nq, nkv, hd, window, rows=rows, segments=True)
    assert p.kind == "tile" and p.waves == waves and (p.kparts > 1) == split, p
    H, vocab, seed = 256, 500, 900
    m = Model(ctx, hidden=H, ffn=256, n_heads=nq, n_kv_heads=nkv, n_layers=1, vocab=vocab,
              sliding_window=window or 512, max_seq_len=2048, max_batch_tokens=8192,
              layer_types=[0 if window else 1], full_head_dim=hd)

    def q8(name, n, k, scale=1.0):
        nonlocal seed
        w = oracle.q8_0_weight(n, k, seed=seed)
        m.set_tensor(name, w if scale else np.zeros_like(w), n, k, True)
        seed += 1

    def f32(name, n, scale=1.0):
        nonlocal seed
        m.set_tensor(name, (1 + 0.1 * oracle.normal(n, seed=seed)) * np.float32(scale), 1, n, False)
        seed += 1

    q8("token_embd.weight", vocab, H)
    f32("output_norm.weight", H)
    for name, n, k, scale in [("attn_q", nq * hd, H, 1), ("attn_k", nkv * hd, H, 1),
                              ("attn_v", nkv * hd, H, 1), ("attn_output", H, nq * hd, 1),
                              ("ffn_gate", 256, H, 1), ("ffn_up", 256, H, 1),
                              ("ffn_down", H, 256, 0)]:
        q8(f"blk.0.{name}.weight", n, k, scale)
    for name in ("attn_norm", "post_attention_norm", "ffn_norm", "post_ffw_norm"):
        f32(f"blk.0.{name}.weight", H)
    f32("blk.0.attn_q_norm.weight", hd, 0.5)
    f32("blk.0.attn_k_norm.weight", hd, 0.5)
    m.finalize()
    seqs = [oracle.uniform_ids(n, seed=70 + i, vocab=vocab) for i, n in enumerate(lens)]
    got = host(m.embed_batch(seqs)).astype(np.float64)
    errs = [float(np.linalg.norm(got[i] - host(m.embed(q)))) for i, q in enumerate(seqs)]
    say("  relative differences " + " ".join(f"{n}:{e:.1e}" for n, e in zip(lens, errs)))
    for n, e in zip(lens, errs):
        assert e <= 2.8e-3, (n, e)
    m.close()
