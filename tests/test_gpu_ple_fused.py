"""The per-layer-embedding path's fused launches (gather + Q8_0, scale + RMSNorm,
gate GEMM + GeGLU + Q8_0) and the separate launches that more than 2048 rows
take, bit for bit: every o projection is zero, so attention adds exactly 0 and
the rest of the model is in the reference's order (ple.rs, layer.rs:20-50)."""
import ctypes

import numpy as np
import pytest
import torch

from glypr_amd import _lib
from glypr_amd.ops import INT8_EXACT, INT8_FMA, Model
from test_gpu_backbone import host, make_model, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,P", [(1, 32), (17, 96), (300, 256), (333, 160), (1500, 64),
                                 (2048, 32), (2049, 32)])
def test_ple_model_attention_silenced_bit_exact(ctx, oracle, t, P):
    n_layers, vocab, D = 2, 500, 128
    say(f"attention-silenced PLE backbone t={t} P={P}")
    m0, tensors = make_model(ctx, oracle, n_layers, vocab, seed=60, ple_dim=P, out_dim=D)
    m0.close()
    for i in range(n_layers):
        data, r, c, q8 = tensors[f"blk.{i}.attn_output.weight"]
        tensors[f"blk.{i}.attn_output.weight"] = (np.zeros_like(data), r, c, q8)
    m = Model(ctx, n_layers=n_layers, vocab=vocab, ple_dim=P, out_dim=D)
    for name, (data, r, c, q8) in tensors.items():
        m.set_tensor(name, data, r, c, q8)
    m.finalize()
    ids = oracle.uniform_ids(t, seed=t + 1, vocab=vocab)
    tokens = torch.empty((t, D), dtype=torch.float32, device="cuda")
    m.embed(ids, trunc=128, hidden=tokens)
    flat = {k: (v[0] if v[3] else np.asarray(v[0], np.float32).reshape(-1))
            for k, v in tensors.items()}
    _, ref = oracle.model_forward(flat, ids, 128, hidden=768, ffn=1152, n_heads=3, n_kv_heads=1,
                                  head_dim=256, n_layers=n_layers, vocab=vocab)
    got = host(tokens)
    assert int((got.view(np.uint32) != ref.astype(np.float32).view(np.uint32)).sum()) == 0
    m.close()


def ple_model(ctx, oracle, H, P, n_layers, vocab, D):
    """A PLE model of hidden width H whose attention adds exactly 0."""
    tensors = {}
    seed = 60 * H

    def q8(name, n, k, sigma=0.02, zero=False):
        nonlocal seed
        seed += 1
        w = oracle.q8_0_weight(n, k, seed=seed, sigma=sigma)
        tensors[name] = (np.zeros_like(w) if zero else w, n, k, True)

    def f32(name, n, scale=1.0):
        nonlocal seed
        seed += 1
        tensors[name] = ((1 + 0.1 * oracle.normal(n, seed=seed)) * np.float32(scale), 1, n, False)

    q8("token_embd.weight", vocab, H)
    f32("output_norm.weight", H)
    q8("per_layer_model_proj.weight", n_layers * P, H, 0.05)
    f32("per_layer_proj_norm.weight", P)
    q8("output.weight", D, H, 0.05)
    for i in range(n_layers):
        b = f"blk.{i}."
        for name, n, k in [("attn_q", 256, H), ("attn_k", 256, H), ("attn_v", 256, H),
                           ("ffn_gate", 256, H), ("ffn_up", 256, H), ("ffn_down", H, 256)]:
            q8(f"{b}{name}.weight", n, k)
        q8(f"{b}attn_output.weight", H, 256, zero=True)
        for name in ("attn_norm", "post_attention_norm", "ffn_norm", "post_ffw_norm", "post_norm"):
            f32(f"{b}{name}.weight", H)
        f32(f"{b}attn_q_norm.weight", 256, 0.25)
        f32(f"{b}attn_k_norm.weight", 256, 0.25)
        q8(f"{b}inp_gate.weight", P, H, 0.05)
        q8(f"{b}proj.weight", H, P, 0.05)
        tensors[f"{b}layer_output_scale.weight"] = (np.array([0.6], np.float32), 1, 1, False)
    m = Model(ctx, hidden=H, ffn=256, n_heads=1, n_kv_heads=1, n_layers=n_layers, vocab=vocab,
              ple_dim=P, out_dim=D)
    for name, (data, r, c, q) in tensors.items():
        m.set_tensor(name, data, r, c, q)
    m.finalize()
    return m, tensors


@pytest.mark.parametrize("H,P", [(256, 64), (512, 256), (640, 64), (768, 32), (1024, 96)])
def test_fused_gate_widths_bit_exact(ctx, oracle, H, P):
    """Every width the gate kernel is built for (1024 with the padded scale rows),
    and one that keeps the two launches: 300 tokens in the reference's order
    (INT8_EXACT), and with either epilogue the same rows as the unfused launches
    that more than 2048 tokens take."""
    say(f"fused PLE gate H={H} P={P}")
    vocab, D, t = 300, 64, 300
    gate = _lib.lib().glypr_internal_gemm_i8_gate_ok
    assert gate(*map(ctypes.c_int64, (t, P, H))) == (H != 640)
    assert gate(*map(ctypes.c_int64, (2049, P, H))) == 0
    m, tensors = ple_model(ctx, oracle, H, P, 2, vocab, D)
    ids = oracle.uniform_ids(2049, seed=H, vocab=vocab)
    long, short = (torch.empty((n, D), device="cuda") for n in (2049, t))
    for variant in (INT8_EXACT, INT8_FMA):
        m.set_variant(variant)
        m.embed(ids, trunc=D, hidden=long)
        m.embed(ids[:t], trunc=D, hidden=short)
        a, b = host(long)[:t], host(short)
        assert np.isfinite(b).all()
        assert int((a.view(np.uint32) != b.view(np.uint32)).sum()) == 0, variant
        if variant == INT8_EXACT:
            flat = {k: (v[0] if v[3] else np.asarray(v[0], np.float32).reshape(-1))
                    for k, v in tensors.items()}
            _, ref = oracle.model_forward(flat, ids[:t], D, hidden=H, ffn=256, n_heads=1,
                                          n_kv_heads=1, head_dim=256, n_layers=2, vocab=vocab)
            assert int((b.view(np.uint32) != ref.astype(np.float32).view(np.uint32)).sum()) == 0
    m.close()
