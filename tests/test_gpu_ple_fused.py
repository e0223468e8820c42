"""The per-layer-embedding path's fused launches (gather + Q8_0, scale + RMSNorm,
gate GEMM + GeGLU + Q8_0) and the separate launches that more than 2048 rows
take, bit for bit: every o projection is zero, so attention adds exactly 0 and
the rest of the model is in the reference's order (ple.rs, layer.rs:20-50)."""
import numpy as np
import pytest
import torch

from glypr_amd.ops import Model
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
