"""The device tanh of GeGLU against the oracle's on every gate where its quotient
runs: device_common.hpp forms -t / (t + 2) with a Newton step and one residual
correction in place of the general division, equal to the IEEE quotient."""
import numpy as np
import pytest
import torch

from glypr_amd import ops
from test_gpu_backbone import host, say

pytestmark = pytest.mark.gpu


def test_geglu_of_every_gate(ctx, oracle):
    """All 1.4e8 floats from 2^-13 (tanh's linear range begins above) to 10
    (saturated), and a seventeenth of their negatives, at up = 1: bit for bit."""
    lo, hi = (int(np.float32(v).view(np.uint32)) for v in (2.0 ** -13, 10.5))
    step = 1 << 24
    one = torch.ones(step, device="cuda")
    for start in range(lo, hi, step):
        say(f"geglu gates from {np.uint32(start).view(np.float32)!r}")
        g = np.arange(start, min(start + step, hi), dtype=np.uint32).view(np.float32)
        for gate in (g, -g[::17]):
            gate = np.ascontiguousarray(gate)
            got = host(ops.geglu(ctx, torch.from_numpy(gate).cuda(), one[:gate.size]))
            ref = oracle.geglu(gate, np.ones_like(gate))
            bad = np.flatnonzero(got.view(np.uint32) != ref.view(np.uint32))
            assert bad.size == 0, (gate[bad[:3]], got[bad[:3]], ref[bad[:3]])
