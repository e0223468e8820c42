"""What one attention launch runs (attn_plan.cpp through the library's probe)."""
import collections
import ctypes

from glypr_amd import _lib

# kind: "short" (one launch), "tile" (32 x 32 tiles on `waves` waves), "q16" or "q64"
Plan = collections.namedtuple("Plan", "kind waves per kparts")


def plan(t, nq, nkv, hd=256, window=0, rows=0, segments=False):
    out = (ctypes.c_int * 5)()
    f = _lib.lib().glypr_internal_attn_plan
    f.restype = None
    f(*map(ctypes.c_int64, (t, rows, nq, nkv, hd, window)), ctypes.c_int(segments), out)
    short, qs, waves, per, kparts = out
    return Plan("short" if short else "tile" if qs == 0 else f"q{16 * qs}", waves, per, kparts)
