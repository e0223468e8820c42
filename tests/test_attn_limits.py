"""attention_supported (attn_plan.cpp), host arithmetic: 131,072 keys in a
block's reach (64 partitions of 64 tiles of 32 keys) run, one more is refused,
a narrower band runs at any length, and every plan's partitions cover the keys
within the combine's 64."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "glypr_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"

DRIVER = r"""
#include <stdio.h>
#include "internal.hpp"
using namespace glypr;
int main() {
  int bad = 0;
  for (const int64_t hd : {256, 512}) {
    bad += !attention_supported(131072, 4, 1, hd, 0);
    bad += attention_supported(131073, 4, 1, hd, 0);
    bad += attention_supported(200000, 4, 1, hd, 70000);
    bad += !attention_supported(200000, 4, 1, hd, 512);
    for (const int64_t t : {1, 33, 1025, 4097, 40000, 131072})
      for (const int64_t w : {0, 512})
        for (const bool seg : {false, true}) {
          const AttnPlan p = attn_plan(t, attn_padded_len(t), hd, 4, 1, w, seg);
          const int64_t tiles = w == 0 ? (t + ATTN_AK - 1) / ATTN_AK : 1;
          bad += p.kparts < 1 || p.kparts > 64 || (int64_t)p.kparts * p.per < tiles;
        }
  }
  printf("%d wrong\n", bad);
  return bad != 0;
}
"""


def test_attention_limits_and_partitions(tmp_path):
    src = tmp_path / "limits.cpp"
    src.write_text(DRIVER)
    exe = tmp_path / "limits"
    r = subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O2",
                        f"-I{ROOT}/include", f"-I{CSRC}", os.path.join(CSRC, "attn_plan.cpp"),
                        str(src), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
