"""attention_supported (attn_plan.cpp), host arithmetic: 131,072 keys in a
block's reach (64 partitions of 64 tiles of 32 keys) run, one more is refused,
a narrower band runs at any length, and every plan's partitions cover the key
tiles of every one of its query blocks within the combine's 64."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "glypr_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"

DRIVER = r"""
#include <stdio.h>
#include "internal.hpp"
using namespace glypr;
// Whether p's partitions cover the key tiles of each of its blocks over t queries of
// one sequence (of rows starting at 0): kb_lo and kb_hi as the kernels form them
static bool covers(const AttnPlan& p, int64_t t, int64_t G, int64_t w) {
  const int64_t rows = attn_padded_len(t);
  const bool banded = w > 0 && t > w;
  const int64_t groups = (rows / 32) * G, blocks =
      p.qs ? rows / (16 * p.qs) : (groups + p.waves - 1) / p.waves;
  for (int64_t b = 0; b < blocks; b++) {
    int64_t q0 = 16 * p.qs * b, q1 = q0 + 16 * p.qs;
    if (p.qs == 0) {   // column groups: 32 queries of one head, head-minor
      const int64_t c0 = b * p.waves, c1 = c0 + p.waves < groups ? c0 + p.waves : groups;
      q0 = 32 * (c0 / G);
      q1 = 32 * ((c1 - 1) / G) + 32;
    }
    int64_t lo = 0, hi = (t + ATTN_AK - 1) / ATTN_AK;
    if (banded) {
      lo = (q0 - w > 0 ? q0 - w : 0) / ATTN_AK;
      hi = (q1 - 1 + w < t - 1 ? q1 - 1 + w : t - 1) / ATTN_AK + 1;
    }
    if (hi - lo > (int64_t)p.kparts * p.per) return false;
  }
  return true;
}
int main() {
  int bad = 0;
  for (const int64_t hd : {256, 512}) {
    bad += !attention_supported(131072, 4, 1, hd, 0);
    bad += attention_supported(131073, 4, 1, hd, 0);
    bad += attention_supported(200000, 4, 1, hd, 70000);
    bad += !attention_supported(200000, 4, 1, hd, 512);
    for (int64_t t = 1; t <= 131072; t += t < 1400 ? 13 : t < 9000 ? 381 : 40691)
      for (const int64_t w : {0, 1, 31, 33, 100, 512, 3000})
        for (const int64_t G : {1, 2, 3, 4})
          for (const int64_t nkv : {1, 2, 8})
            for (const int64_t extra : {0, 4096})   // rows of other sequences
              for (const bool seg : {false, true}) {
                const AttnPlan p =
                    attn_plan(t, attn_padded_len(t) + extra, hd, nkv * G, nkv, w, seg);
                bad += p.kparts < 1 || p.kparts > 64 || !covers(p, t, G, w);
                bad += p.qs == 0 && seg && 64 % (32 * p.waves / G) != 0;   // one sequence each
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
